// C-ABI layer of the MI355X XC build (declared in include/pgxc.h).
//
// A build is a plan: for every super-step, the units (grid chunks) of every
// molecule taking part, and per stage the list of work items over those units.
// Stage kernels walk their lists persistently; one molecule is a batch of one.
// Per super-step:  basis -> density contraction -> functional -> W ->
// potential contraction; then per molecule a fold of the split partials (H + H^T)
// and one packing into the lower triangle.
// Chunks are whole numbers of reference batches, so the sums are those of
// calc_xcks_nl (ParaGauss modules/xc_hamiltonian.f90:1348-1575), regrouped.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <memory>
#include <mutex>
#include <numeric>
#include <string>
#include <type_traits>
#include <vector>

#include "../../include/pgxc.h"

#include "pgxc_internal.h"

using namespace pgxc;

namespace {

struct Plan;

long round_up(long a, long b) { return (a + b - 1) / b * b; }

// schedule of the contraction stages (PGXC_SCHED_*) and item logging
struct Sched {
  int mode = PGXC_SCHED_ANALYTIC;  // no slower than the static walk in any measurement
  pgxc_costmodel *model = nullptr;
  int log = 0;
};

void dfree(void *p) {
  if (p) (void)hipFree(p);
}

// Device buffers freed when the scope ends, on every return path.
struct ScopedDev {
  std::vector<void *> bufs;
  ~ScopedDev() {
    for (void *b : bufs) dfree(b);
  }
  template <typename T>
  T *keep(T *p) {
    bufs.push_back((void *)p);
    return p;
  }
};

}  // namespace

// Host memory the device copies to and from directly, in two halves that take
// turns: one is filled by the device while the host empties the other.  1 MiB a
// half: a copy of it takes longer than starting one.  The copies are kernels:
// from 32 KiB on, hipMemcpyAsync takes the copy engine, which for some contexts
// starts 110 us late behind each build (V of 132 functions 26 or 124 us, by kernel
// 23; orbitals of 132 functions 35 or 138, by kernel 35; (H2O)32's V 737, by kernel
// 219; through pageable memory 19, 58 and 451).  A thread may read a build's results while others read them or set
// the next orbitals: whoever uses the halves holds mu until their contents are
// taken.
struct PinnedPair {
  static constexpr size_t kHalf = 1 << 20;
  char *buf = nullptr;
  std::recursive_mutex mu;
  hipEvent_t ev[2] = {nullptr, nullptr};
  hipError_t init() {
    hipError_t e = hipHostMalloc((void **)&buf, 2 * kHalf, hipHostMallocCoherent);
    for (int i = 0; i < 2 && e == hipSuccess; ++i) e = hipEventCreateWithFlags(&ev[i], hipEventDisableTiming);
    return e;
  }
  void release() {
    if (buf) (void)hipHostFree(buf);
    for (auto &v : ev)
      if (v) (void)hipEventDestroy(v);
    buf = nullptr;
  }
  // n doubles at dev, in order, to take(first, count, values); waits for the
  // stream's earlier work
  template <class Take>
  hipError_t fetch(hipStream_t s, const double *dev, size_t n, Take take) {
    std::lock_guard<std::recursive_mutex> lk(mu);
    const size_t per = kHalf / 8, parts = (n + per - 1) / per;
    hipError_t e = hipSuccess;
    auto len = [&](size_t i) { return std::min(per, n - i * per); };
    for (size_t i = 0; i <= parts && e == hipSuccess; ++i) {
      if (i < parts) {
        launch_copy(s, dev + i * per, (double *)(buf + (i & 1) * kHalf), (long)len(i));
        e = hipGetLastError();
        if (e == hipSuccess) e = hipEventRecord(ev[i & 1], s);
      }
      if (i > 0 && e == hipSuccess) {
        e = hipEventSynchronize(ev[(i - 1) & 1]);
        if (e == hipSuccess) take((i - 1) * per, len(i - 1), (const double *)(buf + ((i - 1) & 1) * kHalf));
      }
    }
    return e;
  }
};

struct pgxc_ctx {
  int device = 0;
  PinnedPair pin;
  double *orb = nullptr;  // orbitals and occupations of the last pgxc_set_orbitals
  size_t orb_n = 0;
  hipStream_t stream = nullptr;
  // chunks alternate between two lanes (this stream and stream2, each with its
  // own work buffers) so one chunk's stages overlap the next chunk's
  hipStream_t stream2 = nullptr;
  hipEvent_t fork = nullptr, join = nullptr;
  int nlanes = 1, nlanes_cap = 1;  // lanes in use / with buffers
  std::string err;
  // sizes
  int n_atoms = 0, n_shells = 0, nbas = 0, NP = 0, veclen = 128, tf = 128;
  int pt = 0;  // chunk of the potential contraction: the tile asked for, else setup_screen's choice
  int lmax = 0;  // largest angular momentum of the basis
  int var[2] = {0, 1};  // contraction variant for FP64 and for FP32 builds
  long npts = 0, npad = 0, Mc = 0;
  int icols = 128;  // most columns of a density item (setup_screen)
  int nchunks = 0, nsplit = 1, nparts = 0;  // nsplit: the chunk rounding's blocks (pgxc_layout)
  int nsp = 1;  // point splits of the potential contraction per chunk (setup_screen)
  long nblk_total = 0;
  // device: geometry and basis
  double *grid = nullptr;  // [4][npad] x, y, z, w
  AtomD *atoms = nullptr;
  ShellD *shells = nullptr;
  RangeD *ranges = nullptr;  // atom ranges of the basis stage
  int *ratoms = nullptr;     // atoms in shell order
  int n_ranges = 0;
  std::vector<RangeD> h_ranges;
  double *tabd = nullptr;  // shell tables (exponents, norms, coefficients), FP64 and FP32
  float *tabf = nullptr;
  // device: density (NP x NP); D holds the operand in the build's precision
  double *P = nullptr, *Pref = nullptr;
  void *D = nullptr;
  // device: work buffers of one chunk
  void *phi = nullptr, *W = nullptr;
  size_t phi_bytes = 0, w_bytes = 0, phi_elem = 0;
  size_t w_lane = 0, phi_lane = 0;  // bytes of one lane's W / basis chunk buffer
  // basis values of every chunk kept across builds, per element type
  // ([0] FP64, [1] FP32): built once, reused while the geometry lives
  int cache_off = 0;
  void *phic[2] = {nullptr, nullptr};
  int phic_valid[2] = {0, 0}, phic_failed[2] = {0, 0};
  int phic_grad[2] = {0, 0};  // the cache also holds the gradient planes (a GGA basis pass ran)
  size_t phic_bytes[2] = {0, 0};
  void *phi_base = nullptr;  // Phi of the current build: chunk k at phi_base + k * phi_stride
  size_t phi_stride = 0;
  int skip_basis = 0;        // the current build reads cached basis values
  double *part = nullptr, *coef = nullptr;
  // potential partials (hsize doubles): those of all chunks, or (hflush, when
  // they pass kPartialBytes) of as many chunks as a lane's share holds, summed
  // into HS whenever it is full: after the chunks k with h_flush[lanes - 1][k].
  // HS: [nseg][NP][NP] their symmetric sums
  double *Hc = nullptr, *HS = nullptr;
  long hsize = 0;
  int hflush = 0, nseg = 1;
  std::vector<char> h_flush[2];
  // open shell (ispin = 2): the fields above and below serve the alpha spin,
  // these the beta spin (allocated with the first open-shell density; the
  // basis values and the work tables are shared)
  int ispin = 1;
  struct Beta {
    double *P = nullptr, *Pref = nullptr, *part = nullptr, *coef = nullptr, *Hc = nullptr, *HS = nullptr;
    double *state = nullptr, *Vstate = nullptr, *Vout = nullptr;
    void *D = nullptr, *W = nullptr;
    size_t w_bytes = 0;
    int ready = 0;  // every buffer but W is there
  } beta;
  // device: state and results
  double *state = nullptr;                    // [S_NSLOT][npad]
  double *Vstate = nullptr, *Vout = nullptr;  // packed
  double *epart = nullptr;
  // host
  int have_density = 0, density_mode = 0, have_state = 0;
  uint32_t state_functional = 0;
  uint64_t geom = 0;  // hash of the inputs that fix the layout (state files)
  double last_exc = 0, last_charge = 0;
  double timing[6] = {0, 0, 0, 0, 0, 0};
  double stats[5] = {0, 0, 0, 0, 0};
  std::vector<hipEvent_t> ev;
  Plan *plan = nullptr;
  Plan *plan_e = nullptr;  // energy-only builds (pgxc_energy)
  Plan *plan_g = nullptr;  // the nuclear gradient's stages
  double *eterm = nullptr;  // [nblk_total][5] energy-term block sums
  double last_terms[5] = {0, 0, 0, 0, 0};
  double exps_per_point = 0;
  // screening and work tables over the padded grid (setup_screen)
  int screen = 0, n8 = 0, nw8 = 0;
  int *nbt = nullptr;
  uint32_t *sig8 = nullptr;
  ScreenShell *sshells = nullptr;
  double flops_screened = 0, flops_dense = 0;  // algorithmic work of one build
  double sum_bn = 0, sum_n2 = 0;  // sums over 128-point tiles of B n_b and n_b^2 (screened)
  // host and device copies: per tile run and function lists, per split
  // function unions, per chunk density and potential items
  std::vector<int> h_tl_off, h_su_off, h_tf_off;
  std::vector<uint16_t> h_tl, h_su, h_tfl;
  std::vector<uint8_t> h_tlm;
  std::vector<long> h_di_off, h_pi_off;
  std::vector<uint32_t> h_di, h_pi;
  int *tl_off = nullptr, *su_off = nullptr, *tf_off = nullptr;
  uint16_t *tl = nullptr, *su = nullptr, *tfl = nullptr;
  uint8_t *tlm = nullptr;
  uint32_t *tfb = nullptr;  // per tile, its functions as a bitmap of nwf words
  int nwf = 0;
  // per entry of a split's function list: bit t set when the function is
  // in the list of the split's tile t
  std::vector<uint32_t> h_sumask;
  uint32_t *sumask = nullptr;
  // per split: where its partial lies in a slot, the functions' places in its
  // list, and (per 32 functions, a bit per split) whether it has any of them
  long *ho = nullptr;
  uint16_t *pos = nullptr;
  uint8_t *rbits = nullptr;
  // nuclear gradient work space (first gradient on): products of one chunk
  // (XZ, two planes) and per-(basis item, atom, wave) sums; with the grid moving
  // (first such gradient on) gpm, the points' terms, and gmov, the rest
  double *gXZ = nullptr, *gpart = nullptr, *gsum = nullptr, *gpm = nullptr;
  char *gmov = nullptr;
  int *perm_d = nullptr;  // caller index of each internal point
  uint32_t *di = nullptr, *pi = nullptr;
  // blocks of the basis values some stage reads (see setup_screen): per
  // chunk the basis items (256-point block << 16 | atom range) that touch
  // them and their write flags
  uint32_t *bi = nullptr, *bfl = nullptr;
  std::vector<long> h_bi_off;
  std::vector<int> fpos;          // internal position of each caller function
  std::vector<double> axyz;       // atom positions (bohr), caller order
  int *d_fpos = nullptr, *d_finv = nullptr;  // and its inverse, caller function of each position
  Sched sched;
};

namespace {

int fail(pgxc_ctx *c, int code, const std::string &msg) {
  if (c) c->err = msg;
  return code;
}

// An error that goes back to the caller leaves the runtime's record too, where
// the next call's check of its launches would find it and fail as well.
#define HIPCHK(ctx, call)                                                              \
  do {                                                                                 \
    hipError_t e_ = (call);                                                            \
    if (e_ != hipSuccess) {                                                            \
      (void)hipGetLastError();                                                         \
      return fail(ctx, e_ == hipErrorOutOfMemory ? PGXC_ERR_NOMEM : PGXC_ERR_HIP,       \
                  std::string(#call) + ": " + hipGetErrorString(e_));                  \
    }                                                                                  \
  } while (0)

template <typename T>
int dalloc(pgxc_ctx *c, T **p, size_t count) {
  if (*p) return PGXC_OK;
  hipError_t e = hipMalloc((void **)p, sizeof(T) * std::max<size_t>(count, 1));
  if (e != hipSuccess) {
    *p = nullptr;
    (void)hipGetLastError();
    return fail(c, PGXC_ERR_NOMEM, std::string("hipMalloc: ") + hipGetErrorString(e));
  }
  return PGXC_OK;
}

// potential partials held at a time per molecule and spin, and work items of
// their sum below which it is cut into segments
constexpr long kPartialBytes = 4L << 30, kFoldItems = 1536;
// A contraction of at most kQueueItems items is walked without queues, whose
// claims a launch of one item per workgroup waits for and gains nothing from
// (water, mixed step: density 54 -> 15 us, potential 34 -> 13): two workgroups
// on each of the 256 CUs.  The split-BF16 density with wide items has one
// workgroup a CU, and above 256 items the walk deals a second round before the
// first has ended.  The other lane's launches fill that gap; on one lane the
// queues take it (290 to 400 items a chunk, 1320 functions: density stage 2.99 ->
// 2.64 and 2.90 -> 2.58 ms, on two lanes energies 2.05 -> 2.10 ms).
constexpr long kQueueItems = 512, kQueueItemsWide = 256;
constexpr long kBasisItems = 2048;
constexpr double kWideTile = 384.0;    // setup_screen: mean functions of a tile for wide density items
constexpr double kSplitItems = 256.0;  // setup_screen: potential items a chunk has at least

const uint32_t kSupported = PGXC_XC_PBE;
const int kTiles[3] = {64, 96, 128};

// ------------------------------------------------------------------- plans
// density / potential lists per (function tile, variant): index 3 * t + v
constexpr int kLists = 3 * kNumVariants;

struct FoldList {
  const FoldD *d = nullptr;
  const long *base = nullptr;
  int n = 0;
  long total = 0;
};

struct StepPlan {
  int nunits = 0;
  FoldList flush;  // the partials summed after this step (lanes whose slots are full)
  StageList basis, func, func2, wmat, wmat2;  // func2, wmat2: open-shell units
  StageList dens[kLists], pot[kLists];
};

// The work buffers of a molecule that a plan's units hold (ensure_work makes and
// moves them).
struct WorkBufs {
  const void *phi, *W, *W2;
  size_t phi_stride, phi_lane, w_lane;
  int skip_basis;
  bool operator==(const WorkBufs &o) const {
    return phi == o.phi && W == o.W && W2 == o.W2 && phi_stride == o.phi_stride && phi_lane == o.phi_lane &&
           w_lane == o.w_lane && skip_basis == o.skip_basis;
  }
};

struct Plan {
  uint32_t functional = 0;
  int precision = 0;
  std::vector<int> incr;  // per molecule
  long order_version = -1;
  int sched_mode = 0, log = 0;
  int energy = 0;  // energy terms only: no W, potential, fold or packing
  int wbasis = 0;  // W from the basis evaluated again (k_wbasis)
  const pgxc_costmodel *model = nullptr;
  long model_version = -1;
  int *d_ctr = nullptr;  // queue counters of every contraction list
  long nctr = 0;
  // item log: features of every contraction item (row-major), and per list
  // the device log and the list's first feature row
  std::vector<double> feat;
  std::vector<std::pair<uint32_t *, long>> logs;  // (device ticks, items)
  double tick_us = 0.0;
  std::vector<StepPlan> steps;
  int nlanes = 1;  // 2: chunk k runs on lane k % 2 (two streams)
  std::vector<int> lanes;  // lanes in use per molecule when the plan was made
  std::vector<int> spins;  // ispin per molecule when the plan was made
  std::vector<WorkBufs> bufs;  // and its work buffers
  PackD *d_pack = nullptr;
  long *d_pack_base = nullptr, *d_prep_base = nullptr;
  long pack_total = 0, prep_total = 0;
  FoldList fold;
  int nmol = 0;
  char *blob = nullptr;  // device memory holding every list
  hipGraphExec_t graph = nullptr;
  hipGraph_t graph_src = nullptr;
  ~Plan() {
    if (graph) (void)hipGraphExecDestroy(graph);
    if (graph_src) (void)hipGraphDestroy(graph_src);
    dfree(blob);
  }
};

void free_plan(Plan *&p) {
  delete p;
  p = nullptr;
}

// Schedule of one stage list: a unit's items stay together, units in
// descending priority (largest predicted cost first).  Position L of the
// persistent walk runs on XCD L % 8, so contiguous runs of the sequence are
// spread to keep neighbouring items on one XCD.  Without priorities the kernels
// use the natural XCD-blocked order.
void make_order(const std::vector<long> &base, const std::vector<double> &prio,
                std::vector<int> &order) {
  order.clear();
  if (prio.empty()) return;
  const int nu = (int)base.size() - 1;
  std::vector<int> us(nu);
  std::iota(us.begin(), us.end(), 0);
  std::stable_sort(us.begin(), us.end(), [&](int a, int b) { return prio[a] > prio[b]; });
  std::vector<int> seq;
  seq.reserve(base[nu]);
  for (int u : us)
    for (long i = base[u]; i < base[u + 1]; ++i) seq.push_back((int)i);
  const long total = base[nu];
  order.resize(total);
  const long per = total / 8;
  for (long L = 0; L < total; ++L) {
    long r = L;
    if (L < per * 8) r = (L % 8) * per + L / 8;
    order[L] = seq[r];
  }
}

enum ItemKind { K_BASIS, K_FUNC, K_WMAT, K_DENS, K_POT, K_WBASIS };

long unit_items(const UnitD &U, ItemKind k, int tf) {
  switch (k) {
    case K_BASIS:
    case K_WBASIS: return U.nbi;
    case K_FUNC: return items_functional(U.Mc);
    case K_WMAT: return items_wmat(U.Mc, U.NP);
    case K_DENS: return U.ndi;
    default: return U.npi;
  }
}

}  // namespace

// Features (PGXC_NFEATURES) and counted flops of the contraction items of
// one unit, in the items' order.  cols: the columns of the tile's items (density)
// or the functions of a chunk (potential); kact: K length left after screening (functions of a
// density item: the tile's own, or in split-BF16 their runs; points of a
// potential item); kdense: the dense K length.
static void unit_item_features(const pgxc_ctx *c, int step, ItemKind kind, int precision,
                               std::vector<double> &feat, std::vector<double> &flops) {
  const int tf = c->pt;
  const int var = precision == PGXC_PREC_FP64 ? c->var[0] : precision == PGXC_PREC_FP32 ? c->var[1] : 0;
  auto push = [&](int kd, double cols, double kact, double kdense, bool active, double fl) {
    const double f[PGXC_NFEATURES] = {(double)kd,
                                      precision == PGXC_PREC_FP64 ? 1.0 : 0.0,
                                      precision == PGXC_PREC_FP32 ? 1.0 : 0.0,
                                      precision == PGXC_PREC_BF16X3 ? 1.0 : 0.0,
                                      cols / 128.0,
                                      std::log2(1.0 + kact) / 16.0,
                                      std::log2(1.0 + kdense) / 16.0,
                                      active ? 1.0 : 0.0,
                                      var / 2.0};
    feat.insert(feat.end(), f, f + PGXC_NFEATURES);
    flops.push_back(fl);
  };
  if (kind == K_DENS) {
    const long T0 = (long)step * c->Mc / kScreenTile;
    for (long i = c->h_di_off[step]; i < c->h_di_off[step + 1]; ++i) {
      const uint32_t e = c->h_di[(size_t)i];
      const long T = T0 + (e >> 8);
      const int nf = c->h_tf_off[(size_t)T + 1] - c->h_tf_off[(size_t)T];
      // The columns as the kernels take them: n chunks of cc (at most dcols), per an
      // item.  Feature and cost are the same for all items of a tile, its share and
      // its flops over its items, not those of what is left for the last one: items
      // of equal cost keep their natural order in a queue, and a tile's items then
      // read its values together.  (H2O)32 in FP64, counted flops 15.6 -> 15.3 ms,
      // the model 15.8 -> 15.5.
      const int dcols = precision == PGXC_PREC_BF16X3 ? c->icols : kPartCols, per = c->icols / dcols;
      const int n = (nf + dcols - 1) / dcols, cc = 16 * (((nf + 15) / 16 + n - 1) / n);
      const double cols = (double)nf / ((n + per - 1) / per);
      const double K = precision == PGXC_PREC_BF16X3 ? kRun * (c->h_tl_off[(size_t)T + 1] - c->h_tl_off[(size_t)T]) : nf;
      push(0, std::min(per, n) * cc, K, c->NP, true, 2.0 * kScreenTile * cols * K);
    }
  } else {
    const long spts = c->Mc / c->nsp;
    std::vector<uint32_t> cm;  // per chunk of the current split: its tiles
    long last = -1;
    for (long i = c->h_pi_off[step]; i < c->h_pi_off[step + 1]; ++i) {
      const uint32_t e = c->h_pi[(size_t)i];
      const long S = (long)step * c->nsp + (e >> 20);
      const int ci = (int)((e >> 10) & 1023), cj = (int)(e & 1023);
      const int so = c->h_su_off[(size_t)S], nu = c->h_su_off[(size_t)S + 1] - so;
      if (S != last) {
        cm.assign((size_t)(nu + tf - 1) / tf, 0u);
        for (int f = 0; f < nu; ++f) cm[(size_t)f / tf] |= c->h_sumask[(size_t)so + f];
        last = S;
      }
      const long cnt = __builtin_popcount(cm[(size_t)ci] & cm[(size_t)cj]) * (long)kScreenTile;
      const double rows = (double)std::min(tf, nu - ci * tf);
      const double cols = (double)std::min(tf, nu - cj * tf);
      push(1, tf, (double)cnt, (double)spts, cnt > 0, 2.0 * rows * cols * cnt);
    }
  }
}

// Make (or reuse) the plan of a set of molecules for one configuration.  A plan
// that could not be made whole leaves the slot empty.
static int get_plan(std::vector<pgxc_ctx *> &mols, uint32_t functional, int precision,
                    const std::vector<int> &incr, const std::vector<double> &unit_prio,
                    long order_version, const Sched &sc, Plan *&slot, pgxc_ctx *errc,
                    int energy = 0) {
  const int smode = sc.model ? sc.mode : std::min(sc.mode, (int)PGXC_SCHED_ANALYTIC);
  std::vector<int> lanes, spins;
  std::vector<WorkBufs> bufs;  // a call on a member alone may have moved them
  for (auto *c : mols) {
    lanes.push_back(c->nlanes);
    spins.push_back(c->ispin);
    bufs.push_back({c->phi_base, c->W, c->ispin == 2 ? c->beta.W : nullptr, c->phi_stride, c->phi_lane, c->w_lane,
                    c->skip_basis});
  }
  if (slot && slot->functional == functional && slot->precision == precision &&
      slot->incr == incr && slot->lanes == lanes && slot->spins == spins && slot->bufs == bufs &&
      slot->energy == energy &&
      slot->order_version == order_version &&
      slot->sched_mode == smode &&
      slot->log == sc.log && slot->model == sc.model &&
      slot->model_version == costmodel_version(sc.model))
    return PGXC_OK;
  free_plan(slot);
  std::unique_ptr<Plan> made(new Plan());
  Plan *plan = made.get();
  plan->functional = functional;
  plan->precision = precision;
  plan->incr = incr;
  plan->lanes = lanes;
  plan->spins = spins;
  plan->bufs = bufs;
  plan->energy = energy;
  plan->order_version = order_version;
  plan->sched_mode = smode;
  plan->log = sc.log;
  plan->model = sc.model;
  plan->model_version = costmodel_version(sc.model);
  {
    int khz = 0;
    if (hipDeviceGetAttribute(&khz, hipDeviceAttributeWallClockRate, errc->device) != hipSuccess ||
        khz <= 0)
      khz = 100000;
    plan->tick_us = 1000.0 / khz;
  }
  const bool queues = smode != PGXC_SCHED_STATIC;
  const int nm = (int)mols.size();
  int nsteps = 0;
  for (auto *c : mols) nsteps = std::max(nsteps, c->nchunks);
  // Two lanes (step k on stream k & 1) only when every member of more than
  // one chunk asked for two.  A member's chunk k then takes the work buffers
  // of the lane whose stream runs it, so two chunks that share buffers never
  // run at the same time; a member of one chunk only has lane 0.
  int plan_lanes = 0;
  for (auto *c : mols)
    if (c->nchunks > 1) plan_lanes = plan_lanes ? std::min(plan_lanes, c->nlanes) : c->nlanes;
  if (plan_lanes < 1 || nsteps < 2) plan_lanes = 1;
  auto lanes_of = [plan_lanes](const pgxc_ctx *c) { return c->nchunks > 1 ? plan_lanes : 1; };

  // host image of everything that goes to the device
  std::vector<char> img;
  auto put = [&](const void *src, size_t bytes) {  // src == nullptr: zeros
    const size_t off = (size_t)round_up((long)img.size(), 256);
    img.resize(off + std::max<size_t>(bytes, 1));
    if (bytes && src) memcpy(img.data() + off, src, bytes);
    return off;
  };
  struct Pending {
    size_t units_off = 0, base_off = 0, order_off = 0, qbeg_off = 0, ctr_off = 0, tlog_off = 0;
    int nu = 0;
    long total = 0;
    bool has_order = false, has_queues = false, has_log = false;
    size_t frow = 0;  // first feature row of the list's items
    int lmax = 0;     // basis lists: the largest angular momentum of their molecules
  };
  std::vector<double> flops;  // counted flops per feature row
  size_t plan_ctr_off_tmp = 0;
  auto stage = [&](const std::vector<UnitD> &us, const std::vector<int> &um, ItemKind kind,
                   int tf, int step) {
    Pending P;
    P.nu = (int)us.size();
    std::vector<long> base(us.size() + 1, 0);
    for (size_t i = 0; i < us.size(); ++i) base[i + 1] = base[i] + unit_items(us[i], kind, tf);
    P.total = base.back();
    P.units_off = put(us.data(), sizeof(UnitD) * us.size());
    P.base_off = put(base.data(), sizeof(long) * base.size());
    const bool contr = kind == K_DENS || kind == K_POT;
    if (contr && (queues || sc.log) && P.total > 0) {
      P.frow = plan->feat.size() / PGXC_NFEATURES;
      for (int m : um) unit_item_features(mols[m], step, kind, precision, plan->feat, flops);
    }
    const bool wide = kind == K_DENS && precision == PGXC_PREC_BF16X3 && !um.empty() && mols[um[0]]->icols > 128;
    if (contr && queues && P.total > (wide && plan_lanes == 1 ? kQueueItemsWide : kQueueItems)) {
      P.has_queues = true;  // queue bounds filled in once every cost is known
    } else {
      std::vector<double> pr;
      if (!unit_prio.empty())
        for (int m : um) pr.push_back(unit_prio[m]);
      std::vector<int> order;
      make_order(base, pr, order);
      P.has_order = !order.empty();
      if (P.has_order) P.order_off = put(order.data(), sizeof(int) * order.size());
    }
    if (contr && sc.log && P.total > 0) {
      P.has_log = true;
      P.tlog_off = put(nullptr, sizeof(uint32_t) * P.total);
    }
    return P;
  };
  // per step: basis, func, wmat, dens lists, pot lists, func2, wmat2
  std::vector<std::vector<Pending>> pend(nsteps);
  for (int k = 0; k < nsteps; ++k) {
    std::vector<UnitD> units;
    std::vector<int> umol, uspin;
    for (int m = 0; m < nm; ++m) {
      pgxc_ctx *c = mols[m];
      if (k >= c->nchunks) continue;
      const long p0 = (long)k * c->Mc;
      UnitD U;
      memset(&U, 0, sizeof(U));
      U.gx = c->grid + p0;
      U.gy = c->grid + c->npad + p0;
      U.gz = c->grid + 2 * c->npad + p0;
      U.gw = c->grid + 3 * c->npad + p0;
      U.atoms = c->atoms;
      U.shells = c->shells;
      U.ranges = c->ranges;
      U.ratoms = c->ratoms;
      U.n_ranges = c->n_ranges;
      U.tabd = c->tabd;
      U.tabf = c->tabf;
      const int lane = k % lanes_of(c);  // work buffers of chunk k: its stream's lane
      U.phi = (char *)c->phi_base + (c->phi_stride ? (size_t)k * c->phi_stride : (size_t)lane * c->phi_lane);
      U.W = (char *)c->W + (size_t)lane * c->w_lane;
      U.D = c->D;
      U.part = c->part + (size_t)lane * c->nparts * 4 * c->Mc;
      U.coef = c->coef + (size_t)lane * 4 * c->Mc;
      U.state = c->state + p0;
      U.epart = c->epart + 2 * (p0 / kThreads);
      U.eterm = c->eterm + 5 * (p0 / kThreads);
      U.Hc = c->Hc;
      U.ho = c->ho + ((long)(lanes_of(c) - 1) * c->nchunks + k) * c->nsp;
      U.Mc = c->Mc;
      U.npad = c->npad;
      U.n_atoms = c->n_atoms;
      U.NP = c->NP;
      U.nsplit = c->nsp;
      U.incremental = incr[m];
      U.mask = functional;
      U.icols = c->icols;
      U.dcols = precision == PGXC_PREC_BF16X3 ? c->icols : kPartCols;
      U.ditems = c->di + c->h_di_off[k];
      U.pitems = c->pi + c->h_pi_off[k];
      U.ndi = c->h_di_off[k + 1] - c->h_di_off[k];
      U.npi = c->h_pi_off[k + 1] - c->h_pi_off[k];
      U.tl_off = c->tl_off + p0 / kScreenTile;
      U.tl = c->tl;
      U.tf_off = c->tf_off + p0 / kScreenTile;
      U.tfl = c->tfl;
      U.tfb = c->tfb + (p0 / kScreenTile) * c->nwf;
      U.tlm = c->tlm;
      U.nwf = c->nwf;
      U.su_off = c->su_off + (long)k * c->nsp;
      U.su = c->su;
      U.sumask = c->sumask;
      U.bitems = c->bi + c->h_bi_off[k];
      U.bflags = c->bfl + 2 * c->h_bi_off[k];
      U.nbi = c->h_bi_off[k + 1] - c->h_bi_off[k];
      if (c->ispin == 2) {  // the beta spin's unit: same points and basis values
        UnitD B = U;
        B.W = (char *)c->beta.W + (size_t)lane * c->w_lane;
        B.D = c->beta.D;
        B.part = c->beta.part + (size_t)lane * c->nparts * 4 * c->Mc;
        B.coef = c->beta.coef + (size_t)lane * 4 * c->Mc;
        B.state = c->beta.state + p0;
        B.Hc = c->beta.Hc;
        U.part2 = B.part;
        U.coef2 = B.coef;
        U.state2 = B.state;
        U.W2 = B.W;
        units.push_back(U);
        umol.push_back(m);
        uspin.push_back(0);
        units.push_back(B);
        umol.push_back(m);
        uspin.push_back(1);
      } else {
        units.push_back(U);
        umol.push_back(m);
        uspin.push_back(0);
      }
    }
    // the units of one spin (0: closed-shell and alpha units, 1: beta)
    // meeting a condition on the molecule
    auto pick = [&](int spin, auto cond, std::vector<UnitD> &out, std::vector<int> &om) {
      for (size_t i = 0; i < units.size(); ++i)
        if (uspin[i] == spin && cond(mols[umol[i]])) {
          out.push_back(units[i]);
          om.push_back(umol[i]);
        }
    };
    {  // molecules whose basis values are cached skip the basis stage
      std::vector<UnitD> bu;
      std::vector<int> bm;
      for (size_t i = 0; i < units.size(); ++i)
        if (uspin[i] == 0 && !mols[umol[i]]->skip_basis) {
          bu.push_back(units[i]);
          bm.push_back(umol[i]);
        }
      pend[k].push_back(stage(bu, bm, K_BASIS, 0, k));
      for (int m : bm) pend[k].back().lmax = std::max(pend[k].back().lmax, mols[m]->lmax);
    }
    {
      std::vector<UnitD> fu;
      std::vector<int> fm;
      pick(0, [](const pgxc_ctx *c) { return c->ispin == 1; }, fu, fm);
      pend[k].push_back(stage(fu, fm, K_FUNC, 0, k));
    }
    // W: the basis evaluated again over the basis items (test switch
    // PGXC_W_READ=1: the stored values read back instead, the same bits)
    const bool wb = !getenv("PGXC_W_READ");
    plan->wbasis = wb ? 1 : 0;
    const ItemKind wkind = wb ? K_WBASIS : K_WMAT;
    {  // closed-shell units; the open-shell ones in wmat2 below
      std::vector<UnitD> wu;
      std::vector<int> wm;
      pick(0, [](const pgxc_ctx *c) { return c->ispin == 1; }, wu, wm);
      pend[k].push_back(stage(wu, wm, wkind, 0, k));
      for (int m : wm) pend[k].back().lmax = std::max(pend[k].back().lmax, mols[m]->lmax);
    }
    const int cls = precision == PGXC_PREC_FP64 ? 0 : 1;
    const bool x3 = precision == PGXC_PREC_BF16X3;
    for (int kind = 0; kind < 2; ++kind)
      for (int li = 0; li < kLists; ++li) {
        const int t = li / kNumVariants, v = li % kNumVariants;
        std::vector<UnitD> sub;
        std::vector<int> subm;
        for (size_t i = 0; i < units.size(); ++i) {
          const pgxc_ctx *c = mols[umol[i]];
          const bool mine = kind == 0 && x3 ? li == (c->icols == 128 ? 0 : 1)  // split-BF16: by item width
                                            : (kind == 0 ? c->tf : c->pt) == kTiles[t] && c->var[cls] == v;
          if (mine) {
            sub.push_back(units[i]);
            subm.push_back(umol[i]);
          }
        }
        pend[k].push_back(stage(sub, subm, kind == 0 ? K_DENS : K_POT, kTiles[t], k));
      }
    {  // spin functional over the alpha units of open-shell molecules
      std::vector<UnitD> fu;
      std::vector<int> fm;
      pick(0, [](const pgxc_ctx *c) { return c->ispin == 2; }, fu, fm);
      pend[k].push_back(stage(fu, fm, K_FUNC, 0, k));
      pend[k].push_back(stage(fu, fm, wkind, 0, k));  // both spins' W per alpha unit
      for (int m : fm) pend[k].back().lmax = std::max(pend[k].back().lmax, mols[m]->lmax);
    }
  }
  // queue bounds: each list's positions (natural order, so neighbouring items
  // keep sharing operand panels) cut into kQueues runs of equal predicted cost
  {
    std::vector<double> cost = flops;
    const size_t nrow = flops.size();
    if (smode == PGXC_SCHED_MODEL && nrow) {
      if (costmodel_features(sc.model) != PGXC_NFEATURES)
        return fail(errc, PGXC_ERR_ARG, "cost model does not take PGXC_NFEATURES features");
      std::vector<double> pred(nrow);
      int rc = pgxc_costmodel_predict(sc.model, plan->feat.data(), (int64_t)nrow, pred.data());
      if (rc) return fail(errc, rc, std::string("cost model: ") + pgxc_costmodel_last_error(sc.model));
      for (size_t i = 0; i < nrow; ++i) cost[i] = std::exp(std::min(pred[i], 50.0));
    } else {
      for (size_t i = 0; i < nrow; ++i) cost[i] = flops[i] + 1.0;
    }
    long nq = 0;
    for (auto &pk : pend)
      for (auto &P : pk) nq += P.has_queues;
    std::vector<int> zeros((size_t)std::max<long>(1, nq * kQueues), 0);
    const size_t ctr0 = put(zeros.data(), sizeof(int) * zeros.size());
    plan->nctr = nq * kQueues;
    long qi = 0;
    for (auto &pk : pend)
      for (auto &P : pk) {
        if (!P.has_queues) continue;
        double tot = 0.0;
        for (long i = 0; i < P.total; ++i) tot += cost[P.frow + i];
        long qb[kQueues + 1];
        qb[0] = 0;
        double acc = 0.0;
        int q = 1;
        for (long i = 0; i < P.total && q < kQueues; ++i) {
          acc += cost[P.frow + i];
          while (q < kQueues && acc >= tot * q / kQueues) qb[q++] = i + 1;
        }
        while (q <= kQueues) qb[q++] = P.total;
        P.qbeg_off = put(qb, sizeof(qb));
        // within a queue the costliest items go first, so its last items,
        // which set when the stage ends, are the cheapest; equal costs keep
        // their natural order (the items of one density tile stay together)
        std::vector<int> order((size_t)P.total);
        std::iota(order.begin(), order.end(), 0);
        for (int k = 0; k < kQueues; ++k)
          std::stable_sort(order.begin() + qb[k], order.begin() + qb[k + 1], [&](int a, int b) {
            return cost[P.frow + a] > cost[P.frow + b];
          });
        P.has_order = true;
        P.order_off = put(order.data(), sizeof(int) * order.size());
        P.ctr_off = ctr0 + sizeof(int) * kQueues * qi++;
      }
    plan_ctr_off_tmp = ctr0;
  }
  // operand preparation and packing per molecule and spin
  std::vector<PackD> packs;
  for (int m = 0; m < nm; ++m) {
    pgxc_ctx *c = mols[m];
    for (int sp = 0; sp < c->ispin; ++sp) {
      PackD Q;
      memset(&Q, 0, sizeof(Q));
      Q.HS = sp ? c->beta.HS : c->HS;
      Q.Vout = sp ? c->beta.Vout : c->Vout;
      Q.Vstate = sp ? c->beta.Vstate : c->Vstate;
      Q.P = sp ? c->beta.P : c->P;
      Q.Pref = sp ? c->beta.Pref : c->Pref;
      Q.D = sp ? c->beta.D : c->D;
      Q.fpos = c->d_fpos;
      Q.n = c->nbas;
      Q.NP = c->NP;
      Q.nseg = c->hflush ? lanes_of(c) : c->nseg;
      Q.incremental = incr[m];
      packs.push_back(Q);
    }
  }
  const int npack = (int)packs.size();
  std::vector<long> pbase(npack + 1, 0), qbase(npack + 1, 0);
  for (int q = 0; q < npack; ++q) {
    const PackD &Q = packs[q];
    const long npk = Q.n * (Q.n + 1) / 2;
    pbase[q + 1] = pbase[q] + (npk + kThreads - 1) / kThreads;
    qbase[q + 1] = qbase[q] + (Q.NP * Q.NP + kThreads - 1) / kThreads;
  }
  // sums of the potential partials: after the steps that fill a lane's share or
  // end the lane (hflush), else all at the end, in segments of the splits
  auto fold_of = [&](const pgxc_ctx *c, int sp) {
    FoldD F;
    memset(&F, 0, sizeof(F));
    F.Hc = sp ? c->beta.Hc : c->Hc;
    F.ho = c->ho + (long)(lanes_of(c) - 1) * c->nchunks * c->nsp;
    F.su_off = c->su_off;
    F.pos = c->pos;
    F.rbits = c->rbits;
    F.out = sp ? c->beta.HS : c->HS;
    F.NP = c->NP;
    F.nsplit = c->nsp;
    F.bytes_c = (c->nsp + 7) / 8;
    F.nbytes = F.bytes_c * c->nchunks;
    return F;
  };
  struct FoldOff {
    size_t d = 0, base = 0;
    int n = 0;
    long total = 0;
  };
  auto put_folds = [&](const std::vector<FoldD> &fs) {
    FoldOff o;
    std::vector<long> fb(fs.size() + 1, 0);
    for (size_t i = 0; i < fs.size(); ++i) {
      const long nb = fs[i].NP / 32;
      fb[i + 1] = fb[i] + nb * (nb + 1) / 2;
    }
    o.n = (int)fs.size();
    o.total = fb.back();
    o.d = put(fs.data(), sizeof(FoldD) * fs.size());
    o.base = put(fb.data(), sizeof(long) * fb.size());
    return o;
  };
  std::vector<FoldD> last;
  std::vector<std::vector<FoldD>> flush((size_t)nsteps);
  for (int m = 0; m < nm && !energy; ++m) {
    const pgxc_ctx *c = mols[m];
    for (int sp = 0; sp < c->ispin; ++sp) {
      FoldD F = fold_of(c, sp);
      if (!c->hflush) {
        F.step = 1;
        F.nchunks = c->nchunks;
        F.nseg = c->nseg;
        double *out = F.out;
        for (F.seg = 0; F.seg < F.nseg; ++F.seg) {
          F.out = out + (size_t)F.seg * c->NP * c->NP;
          last.push_back(F);
        }
        continue;
      }
      F.step = lanes_of(c);
      F.nseg = 1;
      double *out = F.out;
      for (int ln = 0; ln < F.step; ++ln) {
        F.out = out + (size_t)ln * c->NP * c->NP;
        F.chunk0 = ln;
        F.acc = 0;
        for (int k = ln; k < c->nchunks; k += F.step) {
          if (!c->h_flush[F.step - 1][(size_t)k]) continue;
          F.nchunks = (k - F.chunk0) / F.step + 1;
          flush[(size_t)k].push_back(F);
          F.chunk0 = k + F.step;
          F.acc = 1;
        }
      }
    }
  }
  const FoldOff last_off = put_folds(last);
  std::vector<FoldOff> flush_off;
  for (int k = 0; k < nsteps; ++k) flush_off.push_back(put_folds(flush[(size_t)k]));
  plan->nmol = npack;
  const size_t pack_off = put(packs.data(), sizeof(PackD) * npack);
  const size_t pb_off = put(pbase.data(), sizeof(long) * pbase.size());
  const size_t qb_off = put(qbase.data(), sizeof(long) * qbase.size());
  HIPCHK(errc, hipMalloc((void **)&plan->blob, std::max<size_t>(img.size(), 256)));
  HIPCHK(errc, hipMemcpy(plan->blob, img.data(), img.size(), hipMemcpyHostToDevice));
  char *B = plan->blob;
  plan->d_ctr = (int *)(B + plan_ctr_off_tmp);
  auto mk = [&](const Pending &P) {
    StageList L{};
    L.units = (const UnitD *)(B + P.units_off);
    L.nu = P.nu;
    L.base = (const long *)(B + P.base_off);
    L.order = P.has_order ? (const int *)(B + P.order_off) : nullptr;
    L.total = P.total;
    L.ctr = P.has_queues ? (int *)(B + P.ctr_off) : nullptr;
    L.qbeg = P.has_queues ? (const long *)(B + P.qbeg_off) : nullptr;
    L.tlog = P.has_log ? (uint32_t *)(B + P.tlog_off) : nullptr;
    L.lmax = P.lmax;
    if (P.has_log) plan->logs.push_back({L.tlog, P.total});
    return L;
  };
  auto mkf = [&](const FoldOff &o) {
    FoldList f;
    f.d = (const FoldD *)(B + o.d);
    f.base = (const long *)(B + o.base);
    f.n = o.n;
    f.total = o.total;
    return f;
  };
  plan->steps.resize(nsteps);
  for (int k = 0; k < nsteps; ++k) {
    StepPlan &S = plan->steps[k];
    S.basis = mk(pend[k][0]);
    S.func = mk(pend[k][1]);
    S.wmat = mk(pend[k][2]);
    for (int li = 0; li < kLists; ++li) S.dens[li] = mk(pend[k][3 + li]);
    for (int li = 0; li < kLists; ++li) S.pot[li] = mk(pend[k][3 + kLists + li]);
    S.func2 = mk(pend[k][3 + 2 * kLists]);
    S.wmat2 = mk(pend[k][4 + 2 * kLists]);
    S.nunits = pend[k][0].nu;
    S.flush = mkf(flush_off[(size_t)k]);
  }
  plan->fold = mkf(last_off);
  plan->nlanes = plan_lanes;
  plan->d_pack = (PackD *)(B + pack_off);
  plan->d_pack_base = (long *)(B + pb_off);
  plan->d_prep_base = (long *)(B + qb_off);
  plan->pack_total = pbase[npack];
  plan->prep_total = qbase[npack];
  slot = made.release();
  return PGXC_OK;
}

// Item log of a plan's last build: features and microseconds per item.
static int64_t read_item_log(const Plan *pl, hipStream_t s, double *features, double *us,
                             int64_t cap) {
  if (!pl || !pl->log) return 0;
  int64_t n = 0;
  for (auto &lg : pl->logs) n += lg.second;
  if (!features || !us || cap < n) return n;
  if (hipStreamSynchronize(s) != hipSuccess) return -PGXC_ERR_HIP;
  int64_t row = 0;
  std::vector<uint32_t> t;
  for (auto &lg : pl->logs) {
    t.resize((size_t)lg.second);
    if (hipMemcpy(t.data(), lg.first, sizeof(uint32_t) * lg.second, hipMemcpyDeviceToHost) != hipSuccess)
      return -PGXC_ERR_HIP;
    for (long i = 0; i < lg.second; ++i, ++row) us[row] = t[(size_t)i] * pl->tick_us;
  }
  memcpy(features, pl->feat.data(), sizeof(double) * PGXC_NFEATURES * n);
  return n;
}

static int check_sched(int32_t mode, const pgxc_costmodel *model) {
  if (mode < PGXC_SCHED_STATIC || mode > PGXC_SCHED_MODEL) return PGXC_ERR_ARG;
  if (mode == PGXC_SCHED_MODEL && !model) return PGXC_ERR_ARG;
  return PGXC_OK;
}

// Events of a timed build: kEvStart / kEvPack / kEvEnd bracket the build and
// its packing; step k of the plan records five more from kEvStep + 5 k on
// (before basis, after basis, after the density contraction, after the
// functional + W, after the potential contraction).  Nothing waits on them
// until the build has ended, so timing adds no host synchronisation.
constexpr int kEvStart = 0, kEvPack = 1, kEvEnd = 2, kEvStep = 3;

// Launch a plan, recording the events above when ev is given.  Chunk k runs
// on lane k % 2 of a two-lane plan: stream s or s2, each lane with its own
// work buffers, so one chunk's stages (and the ends of its launches) overlap
// the next chunk's; s2 starts after the operand preparation (fork) and the
// fold waits for its last chunk (join).
template <typename T>
static void launch_plan(hipStream_t s, hipStream_t s2, hipEvent_t fork, hipEvent_t join,
                        const Plan &pl, bool gga, std::vector<hipEvent_t> *ev) {
  const bool x3 = pl.precision == PGXC_PREC_BF16X3;
  const bool two = pl.nlanes > 1 && pl.steps.size() > 1;
  launch_prep(s, pl.d_pack, pl.nmol, pl.d_prep_base, pl.prep_total,
              x3 ? 2 : std::is_same<T, double>::value ? 0 : 1, pl.d_ctr, (int)pl.nctr);
  if (two) {
    (void)hipEventRecord(fork, s);
    (void)hipStreamWaitEvent(s2, fork, 0);
  }
  for (size_t k = 0; k < pl.steps.size(); ++k) {
    const StepPlan &S = pl.steps[k];
    const hipStream_t t = two && (k & 1) ? s2 : s;
    hipEvent_t *E = ev ? ev->data() + kEvStep + 5 * k : nullptr;
    if (E) (void)hipEventRecord(E[0], t);
    launch_basis<T>(t, gga, S.basis);
    if (E && S.basis.total) (void)hipEventRecord(E[1], t);  // cached values: no stage, no mark
    for (int li = 0; li < kLists; ++li) {
      const int v = li % kNumVariants;
      if constexpr (std::is_same<T, float>::value) {
        if (x3) {
          launch_density_bf16x3(t, gga, li == 0 ? 128 : 256, S.dens[li]);
          continue;
        }
      }
      launch_density<T>(t, gga, v, S.dens[li]);
    }
    if (E) (void)hipEventRecord(E[2], t);
    if (pl.energy) {
      launch_energy(t, gga, false, S.func);
      launch_energy(t, gga, true, S.func2);
      continue;
    }
    launch_functional(t, gga, S.func);
    launch_functional_spin(t, gga, S.func2);
    if (pl.wbasis) {
      launch_wbasis<T>(t, gga, x3, false, S.wmat);
      launch_wbasis<T>(t, gga, x3, true, S.wmat2);
    } else {
      launch_wmat<T>(t, gga, x3, false, S.wmat);
      launch_wmat<T>(t, gga, x3, true, S.wmat2);
    }
    if (E) (void)hipEventRecord(E[3], t);
    for (int li = 0; li < kLists; ++li) {
      const int tf = kTiles[li / kNumVariants], v = li % kNumVariants;
      if constexpr (std::is_same<T, float>::value) {
        if (x3) {
          launch_potential_bf16x3(t, tf, S.pot[li]);
          continue;
        }
      }
      launch_potential<T>(t, tf, v, S.pot[li]);
    }
    if (E) (void)hipEventRecord(E[4], t);
    launch_fold(t, S.flush.d, S.flush.n, S.flush.base, S.flush.total);
  }
  if (two) {
    (void)hipEventRecord(join, s2);
    (void)hipStreamWaitEvent(s, join, 0);
  }
  if (pl.energy) return;
  if (ev) (void)hipEventRecord((*ev)[kEvPack], s);
  launch_fold(s, pl.fold.d, pl.fold.n, pl.fold.base, pl.fold.total);
  launch_pack(s, pl.d_pack, pl.nmol, pl.d_pack_base, pl.pack_total, pl.d_prep_base, pl.prep_total);
  if (ev) (void)hipEventRecord((*ev)[kEvEnd], s);
}

// Bytes of basis caches held per device by all contexts of the process.
static std::mutex g_cache_mu;
static std::map<int, size_t> g_cache_bytes;

// bytes of basis values per (function, point): value and gradient planes
static size_t phi_elem_bytes(size_t elem) { return 4 * elem; }

// Test switch PGXC_POISON_BASIS=1: basis buffers, when they get their first
// contents (allocation, or the zeroing of the lane buffers at a change of
// precision), are filled with NaN bytes wherever a build writes basis values
// (rows of the real functions), so a stage
// reading a block the basis stage left unwritten turns the results into NaN.
static hipError_t poison_basis(const pgxc_ctx *c, void *base, size_t elem, size_t per_buf,
                               size_t nbuf, hipStream_t s) {
  const char *pz = getenv("PGXC_POISON_BASIS");
  if (!pz || pz[0] != '1') return hipSuccess;
  const size_t rows = (size_t)c->nbas * c->Mc, plane = (size_t)c->NP * c->Mc;
  hipError_t e = hipSuccess;
  for (size_t k = 0; k < nbuf && e == hipSuccess; ++k) {
    char *b = (char *)base + k * per_buf;
    for (int pl = 0; pl < 4 && e == hipSuccess; ++pl)
      e = hipMemsetAsync(b + pl * plane * elem, 0xff, rows * elem, s);
  }
  return e;
}

// grad: the build reads the gradient planes of the basis values (GGA)
static int ensure_work(pgxc_ctx *c, size_t elem, hipStream_t s, bool grad) {
  const size_t need_phi = phi_elem_bytes(elem) * (size_t)c->NP * c->Mc;
  const size_t need_w = (size_t)c->NP * c->Mc * elem * c->nlanes_cap;
  c->w_lane = (size_t)c->NP * c->Mc * elem;
  if (c->w_bytes < need_w) {
    dfree(c->W);
    c->W = nullptr;
    c->w_bytes = 0;
    HIPCHK(c, hipMalloc(&c->W, need_w));
    c->w_bytes = need_w;
  }
  if (c->ispin == 2 && c->beta.w_bytes < need_w) {
    dfree(c->beta.W);
    c->beta.W = nullptr;
    c->beta.w_bytes = 0;
    HIPCHK(c, hipMalloc(&c->beta.W, need_w));
    c->beta.w_bytes = need_w;
  }
  // basis cache: every chunk's values, when they take at most a quarter of
  // the device, leave 32 GiB free, and the caches of all contexts on the
  // device stay within half of it (the members of a batch keep room for their
  // own work buffers)
  const int e = elem == 8 ? 0 : 1;
  if (!c->cache_off && !c->phic[e] && !c->phic_failed[e]) {
    const size_t need = need_phi * (size_t)c->nchunks;
    size_t fr = 0, tot = 0;
    c->phic_failed[e] = 1;
    std::lock_guard<std::mutex> lk(g_cache_mu);
    size_t &held = g_cache_bytes[c->device];
    if (hipMemGetInfo(&fr, &tot) == hipSuccess && need <= tot / 4 && need + (32ull << 30) <= fr &&
        held + need <= tot / 2 && hipMalloc(&c->phic[e], need) == hipSuccess) {
      c->phic_failed[e] = 0;
      c->phic_bytes[e] = need;
      held += need;
      HIPCHK(c, poison_basis(c, c->phic[e], elem, need_phi, c->nchunks, s));
      c->phic_valid[e] = 0;
      c->phic_grad[e] = 0;
    } else {
      c->phic[e] = nullptr;
      (void)hipGetLastError();
    }
  }
  c->phi_lane = need_phi;
  if (!c->phic[e]) {  // one chunk buffer per lane, rewritten by every build
    if (c->phi_bytes < need_phi * c->nlanes_cap) {
      dfree(c->phi);
      c->phi = nullptr;
      c->phi_bytes = 0;
      HIPCHK(c, hipMalloc(&c->phi, need_phi * c->nlanes_cap));
      c->phi_bytes = need_phi * c->nlanes_cap;
      c->phi_elem = 0;
    }
    // (no stage reads what this build's basis stage does not write: neither the
    // rows past nbas nor what a build of another precision left)
    if (c->phi_elem != elem) {
      c->phi_elem = elem;
      HIPCHK(c, poison_basis(c, c->phi, elem, need_phi, c->nlanes_cap, s));
    }
  }
  void *base = c->phic[e] ? c->phic[e] : c->phi;
  const size_t stride = c->phic[e] ? need_phi : 0;
  // an LDA pass writes only the value planes: a GGA build after it evaluates again
  c->phi_base = base;
  c->phi_stride = stride;
  c->skip_basis = c->phic[e] && c->phic_valid[e] && (c->phic_grad[e] || !grad);
  return PGXC_OK;
}

// after a build: the cache of this element type now holds valid values
static void mark_basis_cached(pgxc_ctx *c, size_t elem, bool grad) {
  const int e = elem == 8 ? 0 : 1;
  if (c->phic[e]) {
    c->phic_valid[e] = 1;
    if (grad) c->phic_grad[e] = 1;
  }
}

static int validate_build(pgxc_ctx *c, uint32_t functional, int32_t precision, int &incr) {
  if (!c) return PGXC_ERR_ARG;
  if (functional == 0 || (functional & ~kSupported))
    return fail(c, PGXC_ERR_UNSUPPORTED, "functional mask has terms other than XAlpha, PWLDAc, PBEx, PBEc");
  if ((functional & PGXC_XC_PBEC) && !(functional & PGXC_XC_PWLDAC))
    return fail(c, PGXC_ERR_ARG, "PBEc needs the PW92 LDA correlation it is built on (PWLDAc)");
  if (precision != PGXC_PREC_FP64 && precision != PGXC_PREC_FP32 && precision != PGXC_PREC_BF16X3)
    return fail(c, PGXC_ERR_UNSUPPORTED, "precision mode " + std::to_string(precision) + " not available");
  if (!c->have_density) return fail(c, PGXC_ERR_STATE, "pgxc_build before pgxc_set_density/orbitals");
  incr = 0;
  if (c->density_mode == PGXC_DENSITY_INCREMENTAL) {
    if (!c->have_state)
      return fail(c, PGXC_ERR_STATE, "incremental density but no previous build on this context");
    if (c->state_functional != functional)
      return fail(c, PGXC_ERR_STATE, "incremental build with a functional different from the previous build");
    incr = 1;
  }
  return PGXC_OK;
}

static void set_stats(pgxc_ctx *c, int precision) {
  const double B = (double)c->npts;
  c->stats[0] = B;
  c->stats[1] = std::ceil(B / c->veclen);
  // sum over 128-point tiles of 4 B n_b^2 + 16 B n_b, n_b = functions of the
  // shells not cut off on the tile (dense: n_b = nbas)
  c->stats[2] = (c->screen ? c->flops_screened : c->flops_dense) * c->ispin;
  c->stats[3] = B * c->exps_per_point;
  // sum over the same tiles of 32 B (x, y, z, w) + 16 n_b^2 per spin (P
  // sub-block read, V partial written) + 4 s B n_b (basis values and
  // gradients materialised at s bytes per element)
  const double sb = precision == PGXC_PREC_FP64 ? 8.0 : 4.0;
  c->stats[4] = 32.0 * B + 16.0 * c->sum_n2 * c->ispin + 4.0 * sb * c->sum_bn;
}

static int collect(pgxc_ctx *c, hipStream_t s, uint32_t functional, int precision) {
  double e = 0.0, q = 0.0;
  HIPCHK(c, c->pin.fetch(s, c->epart, 2 * (size_t)c->nblk_total, [&](size_t, size_t n, const double *v) {
    for (size_t b = 0; b < n; b += 2) {
      e += v[b];
      q += v[b + 1];
    }
  }));
  c->last_exc = e;
  c->last_charge = q;
  c->have_state = 1;
  c->state_functional = functional;
  set_stats(c, precision);
  return PGXC_OK;
}

// FNV-1a style hash over 8-byte words (a shorter tail byte by byte).
static uint64_t hash_words(uint64_t h, const void *p, size_t bytes) {
  const unsigned char *b = (const unsigned char *)p;
  size_t i = 0;
  for (; i + 8 <= bytes; i += 8) {
    uint64_t w;
    memcpy(&w, b + i, 8);
    h = (h ^ w) * 1099511628211ull;
  }
  for (; i < bytes; ++i) h = (h ^ b[i]) * 1099511628211ull;
  return h;
}

// Order of n points (coordinate k of point p at xyz[k * stride + p * step])
// along a Morton curve over their bounding box (10 bits per axis), ties in
// input order.
static void morton_order(const double *xyz, long n, long stride, long step,
                         std::vector<long> &perm) {
  double lo[3], hi[3];
  for (int k = 0; k < 3; ++k) {
    lo[k] = hi[k] = xyz[(size_t)k * stride];
    for (long p = 1; p < n; ++p) {
      lo[k] = std::min(lo[k], xyz[(size_t)k * stride + (size_t)p * step]);
      hi[k] = std::max(hi[k], xyz[(size_t)k * stride + (size_t)p * step]);
    }
  }
  std::vector<std::pair<uint32_t, long>> key((size_t)n);
  for (long p = 0; p < n; ++p) {
    uint32_t code = 0;
    for (int k = 0; k < 3; ++k) {
      const double span = hi[k] - lo[k];
      const double f = span > 0 ? (xyz[(size_t)k * stride + (size_t)p * step] - lo[k]) / span : 0.0;
      const uint32_t q = (uint32_t)std::min(1023.0, std::max(0.0, f * 1023.0));
      for (int b = 0; b < 10; ++b) code |= ((q >> b) & 1u) << (3 * b + k);
    }
    key[(size_t)p] = {code, p};
  }
  std::sort(key.begin(), key.end());
  perm.resize((size_t)n);
  for (long p = 0; p < n; ++p) perm[(size_t)p] = key[(size_t)p].second;
}

// Internal order of the basis functions: shells by reach class (the radius
// sqrt(50 / alpha_min) beyond which the shell is cut off, in steps of 10 % on
// a log scale, longest reach first), then by their atom's place on a Morton
// curve, then in caller order.  Shells of one element share their exponents,
// so a class holds the like shells of neighbouring atoms: the functions that
// can be nonzero on a compact group of points fill whole runs of 8 and few
// 32-function blocks.  A shell keeps its functions together and in caller
// order.  Sets each shell's internal func_off and fpos[caller function] =
// internal position.
static void function_order(std::vector<ShellD> &sh, const double *exps, const double *atom_xyz,
                           int n_atoms, std::vector<int> &fpos) {
  const size_t ns = sh.size();
  std::vector<double> reach(ns);
  for (size_t i = 0; i < ns; ++i) {
    double amin = exps[sh[i].exp_off];
    for (int e = 1; e < sh[i].n_exp; ++e) amin = std::min(amin, exps[sh[i].exp_off + e]);
    reach[i] = std::sqrt(50.0 / amin);
  }
  std::vector<long> aperm;
  morton_order(atom_xyz, n_atoms, 1, 3, aperm);
  std::vector<int> arank(n_atoms);
  for (int r = 0; r < n_atoms; ++r) arank[aperm[r]] = r;
  std::vector<int> idx(ns);
  std::iota(idx.begin(), idx.end(), 0);
  auto cls = [&](int i) { return -(int)std::floor(std::log(reach[i]) / std::log(1.1)); };
  std::stable_sort(idx.begin(), idx.end(), [&](int a, int b) {
    if (cls(a) != cls(b)) return cls(a) < cls(b);
    return arank[sh[a].atom] < arank[sh[b].atom];
  });
  int nbas = 0;
  for (auto &d : sh) nbas += (2 * d.l + 1) * (d.n_unc + d.n_contr);
  fpos.assign(nbas, 0);
  int off = 0;
  for (int i : idx) {
    const int nf = (2 * sh[i].l + 1) * (sh[i].n_unc + sh[i].n_contr);
    for (int f = 0; f < nf; ++f) fpos[sh[i].func_off + f] = off + f;
    sh[i].func_off = off;
    off += nf;
  }
}

// Screening and work tables of the padded grid and the algorithmic work of one
// build.  k_screen marks, per 32-point group, the runs of 8 functions that can
// be nonzero there (all runs when screening is off); the host turns the marks
// into run lists per 128-point tile and per point split, [group][chunk]
// flags per split, and the work items of every chunk.
template <typename V>
static int upload(pgxc_ctx *c, V **dst, const std::vector<V> &src) {
  int rc = dalloc(c, dst, src.size());
  if (rc) return rc;
  if (!src.empty()) HIPCHK(c, hipMemcpy(*dst, src.data(), sizeof(V) * src.size(), hipMemcpyHostToDevice));
  return PGXC_OK;
}

static int alloc_partials(pgxc_ctx *c, double **Hc, double **HS) {
  int rc = dalloc(c, Hc, (size_t)c->hsize);
  if (rc) return rc;
  return dalloc(c, HS, (size_t)std::max(c->nseg, c->nlanes_cap) * c->NP * c->NP);
}

static int setup_screen(pgxc_ctx *c, const std::vector<ShellD> &sh, const double *exps, bool on) {
  const long ntp = c->npad / kScreenTile, ngr = c->npad / kGroup;
  const double n = (double)c->nbas;
  c->flops_dense = 4.0 * c->npts * n * n + 16.0 * c->npts * n;
  c->n8 = c->NP / kRun;
  c->screen = on;
  c->nw8 = (c->n8 + 31) / 32;
  const int n8 = c->n8, nw8 = c->nw8;
  if (n8 > kMaxRuns) return fail(c, PGXC_ERR_UNSUPPORTED, "more than 8192 basis functions (padded)");
  if (c->Mc / c->nsplit > 65536) return fail(c, PGXC_ERR_UNSUPPORTED, "point split above 65536 points");
  std::vector<ScreenShell> ss(sh.size());
  for (size_t i = 0; i < sh.size(); ++i) {
    double amin = exps[sh[i].exp_off];
    for (int e = 1; e < sh[i].n_exp; ++e) amin = std::min(amin, exps[sh[i].exp_off + e]);
    ss[i].amin = amin;
    ss[i].atom = sh[i].atom;
    ss[i].func_off = sh[i].func_off;
    ss[i].nfunc = (2 * sh[i].l + 1) * (sh[i].n_unc + sh[i].n_contr);
    ss[i].pad = 0;
  }
  int rc;
  if ((rc = upload(c, &c->sshells, ss))) return rc;
  if ((rc = dalloc(c, &c->nbt, ntp))) return rc;
  if ((rc = dalloc(c, &c->sig8, (size_t)ngr * nw8))) return rc;
  const int nws = (c->n_shells + 31) / 32;
  ScopedDev tmp;
  uint32_t *d_smark = nullptr;
  HIPCHK(c, hipMalloc((void **)&d_smark, sizeof(uint32_t) * (size_t)ntp * nws));
  tmp.keep(d_smark);
  launch_screen(c->stream, ntp, c->grid, c->grid + c->npad, c->grid + 2 * c->npad, c->n_atoms,
                c->atoms, c->n_shells, c->sshells, n8, c->nbt, c->sig8, d_smark);
  HIPCHK(c, hipGetLastError());
  std::vector<int> nb((size_t)ntp);
  std::vector<uint32_t> sig((size_t)ngr * nw8), smark((size_t)ntp * nws);
  HIPCHK(c, hipMemcpyAsync(nb.data(), c->nbt, sizeof(int) * ntp, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipMemcpyAsync(sig.data(), c->sig8, sizeof(uint32_t) * sig.size(), hipMemcpyDeviceToHost,
                           c->stream));
  HIPCHK(c, hipMemcpyAsync(smark.data(), d_smark, sizeof(uint32_t) * smark.size(),
                           hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (on) {
    double f = 0.0;
    for (long t = 0; t < ntp; ++t) {
      const double B = (double)std::max<long>(0, std::min<long>(kScreenTile, c->npts - t * kScreenTile));
      f += 4.0 * B * nb[(size_t)t] * nb[(size_t)t] + 16.0 * B * nb[(size_t)t];
      if (B > 0) {
        c->sum_bn += B * nb[(size_t)t];
        c->sum_n2 += (double)nb[(size_t)t] * nb[(size_t)t];
      }
    }
    c->flops_screened = f;
  } else {  // every run counts on every group
    c->flops_screened = c->flops_dense;
    c->sum_bn = (double)c->npts * n;
    c->sum_n2 = std::ceil((double)c->npts / kScreenTile) * n * n;
    for (long g = 0; g < ngr; ++g)
      for (int r = 0; r < n8; ++r) sig[(size_t)g * nw8 + r / 32] |= 1u << (r % 32);
    HIPCHK(c, hipMemcpy(c->sig8, sig.data(), sizeof(uint32_t) * sig.size(), hipMemcpyHostToDevice));
    for (long t = 0; t < ntp; ++t)
      for (int si = 0; si < c->n_shells; ++si) smark[(size_t)t * nws + si / 32] |= 1u << (si % 32);
  }
  // per 128-point tile: the functions of its marked shells, ascending (the
  // density contraction's output columns)
  // (and as a bitmap of nwf words per tile)
  c->nwf = (c->NP + 31) / 32;
  std::vector<uint32_t> tfb((size_t)ntp * c->nwf, 0u);
  {
    c->h_tf_off.assign(1, 0);
    c->h_tfl.clear();
    for (long t = 0; t < ntp; ++t) {
      uint32_t *fm = tfb.data() + (size_t)t * c->nwf;
      for (int si = 0; si < c->n_shells; ++si)
        if ((smark[(size_t)t * nws + si / 32] >> (si % 32)) & 1u)
          for (int f = ss[(size_t)si].func_off; f < ss[(size_t)si].func_off + ss[(size_t)si].nfunc; ++f)
            fm[(size_t)f / 32] |= 1u << (f % 32);
      for (int f = 0; f < c->NP; ++f)
        if ((fm[(size_t)f / 32] >> (f % 32)) & 1u) c->h_tfl.push_back((uint16_t)f);
      c->h_tf_off.push_back((int)c->h_tfl.size());
    }
  }
  if ((rc = upload(c, &c->tfb, tfb))) return rc;
  auto bit = [&](long g, int r) { return (sig[(size_t)g * nw8 + r / 32] >> (r % 32)) & 1u; };
  // per 128-point tile: its runs (union over its four groups), and per run
  // its functions in the tile's list
  c->h_tl_off.assign(1, 0);
  c->h_tl.clear();
  c->h_tlm.clear();
  for (long t = 0; t < ntp; ++t) {
    for (int r = 0; r < n8; ++r)
      if (bit(4 * t, r) | bit(4 * t + 1, r) | bit(4 * t + 2, r) | bit(4 * t + 3, r)) {
        c->h_tl.push_back((uint16_t)r);
        c->h_tlm.push_back((uint8_t)(tfb[(size_t)t * c->nwf + (size_t)r / 4] >> (8 * (r % 4))));
      }
    c->h_tl_off.push_back((int)c->h_tl.size());
  }
  // Point splits of the potential contraction: kSplitPts points (at most 32
  // tiles), halved while a chunk has fewer than kSplitItems items (split x pair
  // of function chunks), one per CU.  A shorter split holds fewer functions its
  // tiles do not share, but its partial is written and read once.  Whole call at
  // 1 / 256 / 1024 items: 23-atom LDA build 881 / 743 / 760 us, 14-atom open
  // shell 1268 / 1180 / 1235, water 326 / 284 / 287, (H2O)16 mixed step 4761 /
  // 4759 / 5427, (H2O)8 open-shell FP32 step 3547 / 3547 / 3707.
  {
    long spts = kSplitPts;
    const double nt = (double)c->h_tfl.size() / (double)std::max<long>(1, (c->npts + kScreenTile - 1) / kScreenTile);
    // chunks of 96 functions, or of 64 or 128 where one holds a split's functions
    // (1.3 times a tile's): split-BF16 stage at 64 / 96 / 128, one lane, (H2O)16
    // 0.71 / 0.60 / 0.65 ms, (H2O)32 2.40 / 1.90 / 2.41, (H2O)128 and solute 127 /
    // 89 / 90; FP64 23-atom molecule at 96 / 128 0.30 / 0.15 ms
    if (!c->pt) c->pt = 1.3 * nt <= 64.0 ? 64 : 1.3 * nt <= 128.0 ? 128 : 96;
    const double nch = std::ceil(1.1 * nt / c->pt);
    // density items of 128 columns while a tile has few functions, else 256
    c->icols = nt > kWideTile ? 256 : 128;
    while (spts > kMinSplitPts && (double)(c->Mc / spts) * nch * nch < kSplitItems &&
           (double)(c->npad / spts) * 4.0 * c->NP <= 268435456.0)  // the places: 256 MiB
      spts /= 2;
    c->nsp = (int)(c->Mc / spts);
  }
  // per split: the union of its tiles' functions (the potential's rows and
  // columns, in chunks of tf functions), per entry the split's tiles whose list
  // holds the function, and the functions' places in it
  const long NS = (long)c->nchunks * c->nsp, nst = c->Mc / c->nsp / kScreenTile;
  const int bpc = (c->nsp + 7) / 8;
  c->h_su_off.assign(1, 0);
  c->h_su.clear();
  c->h_sumask.clear();
  std::vector<long> ho((size_t)(2 * NS)), hc((size_t)c->nchunks);  // ho: for one and for two lanes
  std::vector<uint16_t> pos((size_t)NS * c->NP, 0xffff);
  std::vector<uint8_t> rbits((size_t)(c->NP / 32) * bpc * c->nchunks, 0);
  {
    std::vector<uint32_t> tm((size_t)c->NP);
    long at = 0;
    for (long S = 0; S < NS; ++S) {
      if (S % c->nsp == 0) at = 0;
      std::fill(tm.begin(), tm.end(), 0u);
      for (long t = 0; t < nst; ++t)
        for (int i = c->h_tf_off[(size_t)(S * nst + t)]; i < c->h_tf_off[(size_t)(S * nst + t) + 1]; ++i)
          tm[c->h_tfl[(size_t)i]] |= 1u << t;
      const size_t u0 = c->h_su.size();
      const size_t byte = (size_t)(S / c->nsp) * bpc + (size_t)(S % c->nsp) / 8;
      for (int f = 0; f < c->NP; ++f)
        if (tm[(size_t)f]) {
          pos[(size_t)S * c->NP + f] = (uint16_t)(c->h_su.size() - u0);
          rbits[(size_t)(f / 32) * bpc * c->nchunks + byte] |= (uint8_t)(1u << ((S % c->nsp) % 8));
          c->h_su.push_back((uint16_t)f);
          c->h_sumask.push_back(tm[(size_t)f]);
        }
      c->h_su_off.push_back((int)c->h_su.size());
      ho[(size_t)S] = at;
      const long ld = round_up((long)(c->h_su.size() - u0), 16);
      at += ld * ld;
      hc[(size_t)(S / c->nsp)] = at;
    }
  }
  // Room for all chunks' partials, or kPartialBytes shared by the lanes (at least
  // a chunk each): a lane's chunks lie one behind the other until the next does
  // not fit.  Chunks differ (outer points need more functions): by their own sizes
  // the 159 chunks of (H2O)128 and solute fill it 21 times on two lanes, in slots of the largest
  // 54 times, and every sum reads and writes the N^2 sums (fold kernels of a build
  // 49 -> 35 ms, two builds of a step 506 -> 485 ms).
  {
    const long cap = kPartialBytes / 8, most = *std::max_element(hc.begin(), hc.end());
    const long total = std::accumulate(hc.begin(), hc.end(), 0L);
    c->hflush = total > cap;
    c->hsize = c->hflush ? c->nlanes_cap * std::max(most, cap / c->nlanes_cap) : std::max(total, 1L);
    const std::vector<long> rel(ho.begin(), ho.begin() + NS);
    for (int lanes = 1; lanes <= 2; ++lanes) {
      std::vector<char> &fl = c->h_flush[lanes - 1];
      fl.assign((size_t)c->nchunks, 0);
      const long share = c->hsize / std::min(lanes, c->nlanes_cap);
      for (int ln = 0; ln < lanes; ++ln) {
        long at = 0;
        for (int k = ln; k < c->nchunks; k += lanes) {
          if (c->hflush && at + hc[(size_t)k] > share) {
            fl[(size_t)(k - lanes)] = 1;
            at = 0;
          }
          const long base = c->hflush ? ln * share + at : std::accumulate(hc.begin(), hc.begin() + k, 0L);
          for (int j = 0; j < c->nsp; ++j)
            ho[(size_t)((lanes - 1) * NS + (long)k * c->nsp + j)] = base + rel[(size_t)((long)k * c->nsp + j)];
          at += hc[(size_t)k];
          if (k + lanes >= c->nchunks) fl[(size_t)k] = 1;
        }
      }
    }
    if (getenv("PGXC_DEBUG"))
      fprintf(stderr, "pgxc: partials %.4g bytes in %.4g, sums %d times on one lane, %d on two\n", 8.0 * total,
              8.0 * c->hsize, (int)std::count(c->h_flush[0].begin(), c->h_flush[0].end(), 1),
              (int)std::count(c->h_flush[1].begin(), c->h_flush[1].end(), 1));
  }
  if ((rc = upload(c, &c->ho, ho))) return rc;
  if ((rc = upload(c, &c->pos, pos))) return rc;
  if ((rc = upload(c, &c->rbits, rbits))) return rc;
  // What the basis stage writes, per (shell, 32-point group): values and
  // gradients of the shells marked on the group's tile, the functions of the
  // tile's list (the contractions, the density's sums and the W pass read no
  // others: they stage zeros for the rest).  No stage reads any other block of
  // a basis-value buffer.
  {
    const int nr = c->n_ranges;
    std::vector<uint32_t> bi, bfl;
    c->h_bi_off.assign(1, 0);
    const long gpb = kThreads / kGroup;  // groups per basis block
    for (int k = 0; k < c->nchunks; ++k) {
      const long g0 = (long)k * c->Mc / kGroup;
      for (long b = 0; b < c->Mc / kThreads; ++b) {
        const uint32_t *m0 = smark.data() + (size_t)((g0 + b * gpb) / 4) * nws, *m1 = m0 + nws;
        for (int ri = 0; ri < nr; ++ri) {
          // the range's shells read on each tile of the block
          uint32_t fw[2] = {0, 0};
          const RangeD &R = c->h_ranges[(size_t)ri];
          for (int j = 0; j < R.n_shells; ++j) {
            const int sg = R.shell_begin + j;
            fw[0] |= ((m0[sg / 32] >> (sg % 32)) & 1u) << j;
            fw[1] |= ((m1[sg / 32] >> (sg % 32)) & 1u) << j;
          }
          if (!(fw[0] | fw[1])) continue;
          bi.push_back((uint32_t)(b << 16 | ri));
          bfl.insert(bfl.end(), fw, fw + 2);
        }
      }
      c->h_bi_off.push_back((long)bi.size());
    }
    if ((rc = upload(c, &c->bi, bi))) return rc;
    if ((rc = upload(c, &c->bfl, bfl))) return rc;
    if (getenv("PGXC_DEBUG")) {  // sizes of the screened work
      double ev = 0, hu = 0;
      for (size_t t = 0; t + 1 < c->h_tf_off.size(); ++t) ev += (double)kScreenTile * (c->h_tf_off[t + 1] - c->h_tf_off[t]);
      for (long S = 0; S < NS; ++S) hu += c->h_su_off[(size_t)S + 1] - c->h_su_off[(size_t)S];
      fprintf(stderr, "pgxc: basis items %zu (of %ld), elements per build %.4g; %ld splits of %ld points, "
                      "%.1f functions each\n",
              bi.size(), (long)c->nchunks * (c->Mc / kThreads) * c->n_ranges, ev, NS, c->Mc / c->nsp,
              hu / NS);
    }
  }
  // work items per chunk
  const long tpc = c->Mc / kScreenTile;
  c->h_di_off.assign(1, 0);
  c->h_pi_off.assign(1, 0);
  c->h_di.clear();
  c->h_pi.clear();
  for (int k = 0; k < c->nchunks; ++k) {
    for (long t = 0; t < tpc; ++t) {
      const long T = k * tpc + t;
      const int nf = c->h_tf_off[(size_t)T + 1] - c->h_tf_off[(size_t)T];
      // density items: shares of at most icols of the tile's functions
      for (int pr = 0; pr < (nf + c->icols - 1) / c->icols; ++pr) c->h_di.push_back((uint32_t)(t << 8 | pr));
    }
    c->h_di_off.push_back((long)c->h_di.size());
    for (int sl = 0; sl < c->nsp; ++sl) {
      const long S = (long)k * c->nsp + sl;
      const int nu = c->h_su_off[(size_t)S + 1] - c->h_su_off[(size_t)S], nch = (nu + c->pt - 1) / c->pt;
      for (int ci = 0; ci < nch; ++ci)
        for (int cj = 0; cj < nch; ++cj)
          c->h_pi.push_back((uint32_t)sl << 20 | (uint32_t)ci << 10 | (uint32_t)cj);
    }
    c->h_pi_off.push_back((long)c->h_pi.size());
  }
  if ((rc = upload(c, &c->tl_off, c->h_tl_off))) return rc;
  if ((rc = upload(c, &c->tl, c->h_tl))) return rc;
  if ((rc = upload(c, &c->tlm, c->h_tlm))) return rc;
  if ((rc = upload(c, &c->tf_off, c->h_tf_off))) return rc;
  if ((rc = upload(c, &c->tfl, c->h_tfl))) return rc;
  if ((rc = upload(c, &c->su_off, c->h_su_off))) return rc;
  if ((rc = upload(c, &c->su, c->h_su))) return rc;
  if ((rc = upload(c, &c->sumask, c->h_sumask))) return rc;
  if ((rc = upload(c, &c->di, c->h_di))) return rc;
  if ((rc = upload(c, &c->pi, c->h_pi))) return rc;
  return PGXC_OK;
}

extern "C" {

static char g_free_err[256];  // message of the last failed context-free call

const char *pgxc_last_error(const pgxc_ctx *ctx) {
  if (ctx) return ctx->err.c_str();
  return g_free_err[0] ? g_free_err : "null context";
}

int64_t pgxc_nbas(const pgxc_ctx *ctx) { return ctx ? ctx->nbas : -1; }

int pgxc_create_opt(pgxc_ctx **out, int32_t n_atoms, const double *atom_xyz, int32_t n_shells,
                    const int32_t *shell_info, const double *exps, const double *norms,
                    const double *contr, const double *grid, int64_t npts, int32_t veclen,
                    const pgxc_options *opt) {
  if (!out) return PGXC_ERR_ARG;
  *out = nullptr;
  pgxc_ctx *c = new pgxc_ctx();
  *out = c;
  if (n_atoms <= 0 || n_shells <= 0 || !atom_xyz || !shell_info || !exps || !norms ||
      (!contr && n_shells > 0) || !grid || npts <= 0 || veclen <= 0)
    return fail(c, PGXC_ERR_ARG, "pgxc_create: null pointer or non-positive size");
  if (opt && opt->tile != 0 && opt->tile != 64 && opt->tile != 96 && opt->tile != 128)
    return fail(c, PGXC_ERR_ARG, "pgxc_create: tile must be 0, 64, 96 or 128");
  if (opt && (opt->chunk_points < 0 || opt->chunk_points % kSplitPts != 0))
    return fail(c, PGXC_ERR_ARG, "pgxc_create: chunk_points must be a non-negative multiple of 2048");
  if (opt && (opt->variant_fp64 < -1 || opt->variant_fp64 >= kNumVariants || opt->variant_fp32 < -1 ||
              opt->variant_fp32 >= kNumVariants))
    return fail(c, PGXC_ERR_ARG, "pgxc_create: variant must be -1 (default) or 0.." +
                                     std::to_string(kNumVariants - 1));
  if (opt && (opt->no_screen < 0 || opt->no_screen > 1 || opt->no_basis_cache < 0 ||
              opt->no_basis_cache > 1))
    return fail(c, PGXC_ERR_ARG, "pgxc_create: no_screen and no_basis_cache must be 0 or 1");
  c->cache_off = opt ? opt->no_basis_cache : 0;
  if (opt && opt->variant_fp64 >= 0) c->var[0] = opt->variant_fp64;
  if (opt && opt->variant_fp32 >= 0) c->var[1] = opt->variant_fp32;
  if (n_shells > kMaxShells)
    return fail(c, PGXC_ERR_UNSUPPORTED, "pgxc_create: more than " + std::to_string(kMaxShells) + " shells");
  c->n_atoms = n_atoms;
  c->n_shells = n_shells;
  c->npts = npts;
  c->veclen = veclen;

  // ---- basis tables (shells must be grouped by atom) ---------------------
  std::vector<ShellD> sh(n_shells);
  std::vector<AtomD> at(n_atoms);
  for (int a = 0; a < n_atoms; ++a) {
    at[a].x = atom_xyz[3 * a];
    at[a].y = atom_xyz[3 * a + 1];
    at[a].z = atom_xyz[3 * a + 2];
    at[a].shell_begin = at[a].shell_end = 0;
    at[a].lmax = 0;
    at[a].pad = 0;
  }
  long eoff = 0, coff = 0, foff = 0;
  std::vector<double> tab;
  std::map<std::pair<int, std::string>, int> tabs;
  int prev_atom = -1;
  std::vector<int> seen(n_atoms, 0);
  for (int s = 0; s < n_shells; ++s) {
    const int32_t *si = shell_info + 5 * s;
    ShellD &d = sh[s];
    d.atom = si[0];
    d.l = si[1];
    d.n_exp = si[2];
    d.n_unc = si[3];
    d.n_contr = si[4];
    if (d.atom < 0 || d.atom >= n_atoms)
      return fail(c, PGXC_ERR_ARG, "pgxc_create: shell " + std::to_string(s) + " atom out of range");
    if (d.l < 0 || d.l > kLMax)
      return fail(c, PGXC_ERR_UNSUPPORTED, "pgxc_create: l = " + std::to_string(d.l) +
                                               " above the supported maximum " + std::to_string(kLMax));
    if (d.n_exp <= 0 || d.n_unc < 0 || d.n_contr < 0 || d.n_unc > d.n_exp ||
        d.n_unc + d.n_contr <= 0)
      return fail(c, PGXC_ERR_ARG, "pgxc_create: shell " + std::to_string(s) + " has inconsistent counts");
    if (d.n_contr > kMaxContr)
      return fail(c, PGXC_ERR_UNSUPPORTED, "pgxc_create: more than " + std::to_string(kMaxContr) +
                                               " contracted functions in one shell");
    if (d.atom != prev_atom) {
      if (seen[d.atom])
        return fail(c, PGXC_ERR_ARG, "pgxc_create: shells of one atom must be contiguous");
      seen[d.atom] = 1;
      at[d.atom].shell_begin = s;
      prev_atom = d.atom;
    }
    at[d.atom].shell_end = s + 1;
    at[d.atom].lmax = std::max(at[d.atom].lmax, d.l);
    c->lmax = std::max(c->lmax, d.l);
    d.exp_off = (int)eoff;
    d.func_off = (int)foff;
    {  // blocks of kPB primitives: exponents (padded with the last one), norms and each
       // contraction's coefficients; shells with the same contents share a table, so that a large
       // system's few kinds of shell stay in the scalar cache (16 KiB for two CUs)
      const int row = (d.n_exp + kPB - 1) / kPB * kPB;
      std::vector<double> t((size_t)(2 + d.n_contr) * row, 0.0);
      for (int e = 0; e < row; ++e) {
        double *q = t.data() + (2 + d.n_contr) * (e / kPB * kPB) + e % kPB;
        q[0] = exps[eoff + std::min(e, d.n_exp - 1)];
        if (e >= d.n_exp) continue;
        q[kPB] = norms[eoff + e];
        for (int k = 0; k < d.n_contr; ++k) q[(2 + k) * kPB] = contr[coff + (long)k * d.n_exp + e];
      }
      const std::string key((const char *)t.data(), t.size() * sizeof(double));
      const auto ins = tabs.insert({{d.n_contr, key}, (int)tab.size()});
      if (ins.second) tab.insert(tab.end(), t.begin(), t.end());
      d.tab = ins.first->second;
    }
    eoff += d.n_exp;
    coff += (long)d.n_exp * d.n_contr;
    foff += (long)(2 * d.l + 1) * (d.n_unc + d.n_contr);
  }
  for (int a = 0; a < n_atoms; ++a) {
    long np = 0, nc = 0;
    for (int s = at[a].shell_begin; s < at[a].shell_end; ++s) {
      np += sh[s].n_exp;
      nc += (long)sh[s].n_exp * sh[s].n_contr;
    }
    if (at[a].shell_end - at[a].shell_begin > kAtomShells || np > kAtomPrims || nc > kAtomContr)
      return fail(c, PGXC_ERR_UNSUPPORTED,
                  "pgxc_create: atom " + std::to_string(a) + " has more than " +
                      std::to_string(kAtomShells) + " shells, " + std::to_string(kAtomPrims) +
                      " primitives or " + std::to_string(kAtomContr) + " contraction coefficients");
  }
  for (long e = 0; e < eoff; ++e)
    if (!(exps[e] > 0.0) || !std::isfinite(norms[e]))
      return fail(c, PGXC_ERR_ARG, "pgxc_create: exponents must be positive and norms finite");
  c->nbas = (int)foff;
  c->exps_per_point = (double)eoff;
  function_order(sh, exps, atom_xyz, n_atoms, c->fpos);
  // function tile: requested, or the one of 128 / 96 / 64 that pads nbas least
  if (opt && opt->tile) {
    c->tf = c->pt = opt->tile;
    c->NP = (int)round_up(c->nbas, c->tf);
  } else {
    c->tf = 128;
    c->NP = (int)round_up(c->nbas, 128);
    for (int t : {96, 64})
      if (round_up(c->nbas, t) < c->NP) {
        c->NP = (int)round_up(c->nbas, t);
        c->tf = t;
      }
  }
  c->nparts = (c->NP + kPartCols - 1) / kPartCols;  // density partials of a point at most

  // ---- chunking of the grid ----------------------------------------------
  // a chunk holds at most 256 Ki points and 8 GiB of FP64 basis values; a
  // point split of the potential contraction is a whole number m of
  // 2048-point blocks, the fewest that keep the splits of a chunk at 64 or
  // less, and the chunk is rounded up to whole splits (one more chunk when
  // that would pass the limit)
  long mc_max = std::max<long>(kSplitPts, ((8L << 30) / (32L * c->NP)) / kSplitPts * kSplitPts);
  mc_max = std::min<long>(mc_max, 1L << 18);
  if (opt && opt->chunk_points) mc_max = opt->chunk_points;
  for (c->nchunks = (int)((npts + mc_max - 1) / mc_max);; ++c->nchunks) {
    const long q = round_up((npts + c->nchunks - 1) / c->nchunks, kSplitPts) / kSplitPts;
    const long m = (q + 63) / 64;
    c->nsplit = (int)((q + m - 1) / m);
    c->Mc = (long)c->nsplit * m * kSplitPts;
    if (c->Mc <= mc_max) break;
  }
  c->npad = c->Mc * c->nchunks;
  c->nblk_total = c->npad / kThreads;

  HIPCHK(c, hipGetDevice(&c->device));
  HIPCHK(c, hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
  c->nlanes = c->nlanes_cap = c->nchunks > 1 ? 2 : 1;
  HIPCHK(c, hipStreamCreateWithFlags(&c->stream2, hipStreamNonBlocking));
  HIPCHK(c, c->pin.init());
  HIPCHK(c, hipEventCreateWithFlags(&c->fork, hipEventDisableTiming));
  HIPCHK(c, hipEventCreateWithFlags(&c->join, hipEventDisableTiming));
  // atom ranges of the basis stage: consecutive atoms in shell order, at most
  // kRangeAtoms (half as many: FP32 basis stage of (H2O)32 1.50 -> 1.64 ms), fewer
  // where a chunk's blocks would give the device less than kBasisItems items
  const int ra_most = (int)std::min<long>(kRangeAtoms, std::max<long>(1, n_atoms * (c->Mc / kThreads) / kBasisItems));
  std::vector<int> ratoms;
  for (int a = 0; a < n_atoms; ++a)
    if (at[a].shell_end > at[a].shell_begin) ratoms.push_back(a);
  std::sort(ratoms.begin(), ratoms.end(),
            [&](int p, int q) { return at[p].shell_begin < at[q].shell_begin; });
  c->h_ranges.clear();
  for (size_t i = 0; i < ratoms.size(); ++i) {
    const AtomD &a = at[ratoms[i]];
    const int ns = a.shell_end - a.shell_begin;
    if (c->h_ranges.empty() || c->h_ranges.back().n_atoms == ra_most ||
        c->h_ranges.back().n_shells + ns > kRangeShells) {
      RangeD r{};
      r.atom_begin = (int)i;
      r.shell_begin = a.shell_begin;
      c->h_ranges.push_back(r);
    }
    RangeD &r = c->h_ranges.back();
    ++r.n_atoms;
    r.n_shells += ns;
  }
  c->n_ranges = (int)c->h_ranges.size();
  int rc;
  if ((rc = dalloc(c, &c->grid, 4 * (size_t)c->npad))) return rc;
  if ((rc = dalloc(c, &c->atoms, n_atoms))) return rc;
  if ((rc = dalloc(c, &c->shells, n_shells))) return rc;
  if ((rc = dalloc(c, &c->ranges, std::max<size_t>(c->h_ranges.size(), 1)))) return rc;
  if ((rc = dalloc(c, &c->ratoms, std::max<size_t>(ratoms.size(), 1)))) return rc;
  tab.insert(tab.end(), 2 * kPB, 0.0);  // a block is read with two contractions
  if ((rc = upload(c, &c->tabd, tab))) return rc;
  {
    std::vector<float> t32(tab.begin(), tab.end());
    if ((rc = upload(c, &c->tabf, t32))) return rc;
  }
  // grid in space-filling-curve order, padded with far points of zero weight
  std::vector<long> perm;
  morton_order(grid, npts, npts, 1, perm);
  {
    std::vector<int> p32(perm.begin(), perm.end());
    if ((rc = upload(c, &c->perm_d, p32))) return rc;
  }
  c->axyz.assign(atom_xyz, atom_xyz + 3 * (size_t)n_atoms);
  std::vector<double> g(4 * (size_t)c->npad);
  for (int k = 0; k < 4; ++k)
    for (long p = 0; p < c->npad; ++p)
      g[(size_t)k * c->npad + p] =
          p < npts ? grid[(size_t)k * npts + perm[p]] : (k < 3 ? kFar : 0.0);
  HIPCHK(c, hipMemcpy(c->grid, g.data(), g.size() * 8, hipMemcpyHostToDevice));
  {
    uint64_t h = 1469598103934665603ull;
    h = hash_words(h, atom_xyz, 3 * (size_t)n_atoms * 8);
    h = hash_words(h, shell_info, 5 * (size_t)n_shells * 4);
    h = hash_words(h, exps, (size_t)eoff * 8);
    h = hash_words(h, norms, (size_t)eoff * 8);
    h = hash_words(h, contr, (size_t)coff * 8);
    h = hash_words(h, grid, 4 * (size_t)npts * 8);
    const int64_t lay[2] = {c->NP, c->npad};
    c->geom = hash_words(h, lay, sizeof(lay));
  }
  HIPCHK(c, hipMemcpy(c->atoms, at.data(), sizeof(AtomD) * n_atoms, hipMemcpyHostToDevice));
  HIPCHK(c, hipMemcpy(c->shells, sh.data(), sizeof(ShellD) * n_shells, hipMemcpyHostToDevice));
  if (!ratoms.empty()) {
    HIPCHK(c, hipMemcpy(c->ranges, c->h_ranges.data(), sizeof(RangeD) * c->h_ranges.size(),
                        hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(c->ratoms, ratoms.data(), sizeof(int) * ratoms.size(), hipMemcpyHostToDevice));
  }
  if ((rc = dalloc(c, &c->d_fpos, c->nbas))) return rc;
  HIPCHK(c, hipMemcpy(c->d_fpos, c->fpos.data(), sizeof(int) * c->nbas, hipMemcpyHostToDevice));
  {
    std::vector<int> finv((size_t)c->nbas);
    for (int f = 0; f < c->nbas; ++f) finv[(size_t)c->fpos[f]] = f;
    if ((rc = upload(c, &c->d_finv, finv))) return rc;
  }
  if ((rc = setup_screen(c, sh, exps, !(opt && opt->no_screen)))) return rc;
  const size_t np2 = (size_t)c->NP * c->NP;
  if ((rc = dalloc(c, &c->P, np2))) return rc;
  if ((rc = dalloc(c, &c->Pref, np2))) return rc;
  HIPCHK(c, hipMalloc(&c->D, np2 * 8));
  HIPCHK(c, hipMemset(c->P, 0, np2 * 8));
  HIPCHK(c, hipMemset(c->Pref, 0, np2 * 8));
  if ((rc = dalloc(c, &c->state, (size_t)S_NSLOT * c->npad))) return rc;
  HIPCHK(c, hipMemset(c->state, 0, (size_t)S_NSLOT * c->npad * 8));
  const size_t npk = (size_t)c->nbas * (c->nbas + 1) / 2;
  if ((rc = dalloc(c, &c->Vstate, npk))) return rc;
  if ((rc = dalloc(c, &c->Vout, npk))) return rc;
  if ((rc = dalloc(c, &c->epart, 2 * (size_t)c->nblk_total))) return rc;
  if ((rc = dalloc(c, &c->eterm, 5 * (size_t)c->nblk_total))) return rc;
  const size_t L = (size_t)c->nlanes_cap;
  if ((rc = dalloc(c, &c->part, L * c->nparts * 4 * c->Mc))) return rc;
  if ((rc = dalloc(c, &c->coef, L * 4 * c->Mc))) return rc;
  // sums in enough segments of the splits that a small matrix still fills the device
  const long nb32 = c->NP / 32, pairs = nb32 * (nb32 + 1) / 2;
  const long ns = (long)c->nchunks * c->nsp;
  c->nseg = (int)std::min<long>({std::max<long>(kFoldItems / pairs, (ns + 63) / 64), (ns + 3) / 4, 32L});
  if ((rc = alloc_partials(c, &c->Hc, &c->HS))) return rc;
  HIPCHK(c, hipMemset(c->part, 0, L * c->nparts * 4 * c->Mc * 8));
  HIPCHK(c, hipMemset(c->coef, 0, L * 4 * c->Mc * 8));
  return PGXC_OK;
}

int pgxc_create(pgxc_ctx **out, int32_t n_atoms, const double *atom_xyz, int32_t n_shells,
                const int32_t *shell_info, const double *exps, const double *norms,
                const double *contr, const double *grid, int64_t npts, int32_t veclen) {
  return pgxc_create_opt(out, n_atoms, atom_xyz, n_shells, shell_info, exps, norms, contr, grid,
                         npts, veclen, nullptr);
}

int pgxc_layout(const pgxc_ctx *c, int64_t *out8) {
  if (!c || !out8) return PGXC_ERR_ARG;
  out8[0] = c->NP;
  out8[1] = c->tf;
  out8[2] = c->Mc;
  out8[3] = c->nchunks;
  out8[4] = c->nsplit;
  out8[5] = c->npad;
  out8[6] = c->var[0];
  out8[7] = c->var[1];
  return PGXC_OK;
}

}  // extern "C"

// Buffers of the beta spin, zeroed like the alpha spin's at creation.
static int alloc_beta(pgxc_ctx *c) {
  auto &B = c->beta;
  if (B.ready) return PGXC_OK;
  const size_t np2 = (size_t)c->NP * c->NP, npk = (size_t)c->nbas * (c->nbas + 1) / 2;
  const size_t L = (size_t)c->nlanes_cap;
  int rc;
  if ((rc = dalloc(c, &B.P, np2)) || (rc = dalloc(c, &B.Pref, np2))) return rc;
  if (!B.D) HIPCHK(c, hipMalloc(&B.D, np2 * 8));
  if ((rc = dalloc(c, &B.state, (size_t)S_NSLOT * c->npad)) || (rc = dalloc(c, &B.Vstate, npk)) ||
      (rc = dalloc(c, &B.Vout, npk)) || (rc = dalloc(c, &B.part, L * c->nparts * 4 * c->Mc)) ||
      (rc = dalloc(c, &B.coef, L * 4 * c->Mc)) || (rc = alloc_partials(c, &B.Hc, &B.HS)))
    return rc;
  HIPCHK(c, hipMemset(B.P, 0, np2 * 8));
  HIPCHK(c, hipMemset(B.Pref, 0, np2 * 8));
  HIPCHK(c, hipMemset(B.state, 0, (size_t)S_NSLOT * c->npad * 8));
  HIPCHK(c, hipMemset(B.part, 0, L * c->nparts * 4 * c->Mc * 8));
  HIPCHK(c, hipMemset(B.coef, 0, L * 4 * c->Mc * 8));
  B.ready = 1;  // a call that failed before here goes on with those it lacks
  return PGXC_OK;
}

// Switch the context to ispin spins: a build state of the other spin count
// is dropped, and the plan (whose units depend on it) rebuilt.
static int set_spins(pgxc_ctx *c, int ispin) {
  if (ispin == c->ispin) return PGXC_OK;
  if (ispin == 2) {
    int rc = alloc_beta(c);
    if (rc) return rc;
  }
  c->ispin = ispin;
  c->have_state = 0;
  c->have_density = 0;
  free_plan(c->plan);
  free_plan(c->plan_e);
  free_plan(c->plan_g);
  return PGXC_OK;
}

static int check_density_args(pgxc_ctx *c, int32_t ispin, int32_t nbas, int32_t mode) {
  if (!c) return PGXC_ERR_ARG;
  if (ispin != 1 && ispin != 2)
    return fail(c, PGXC_ERR_ARG, "ispin = " + std::to_string(ispin) + ": must be 1 or 2");
  if (nbas != c->nbas)
    return fail(c, PGXC_ERR_ARG, "nbas = " + std::to_string(nbas) + " but the basis has " +
                                     std::to_string(c->nbas) + " functions");
  if (mode != PGXC_DENSITY_FULL && mode != PGXC_DENSITY_INCREMENTAL)
    return fail(c, PGXC_ERR_ARG, "unknown density mode " + std::to_string(mode));
  if (mode == PGXC_DENSITY_INCREMENTAL && c->have_state && ispin != c->ispin)
    return fail(c, PGXC_ERR_STATE, "incremental density with ispin = " + std::to_string(ispin) +
                                       " after a build with ispin = " + std::to_string(c->ispin));
  return set_spins(c, ispin);
}

extern "C" int pgxc_set_density(pgxc_ctx *c, int32_t ispin, int32_t nbas, const double *P,
                                int32_t mode) {
  int rc = check_density_args(c, ispin, nbas, mode);
  if (rc) return rc;
  if (!P) return fail(c, PGXC_ERR_ARG, "pgxc_set_density: P is null");
  const int n = c->nbas, NP = c->NP;
  std::vector<double> h((size_t)NP * NP, 0.0);
  const int *pos = c->fpos.data();
  for (int sp = 0; sp < ispin; ++sp) {
    const double *Ps = P + (size_t)sp * n * n;
    for (int j = 0; j < n; ++j)
      for (int i = 0; i < n; ++i) h[(size_t)pos[i] * NP + pos[j]] = Ps[(size_t)i + (size_t)j * n];
    HIPCHK(c, hipMemcpy(sp ? c->beta.P : c->P, h.data(), h.size() * 8, hipMemcpyHostToDevice));
  }
  c->have_density = 1;
  c->density_mode = mode;
  return PGXC_OK;
}

extern "C" int pgxc_set_orbitals(pgxc_ctx *c, int32_t ispin, int32_t nbas, int32_t nocc,
                                 const double *C, const double *occ, int32_t mode) {
  int rc = check_density_args(c, ispin, nbas, mode);
  if (rc) return rc;
  if (nocc < 0 || (nocc > 0 && (!C || !occ)))
    return fail(c, PGXC_ERR_ARG, "pgxc_set_orbitals: bad nocc or null C/occ");
  const int n = c->nbas;
  const size_t nC = (size_t)ispin * n * nocc, no = (size_t)ispin * nocc;
  if (c->orb_n < nC + no) {
    dfree(c->orb);
    c->orb = nullptr;
    c->orb_n = 0;
    HIPCHK(c, hipMalloc((void **)&c->orb, (nC + no) * 8));
    c->orb_n = nC + no;
  }
  double *dC = c->orb, *docc = c->orb + nC;
  std::lock_guard<std::recursive_mutex> lk(c->pin.mu);  // to the wait below
  if ((nC + no) * 8 <= 2 * PinnedPair::kHalf) {  // one copy from pinned memory
    if (nC) {
      memcpy(c->pin.buf, C, nC * 8);
      memcpy(c->pin.buf + nC * 8, occ, no * 8);
      launch_copy(c->stream, (const double *)c->pin.buf, dC, (long)(nC + no));
    }
  } else {
    HIPCHK(c, hipMemcpy(dC, C, nC * 8, hipMemcpyHostToDevice));
    HIPCHK(c, hipMemcpy(docc, occ, no * 8, hipMemcpyHostToDevice));
  }
  for (int sp = 0; sp < ispin; ++sp)  // nocc = 0: P = 0
    launch_form_density(c->stream, dC + (size_t)sp * n * nocc, docc + (size_t)sp * nocc, c->d_finv, n, nocc,
                        c->NP, sp ? c->beta.P : c->P);
  HIPCHK(c, hipGetLastError());
  HIPCHK(c, hipStreamSynchronize(c->stream));
  c->have_density = 1;
  c->density_mode = mode;
  return PGXC_OK;
}

extern "C" {

int pgxc_build(pgxc_ctx *c, uint32_t functional, int32_t precision, double *ham, double *exc,
               double *charge) {
  int incr = 0;
  int rc = validate_build(c, functional, precision, incr);
  if (rc) return rc;
  const bool gga = (functional & (PGXC_XC_PBEX | PGXC_XC_PBEC)) != 0;
  hipStream_t s = c->stream;
  const size_t elem = precision == PGXC_PREC_FP64 ? 8 : 4;
  if ((rc = ensure_work(c, elem, s, gga))) return rc;
  std::vector<pgxc_ctx *> mols{c};
  std::vector<int> incrv{incr};
  if ((rc = get_plan(mols, functional, precision, incrv, {}, -1, c->sched, c->plan, c))) return rc;
  const size_t nev = kEvStep + 5 * c->plan->steps.size();
  while (c->ev.size() < nev) {
    hipEvent_t e = nullptr;
    HIPCHK(c, hipEventCreate(&e));
    c->ev.push_back(e);
  }
  HIPCHK(c, hipEventRecord(c->ev[kEvStart], s));
  if (elem == 8)
    launch_plan<double>(s, c->stream2, c->fork, c->join, *c->plan, gga, &c->ev);
  else
    launch_plan<float>(s, c->stream2, c->fork, c->join, *c->plan, gga, &c->ev);
  HIPCHK(c, hipGetLastError());
  // waits for the build; a small V comes along in the same wait
  std::unique_lock<std::recursive_mutex> lk(c->pin.mu);
  const size_t npk = (size_t)c->nbas * (c->nbas + 1) / 2;
  const bool along = ham && c->ispin == 1 && 8 * npk <= PinnedPair::kHalf &&
                     16 * (size_t)c->nblk_total <= PinnedPair::kHalf;
  double *v = (double *)(c->pin.buf + PinnedPair::kHalf);
  if (along) launch_copy(s, c->Vout, v, (long)npk);
  if ((rc = collect(c, s, functional, precision))) return rc;
  for (int k = 0; k < 4; ++k) c->timing[k] = 0.0;
  float t = 0;
  for (size_t k = 0; k < c->plan->steps.size(); ++k) {
    const hipEvent_t *E = c->ev.data() + kEvStep + 5 * k;
    const bool cached = !c->plan->steps[k].basis.total;
    for (int j = cached ? 1 : 0; j < 4; ++j) {
      HIPCHK(c, hipEventElapsedTime(&t, E[cached && j == 1 ? 0 : j], E[j + 1]));
      c->timing[j] += t;
    }
  }
  HIPCHK(c, hipEventElapsedTime(&t, c->ev[kEvPack], c->ev[kEvEnd]));
  c->timing[4] = t;
  HIPCHK(c, hipEventElapsedTime(&t, c->ev[kEvStart], c->ev[kEvEnd]));
  c->timing[5] = t;
  mark_basis_cached(c, elem, gga);
  if (along) {
    for (size_t i = 0; i < npk; ++i) ham[i] += v[i];
    ham = nullptr;
  }
  lk.unlock();
  return pgxc_get_result(c, ham, exc, charge);
}

int pgxc_get_result(pgxc_ctx *c, double *ham, double *exc, double *charge) {
  if (!c) return PGXC_ERR_ARG;
  if (!c->have_state) return fail(c, PGXC_ERR_STATE, "no build has run on this context");
  if (ham) {  // ispin = 2: alpha / beta at even / odd positions
    const size_t npk = (size_t)c->nbas * (c->nbas + 1) / 2, is = (size_t)c->ispin;
    for (size_t sp = 0; sp < is; ++sp) {
      double *h = ham + sp;
      HIPCHK(c, c->pin.fetch(c->stream, sp ? c->beta.Vout : c->Vout, npk, [&](size_t i0, size_t n, const double *v) {
        if (is == 1)
          for (size_t i = 0; i < n; ++i) h[i0 + i] += v[i];
        else
          for (size_t i = 0; i < n; ++i) h[(i0 + i) * 2] += v[i];
      }));
    }
  }
  if (exc) *exc += c->last_exc;
  if (charge) *charge += c->last_charge;
  return PGXC_OK;
}

int pgxc_energy(pgxc_ctx *c, uint32_t functional, int32_t precision, double *terms4,
                double *charge) {
  int incr = 0;
  int rc = validate_build(c, functional, precision, incr);
  if (rc == PGXC_ERR_STATE && c->have_density) rc = PGXC_OK;  // the full density is always there
  if (rc) return rc;
  const bool gga = (functional & (PGXC_XC_PBEX | PGXC_XC_PBEC)) != 0;
  hipStream_t s = c->stream;
  const size_t elem = precision == PGXC_PREC_FP64 ? 8 : 4;
  if ((rc = ensure_work(c, elem, s, gga))) return rc;
  std::vector<pgxc_ctx *> mols{c};
  std::vector<int> full{0};
  if ((rc = get_plan(mols, functional, precision, full, {}, -1, c->sched, c->plan_e, c, 1))) return rc;
  if (elem == 8)
    launch_plan<double>(s, c->stream2, c->fork, c->join, *c->plan_e, gga, nullptr);
  else
    launch_plan<float>(s, c->stream2, c->fork, c->join, *c->plan_e, gga, nullptr);
  HIPCHK(c, hipGetLastError());
  double t[5] = {0, 0, 0, 0, 0};
  size_t at = 0;
  HIPCHK(c, c->pin.fetch(s, c->eterm, 5 * (size_t)c->nblk_total, [&](size_t, size_t n, const double *v) {
    for (size_t i = 0; i < n; ++i, ++at) t[at % 5] += v[i];
  }));
  memcpy(c->last_terms, t, sizeof(t));
  mark_basis_cached(c, elem, gga);
  if (terms4) memcpy(terms4, t, 4 * sizeof(double));
  if (charge) *charge = t[4];
  return PGXC_OK;
}

// The basis-centre term into c->gsum ([atom][3] on the device, zeroed first);
// with pm (device [3][npad], zeroed) also w grad f at every point, summed over
// spins.
static int gradient_impl(pgxc_ctx *c, double *pm) {
  const uint32_t functional = c->state_functional;
  const bool gga = (functional & (PGXC_XC_PBEX | PGXC_XC_PBEC)) != 0;
  hipStream_t s = c->stream;
  int rc;
  if ((rc = ensure_work(c, 8, s, true))) return rc;
  // an FP64 plan for its basis and W stages: chunk k's values land where its
  // unit points (the FP64 cache, or the lane's work buffer when there is none)
  std::vector<pgxc_ctx *> mols{c};
  std::vector<int> full{0};
  Sched plain;
  plain.mode = PGXC_SCHED_STATIC;
  if ((rc = get_plan(mols, functional, PGXC_PREC_FP64, full, {}, -1, plain, c->plan_g, c))) return rc;
  const Plan &gp = *c->plan_g;
  const long Mc = c->Mc, NP = c->NP, cs = NP * Mc, np = c->npad;
  // the chunk's products and sums stay with the context for later gradients
  long ni = 1;  // the most basis items of one chunk
  for (int k = 0; k < c->nchunks; ++k) ni = std::max<long>(ni, c->h_bi_off[k + 1] - c->h_bi_off[k]);
  if ((rc = dalloc(c, &c->gXZ, 2 * (size_t)cs)) || (rc = dalloc(c, &c->gpart, 12 * (size_t)kRangeAtoms * ni)) ||
      (rc = dalloc(c, &c->gsum, 3 * (size_t)c->n_atoms)))
    return rc;
  HIPCHK(c, hipMemsetAsync(c->gsum, 0, 24 * (size_t)c->n_atoms, s));
  for (int k = 0; k < c->nchunks; ++k) {
    const long p0 = (long)k * Mc;
    const StepPlan &S = gp.steps[k];
    const int lane = c->nchunks > 1 ? k % gp.nlanes : 0;
    launch_basis<double>(s, true, S.basis);
    if (gga) {
      // W = 2 a Phi + b . grad Phi of every spin, at the coefficients of the build
      for (int sp = 0; sp < c->ispin; ++sp)
        launch_bracket_coef(s, Mc, (sp ? c->beta.state : c->state) + p0, np,
                            (sp ? c->beta.coef : c->coef) + (size_t)lane * 4 * Mc);
      if (gp.wbasis) {
        launch_wbasis<double>(s, true, false, false, S.wmat);
        launch_wbasis<double>(s, true, false, true, S.wmat2);
      } else {
        launch_wmat<double>(s, true, false, false, S.wmat);
        launch_wmat<double>(s, true, false, true, S.wmat2);
      }
    }
    const UnitD *unit = c->ispin == 2 ? S.func2.units : S.func.units;
    for (int sp = 0; sp < c->ispin; ++sp) {
      // X = Phi P, Z = W P with P of the last build (P_ref)
      for (int li = 0; li < kLists; ++li)
        launch_xz(s, li % kNumVariants, S.dens[li], sp ? c->beta.Pref : c->Pref,
                  c->gXZ, gga ? 2 : 1, c->ispin, sp);
      launch_bracket(s, gga, c->lmax, unit, Mc, c->n_ranges, c->gXZ,
                     (sp ? c->beta.state : c->state) + p0, np, pm ? pm + p0 : nullptr, c->gpart, c->gsum);
    }
  }
  if (hipGetLastError() != hipSuccess) return fail(c, PGXC_ERR_HIP, "pgxc_gradient: launch failed");
  mark_basis_cached(c, 8, true);
  return PGXC_OK;
}

int pgxc_gradient(pgxc_ctx *c, double *grad) {
  if (!c || !grad) return PGXC_ERR_ARG;
  if (!c->have_state) return fail(c, PGXC_ERR_STATE, "pgxc_gradient before a build on this context");
  int rc = gradient_impl(c, nullptr);
  if (rc) return rc;
  HIPCHK(c, hipMemcpyAsync(grad, c->gsum, 24 * (size_t)c->n_atoms, hipMemcpyDeviceToHost, c->stream));
  HIPCHK(c, hipStreamSynchronize(c->stream));
  return PGXC_OK;
}

int pgxc_gradient_grid(pgxc_ctx *c, const int32_t *owner, double *grad) {
  if (!c || !owner || !grad) return PGXC_ERR_ARG;
  const long npts = c->npts, np = c->npad;
  const int na = c->n_atoms;
  for (long p = 0; p < npts; ++p)
    if (owner[p] < 0 || owner[p] >= na) return fail(c, PGXC_ERR_ARG, "pgxc_gradient_grid: owner out of range");
  std::vector<double> inv((size_t)na * na, 0.0);
  for (int i = 0; i < na; ++i)
    for (int k = 0; k < na; ++k)
      if (i != k) {
        const double dx = c->axyz[3 * i] - c->axyz[3 * k], dy = c->axyz[3 * i + 1] - c->axyz[3 * k + 1],
                     dz = c->axyz[3 * i + 2] - c->axyz[3 * k + 2];
        const double d = std::sqrt(dx * dx + dy * dy + dz * dz);
        if (!(d > 0.0)) return fail(c, PGXC_ERR_ARG, "pgxc_gradient_grid: two atoms at one position");
        inv[(size_t)i * na + k] = 1.0 / d;
      }
  if (!c->have_state) return fail(c, PGXC_ERR_STATE, "pgxc_gradient before a build on this context");
  // work space, kept with the context: caller owners, owners, f per point,
  // inverse distances, per-wave cells, sums and centre lists
  const long waves = becke_grad_waves(na, np);
  size_t off[8] = {0}, bytes[7] = {4 * (size_t)npts, 4 * (size_t)np, 8 * (size_t)np, 8 * inv.size(),
                                   512 * (size_t)waves * na, 24 * (size_t)waves * na, 4 * (size_t)waves * na};
  for (int i = 0; i < 7; ++i) off[i + 1] = off[i] + (size_t)round_up((long)bytes[i], 256);
  int rc;
  if ((rc = dalloc(c, &c->gmov, off[7])) || (rc = dalloc(c, &c->gpm, 3 * (size_t)np))) return rc;
  int *d_caller = (int *)(c->gmov + off[0]), *d_own = (int *)(c->gmov + off[1]);
  double *fp = (double *)(c->gmov + off[2]), *d_inv = (double *)(c->gmov + off[3]);
  double *scr = (double *)(c->gmov + off[4]), *part = (double *)(c->gmov + off[5]);
  int *list = (int *)(c->gmov + off[6]);
  hipStream_t s = c->stream;
  HIPCHK(c, hipMemsetAsync(c->gpm, 0, 24 * (size_t)np, s));
  HIPCHK(c, hipMemcpyAsync(d_inv, inv.data(), 8 * inv.size(), hipMemcpyHostToDevice, s));
  HIPCHK(c, hipMemcpyAsync(d_caller, owner, 4 * (size_t)npts, hipMemcpyHostToDevice, s));
  launch_gather_owner(s, npts, np, c->perm_d, d_caller, d_own);
  // basis-centre term, and w grad f per point (the points move with their atoms)
  if ((rc = gradient_impl(c, c->gpm))) return rc;
  launch_owner_sum(s, na, np, d_own, c->gpm, waves, part, c->gsum);
  // Becke weight derivatives times f
  const uint32_t functional = c->state_functional;
  const bool gga = (functional & (PGXC_XC_PBEX | PGXC_XC_PBEC)) != 0;
  launch_point_f(s, gga, c->ispin == 2, functional, np, np, c->state, c->ispin == 2 ? c->beta.state : c->state, fp);
  launch_becke_grad(s, na, c->atoms, d_inv, np, c->grid, fp, d_own, waves, scr, list, part, c->gsum);
  if (hipGetLastError() != hipSuccess) return fail(c, PGXC_ERR_HIP, "pgxc_gradient_grid: launch failed");
  HIPCHK(c, hipMemcpyAsync(grad, c->gsum, 24 * (size_t)na, hipMemcpyDeviceToHost, s));
  HIPCHK(c, hipStreamSynchronize(s));
  return PGXC_OK;
}

int pgxc_last_stats(const pgxc_ctx *c, double *s5) {
  if (!c || !s5) return PGXC_ERR_ARG;
  for (int i = 0; i < 5; ++i) s5[i] = c->stats[i];
  return PGXC_OK;
}

int pgxc_last_work(const pgxc_ctx *c, double *w3) {
  if (!c || !w3) return PGXC_ERR_ARG;
  w3[0] = c->sum_bn;
  w3[1] = c->sum_n2;
  w3[2] = std::ceil((double)c->npts / kScreenTile);
  return PGXC_OK;
}

int pgxc_last_timing(const pgxc_ctx *c, double *ms6) {
  if (!c || !ms6) return PGXC_ERR_ARG;
  for (int i = 0; i < 6; ++i) ms6[i] = c->timing[i];
  return PGXC_OK;
}

int pgxc_set_schedule(pgxc_ctx *c, int32_t mode, pgxc_costmodel *model) {
  if (!c) return PGXC_ERR_ARG;
  if (check_sched(mode, model))
    return fail(c, PGXC_ERR_ARG, "pgxc_set_schedule: mode 0..2, and a model for PGXC_SCHED_MODEL");
  c->sched.mode = mode;
  c->sched.model = mode == PGXC_SCHED_MODEL ? model : nullptr;
  return PGXC_OK;
}

// ---- state of incremental builds, for checkpoint / restart ----------------
struct StateHeader {
  char magic[8];
  uint64_t geom;
  int64_t nbas, NP, npad, npk, nslot;
  uint32_t functional;
  int32_t ispin;
  double exc, charge;
};
static const char kStateMagic[8] = {'P', 'G', 'X', 'C', 'S', 'T', '0', '1'};

// one block per spin: Pref, Vstate, state
static int64_t state_block(const pgxc_ctx *c) {
  const int64_t npk = (int64_t)c->nbas * (c->nbas + 1) / 2;
  return 8 * ((int64_t)c->NP * c->NP + npk + (int64_t)S_NSLOT * c->npad);
}

static int64_t state_bytes(const pgxc_ctx *c) {
  return (int64_t)sizeof(StateHeader) + c->ispin * state_block(c);
}

int64_t pgxc_state_bytes(const pgxc_ctx *c) { return c ? state_bytes(c) : -PGXC_ERR_ARG; }

int pgxc_save_state(pgxc_ctx *c, void *buf, int64_t bytes) {
  if (!c || !buf) return PGXC_ERR_ARG;
  if (!c->have_state) return fail(c, PGXC_ERR_STATE, "pgxc_save_state: no build has run on this context");
  if (bytes < state_bytes(c)) return fail(c, PGXC_ERR_ARG, "pgxc_save_state: buffer smaller than pgxc_state_bytes");
  HIPCHK(c, hipStreamSynchronize(c->stream));
  StateHeader h{};
  memcpy(h.magic, kStateMagic, 8);
  h.geom = c->geom;
  h.nbas = c->nbas;
  h.NP = c->NP;
  h.npad = c->npad;
  h.npk = (int64_t)c->nbas * (c->nbas + 1) / 2;
  h.nslot = S_NSLOT;
  h.functional = c->state_functional;
  h.ispin = c->ispin;
  h.exc = c->last_exc;
  h.charge = c->last_charge;
  char *o = (char *)buf;
  memcpy(o, &h, sizeof(h));
  o += sizeof(h);
  for (int sp = 0; sp < c->ispin; ++sp) {
    HIPCHK(c, hipMemcpy(o, sp ? c->beta.Pref : c->Pref, 8 * (size_t)c->NP * c->NP, hipMemcpyDeviceToHost));
    o += 8 * (size_t)c->NP * c->NP;
    HIPCHK(c, hipMemcpy(o, sp ? c->beta.Vstate : c->Vstate, 8 * (size_t)h.npk, hipMemcpyDeviceToHost));
    o += 8 * (size_t)h.npk;
    HIPCHK(c, hipMemcpy(o, sp ? c->beta.state : c->state, 8 * (size_t)S_NSLOT * c->npad,
                        hipMemcpyDeviceToHost));
    o += 8 * (size_t)S_NSLOT * c->npad;
  }
  return PGXC_OK;
}

int pgxc_load_state(pgxc_ctx *c, const void *buf, int64_t bytes) {
  if (!c || !buf) return PGXC_ERR_ARG;
  if (bytes < (int64_t)sizeof(StateHeader)) return fail(c, PGXC_ERR_ARG, "pgxc_load_state: buffer too short");
  StateHeader h;
  memcpy(&h, buf, sizeof(h));
  if (memcmp(h.magic, kStateMagic, 8) != 0) return fail(c, PGXC_ERR_ARG, "pgxc_load_state: not a state record");
  if (h.geom != c->geom || h.nbas != c->nbas || h.NP != c->NP || h.npad != c->npad ||
      h.nslot != S_NSLOT || h.npk != (int64_t)c->nbas * (c->nbas + 1) / 2 ||
      (h.ispin != 1 && h.ispin != 2))
    return fail(c, PGXC_ERR_ARG, "pgxc_load_state: the state belongs to another geometry or layout");
  if (bytes < (int64_t)sizeof(StateHeader) + h.ispin * state_block(c))
    return fail(c, PGXC_ERR_ARG, "pgxc_load_state: buffer too short");
  HIPCHK(c, hipStreamSynchronize(c->stream));
  {  // the next density must be set with the state's spin count
    int rc = set_spins(c, h.ispin);
    if (rc) return rc;
  }
  const char *o = (const char *)buf + sizeof(h);
  for (int sp = 0; sp < c->ispin; ++sp) {
    HIPCHK(c, hipMemcpy(sp ? c->beta.Pref : c->Pref, o, 8 * (size_t)c->NP * c->NP, hipMemcpyHostToDevice));
    o += 8 * (size_t)c->NP * c->NP;
    HIPCHK(c, hipMemcpy(sp ? c->beta.Vstate : c->Vstate, o, 8 * (size_t)h.npk, hipMemcpyHostToDevice));
    o += 8 * (size_t)h.npk;
    HIPCHK(c, hipMemcpy(sp ? c->beta.state : c->state, o, 8 * (size_t)S_NSLOT * c->npad,
                        hipMemcpyHostToDevice));
    o += 8 * (size_t)S_NSLOT * c->npad;
  }
  c->state_functional = h.functional;
  c->last_exc = h.exc;
  c->last_charge = h.charge;
  c->have_state = 1;
  return PGXC_OK;
}

int pgxc_set_lanes(pgxc_ctx *c, int32_t lanes) {
  if (!c) return PGXC_ERR_ARG;
  if (lanes < 1 || lanes > 2) return fail(c, PGXC_ERR_ARG, "pgxc_set_lanes: lanes must be 1 or 2");
  c->nlanes = std::min<int>(lanes, c->nlanes_cap);
  return PGXC_OK;
}

int pgxc_set_item_log(pgxc_ctx *c, int32_t on) {
  if (!c) return PGXC_ERR_ARG;
  c->sched.log = on ? 1 : 0;
  return PGXC_OK;
}

int64_t pgxc_item_log(pgxc_ctx *c, double *features, double *us, int64_t cap) {
  if (!c) return -PGXC_ERR_ARG;
  return read_item_log(c->plan, c->stream, features, us, cap);
}

int pgxc_destroy(pgxc_ctx *c) {
  if (!c) return PGXC_OK;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  if (c->stream2) (void)hipStreamSynchronize(c->stream2);
  free_plan(c->plan);
  free_plan(c->plan_e);
  free_plan(c->plan_g);
  {
    std::lock_guard<std::mutex> lk(g_cache_mu);
    g_cache_bytes[c->device] -= c->phic_bytes[0] + c->phic_bytes[1];
  }
  void *bufs[] = {c->orb, c->grid, c->atoms, c->shells, c->ranges, c->ratoms, c->tabd, c->tabf, c->P, c->Pref,
                  c->D, c->phi, c->W, c->part, c->coef, c->Hc, c->HS, c->state,
                  c->Vstate, c->Vout, c->epart, c->nbt, c->sig8, c->sshells, c->d_fpos, c->d_finv,
                  c->phic[0], c->phic[1], c->tl_off, c->tl, c->tf_off, c->tfl, c->tfb, c->tlm, c->su_off, c->su, c->sumask,
                  c->ho, c->pos, c->rbits, c->di, c->pi, c->bi, c->bfl, c->gXZ, c->gpart, c->gsum, c->gpm, c->gmov, c->perm_d, c->beta.P, c->beta.Pref, c->beta.D,
                  c->beta.W, c->beta.part, c->beta.coef, c->beta.Hc, c->beta.HS, c->beta.state,
                  c->beta.Vstate, c->beta.Vout, c->eterm};
  for (void *b : bufs) dfree(b);
  for (auto &e : c->ev)
    if (e) (void)hipEventDestroy(e);
  if (c->stream) (void)hipStreamDestroy(c->stream);
  if (c->stream2) (void)hipStreamDestroy(c->stream2);
  if (c->fork) (void)hipEventDestroy(c->fork);
  if (c->join) (void)hipEventDestroy(c->join);
  c->pin.release();
  delete c;
  return PGXC_OK;
}

}  // extern "C"

// ------------------------------------------------------------------ batches
struct pgxc_batch {
  std::vector<pgxc_ctx *> mols;
  hipStream_t stream = nullptr, stream2 = nullptr;  // the two lanes of its plans
  hipEvent_t fork = nullptr, join = nullptr;
  std::string err;
  Plan *plan = nullptr;
  std::vector<double> prio;
  long order_version = -1;
  hipEvent_t e0 = nullptr, e1 = nullptr;
  double last_ms = 0;
  Sched sched;
};

extern "C" {

const char *pgxc_batch_last_error(const pgxc_batch *b) { return b ? b->err.c_str() : "null batch"; }

int pgxc_batch_create(pgxc_batch **out, int32_t n, pgxc_ctx *const *ctxs) {
  if (!out) return PGXC_ERR_ARG;
  *out = nullptr;
  if (n <= 0 || !ctxs) return PGXC_ERR_ARG;
  pgxc_batch *b = new pgxc_batch();
  *out = b;
  int dev = -1;
  for (int i = 0; i < n; ++i) {
    if (!ctxs[i]) {
      b->err = "pgxc_batch_create: null context " + std::to_string(i);
      return PGXC_ERR_ARG;
    }
    if (dev >= 0 && ctxs[i]->device != dev) {
      b->err = "pgxc_batch_create: contexts on different devices";
      return PGXC_ERR_ARG;
    }
    dev = ctxs[i]->device;
    for (int j = 0; j < i; ++j)
      if (ctxs[j] == ctxs[i]) {
        b->err = "pgxc_batch_create: context listed twice";
        return PGXC_ERR_ARG;
      }
    b->mols.push_back(ctxs[i]);
  }
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess ||
      hipStreamCreateWithFlags(&b->stream2, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreateWithFlags(&b->fork, hipEventDisableTiming) != hipSuccess ||
      hipEventCreateWithFlags(&b->join, hipEventDisableTiming) != hipSuccess ||
      hipEventCreate(&b->e0) != hipSuccess || hipEventCreate(&b->e1) != hipSuccess) {
    (void)hipGetLastError();
    b->err = "pgxc_batch_create: stream/event creation failed";
    return PGXC_ERR_HIP;
  }
  return PGXC_OK;
}

int pgxc_batch_set_priority(pgxc_batch *b, const double *cost) {
  if (!b) return PGXC_ERR_ARG;
  if (cost)
    b->prio.assign(cost, cost + b->mols.size());
  else
    b->prio.clear();
  ++b->order_version;
  return PGXC_OK;
}

int pgxc_batch_build(pgxc_batch *b, uint32_t functional, int32_t precision, int32_t use_graph) {
  if (!b) return PGXC_ERR_ARG;
  const int nm = (int)b->mols.size();
  std::vector<int> incr(nm, 0);
  for (int m = 0; m < nm; ++m) {
    int rc = validate_build(b->mols[m], functional, precision, incr[m]);
    if (rc) {
      b->err = "molecule " + std::to_string(m) + ": " + b->mols[m]->err;
      return rc;
    }
  }
  const bool gga = (functional & (PGXC_XC_PBEX | PGXC_XC_PBEC)) != 0;
  const size_t elem = precision == PGXC_PREC_FP64 ? 8 : 4;
  hipStream_t s = b->stream;
  for (int m = 0; m < nm; ++m) {
    pgxc_ctx *c = b->mols[m];
    int rc = ensure_work(c, elem, s, gga);
    if (rc) {
      b->err = "molecule " + std::to_string(m) + ": " + c->err;
      return rc;
    }
  }
  int rc = get_plan(b->mols, functional, precision, incr, b->prio, b->order_version, b->sched,
                    b->plan, b->mols[0]);
  if (rc) {
    b->err = b->mols[0]->err;
    return rc;
  }
  Plan &pl = *b->plan;
  if (use_graph && !pl.graph) {
    hipError_t e = hipStreamBeginCapture(s, hipStreamCaptureModeThreadLocal);
    if (e == hipSuccess) {
      if (elem == 8)
        launch_plan<double>(s, b->stream2, b->fork, b->join, pl, gga, nullptr);
      else
        launch_plan<float>(s, b->stream2, b->fork, b->join, pl, gga, nullptr);
      e = hipStreamEndCapture(s, &pl.graph_src);
      if (e == hipSuccess) e = hipGraphInstantiate(&pl.graph, pl.graph_src, nullptr, nullptr, 0);
    }
    if (e != hipSuccess) {
      (void)hipGetLastError();
      b->err = std::string("hipGraph capture: ") + hipGetErrorString(e);
      return PGXC_ERR_HIP;
    }
  }
  if (hipEventRecord(b->e0, s) != hipSuccess) {
    (void)hipGetLastError();
    b->err = "hipEventRecord failed";
    return PGXC_ERR_HIP;
  }
  if (use_graph) {
    if (hipGraphLaunch(pl.graph, s) != hipSuccess) {
      (void)hipGetLastError();
      b->err = "hipGraphLaunch failed";
      return PGXC_ERR_HIP;
    }
  } else if (elem == 8) {
    launch_plan<double>(s, b->stream2, b->fork, b->join, pl, gga, nullptr);
  } else {
    launch_plan<float>(s, b->stream2, b->fork, b->join, pl, gga, nullptr);
  }
  (void)hipEventRecord(b->e1, s);
  hipError_t e = hipGetLastError();
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  if (e != hipSuccess) {
    (void)hipGetLastError();
    b->err = std::string("batch build: ") + hipGetErrorString(e);
    return PGXC_ERR_HIP;
  }
  float t = 0;
  (void)hipEventElapsedTime(&t, b->e0, b->e1);
  b->last_ms = t;
  for (int m = 0; m < nm; ++m) {
    pgxc_ctx *c = b->mols[m];
    rc = collect(c, s, functional, precision);
    if (rc) {
      b->err = c->err;
      return rc;
    }
    c->timing[5] = t;
    mark_basis_cached(c, elem, gga);
  }
  return PGXC_OK;
}

int pgxc_batch_set_schedule(pgxc_batch *b, int32_t mode, pgxc_costmodel *model) {
  if (!b) return PGXC_ERR_ARG;
  if (check_sched(mode, model)) {
    b->err = "pgxc_batch_set_schedule: mode 0..2, and a model for PGXC_SCHED_MODEL";
    return PGXC_ERR_ARG;
  }
  b->sched.mode = mode;
  b->sched.model = mode == PGXC_SCHED_MODEL ? model : nullptr;
  return PGXC_OK;
}

int pgxc_batch_set_item_log(pgxc_batch *b, int32_t on) {
  if (!b) return PGXC_ERR_ARG;
  b->sched.log = on ? 1 : 0;
  return PGXC_OK;
}

int64_t pgxc_batch_item_log(pgxc_batch *b, double *features, double *us, int64_t cap) {
  if (!b) return -PGXC_ERR_ARG;
  return read_item_log(b->plan, b->stream, features, us, cap);
}

int pgxc_batch_last_ms(const pgxc_batch *b, double *ms) {
  if (!b || !ms) return PGXC_ERR_ARG;
  *ms = b->last_ms;
  return PGXC_OK;
}

int pgxc_batch_destroy(pgxc_batch *b) {
  if (!b) return PGXC_OK;
  if (b->stream) (void)hipStreamSynchronize(b->stream);
  if (b->stream2) (void)hipStreamSynchronize(b->stream2);
  free_plan(b->plan);
  if (b->e0) (void)hipEventDestroy(b->e0);
  if (b->e1) (void)hipEventDestroy(b->e1);
  if (b->fork) (void)hipEventDestroy(b->fork);
  if (b->join) (void)hipEventDestroy(b->join);
  if (b->stream) (void)hipStreamDestroy(b->stream);
  if (b->stream2) (void)hipStreamDestroy(b->stream2);
  delete b;
  return PGXC_OK;
}

constexpr int64_t kBeckePart = 1 << 18;

int pgxc_becke_weights(int32_t n_atoms, const double *atom_xyz, int64_t npts, const double *pts,
                       const int32_t *owner, const double *w_atomic, double *w_out) {
  if (n_atoms <= 0 || npts < 0 || !atom_xyz ||
      (npts > 0 && (!pts || !owner || !w_atomic || !w_out)))
    return PGXC_ERR_ARG;
  if (npts == 0) return PGXC_OK;
  for (int64_t p = 0; p < npts; ++p)
    if (owner[p] < 0 || owner[p] >= n_atoms) return PGXC_ERR_ARG;
  for (int i = 0; i < n_atoms; ++i)
    for (int k = 0; k < i; ++k) {
      const double dx = atom_xyz[3 * i] - atom_xyz[3 * k];
      const double dy = atom_xyz[3 * i + 1] - atom_xyz[3 * k + 1];
      const double dz = atom_xyz[3 * i + 2] - atom_xyz[3 * k + 2];
      if (!(dx * dx + dy * dy + dz * dz > 0.0)) return PGXC_ERR_ARG;  // coincident centres
    }
  // Many centres and points go in parts of kBeckePart: a part's upload (from the
  // caller's pageable memory, which the copy has read when it returns) runs while
  // the parts before it are computed, and its weights come back while those after
  // it are.  The kernel of few centres is a small share of its transfers, and one
  // part has nothing to overlap: one stream and no events then (a call of 3 atoms
  // with 41 000 points 250 us with them, 173 without).
  const int64_t per = n_atoms > kAllPairs ? kBeckePart : std::max<int64_t>(npts, 1);
  const size_t ninv = (size_t)n_atoms * n_atoms, na3 = 3 * (size_t)n_atoms;
  const int64_t parts = (npts + per - 1) / per;
  const bool overlap = parts > 1;
  double *dev = nullptr;  // centres, inverse distances, points (3), weights in, weights out; owners
  hipStream_t s = nullptr, s2 = nullptr;
  std::vector<hipEvent_t> up((size_t)(overlap ? parts : 0), nullptr), done(up);
  int rc = PGXC_OK;
  auto chk = [&](hipError_t e) {
    if (e != hipSuccess) (void)hipGetLastError();
    if (e != hipSuccess && rc == PGXC_OK)
      rc = e == hipErrorOutOfMemory ? PGXC_ERR_NOMEM : PGXC_ERR_HIP;
    return rc == PGXC_OK;
  };
  chk(hipStreamCreateWithFlags(&s, hipStreamNonBlocking));
  if (overlap) chk(hipStreamCreateWithFlags(&s2, hipStreamNonBlocking));
  chk(hipMalloc((void **)&dev, 8 * (na3 + ninv) + 44 * (size_t)npts + 8));
  for (size_t i = 0; i < up.size() && rc == PGXC_OK; ++i) {
    chk(hipEventCreateWithFlags(&up[i], hipEventDisableTiming));
    chk(hipEventCreateWithFlags(&done[i], hipEventDisableTiming));
  }
  hipStream_t sc = overlap ? s2 : s;  // the transfers' stream
  double *d_a = dev, *d_inv = d_a + na3, *d_p = d_inv + ninv, *d_w = d_p + 3 * npts, *d_o = d_w + npts;
  int *d_own = (int *)(d_o + npts);
  if (rc == PGXC_OK) {
    chk(hipMemcpyAsync(d_a, atom_xyz, 8 * na3, hipMemcpyHostToDevice, s));
    launch_inv_dist(s, n_atoms, d_a, d_inv);
  }
  for (int64_t i = 0; i < parts + 2 && rc == PGXC_OK; ++i) {
    if (i < parts) {
      const int64_t p0 = i * per, n = std::min<int64_t>(per, npts - p0);
      const int nd = overlap ? 3 : 1;  // the coordinates of all points lie in one piece
      for (int d = 0; d < nd; ++d)
        chk(hipMemcpyAsync(d_p + d * npts + p0, pts + d * npts + p0, 24 * (size_t)n / nd, hipMemcpyHostToDevice, sc));
      chk(hipMemcpyAsync(d_w + p0, w_atomic + p0, 8 * (size_t)n, hipMemcpyHostToDevice, sc));
      chk(hipMemcpyAsync(d_own + p0, owner + p0, 4 * (size_t)n, hipMemcpyHostToDevice, sc));
      if (overlap) {
        chk(hipEventRecord(up[(size_t)i], sc));
        chk(hipStreamWaitEvent(s, up[(size_t)i], 0));
      }
      launch_becke(s, n_atoms, d_a, d_inv, (long)n, (long)npts, d_p + p0, d_own + p0, d_w + p0, d_o + p0);
      chk(hipGetLastError());
      if (overlap) chk(hipEventRecord(done[(size_t)i], s));
    }
    if (i >= 2) {
      const int64_t p0 = (i - 2) * per, n = std::min<int64_t>(per, npts - p0);
      if (overlap) chk(hipStreamWaitEvent(sc, done[(size_t)(i - 2)], 0));
      chk(hipMemcpyAsync(w_out + p0, d_o + p0, 8 * (size_t)n, hipMemcpyDeviceToHost, sc));
    }
  }
  if (s2) chk(hipStreamSynchronize(s2));
  if (s) chk(hipStreamSynchronize(s));
  dfree(dev);
  for (auto *v : {&up, &done})
    for (hipEvent_t e : *v)
      if (e) (void)hipEventDestroy(e);
  if (s) (void)hipStreamDestroy(s);
  if (s2) (void)hipStreamDestroy(s2);
  return rc;
}

// ---- Becke weights without allocation: file-scope scratch -----------------
// The table of inverse pair distances lives in `scratch`, one copy per
// device, held until the process ends.  Host code never passes the array's
// name to a kernel (it is a host-side stand-in there): each device's address
// is taken once with hipGetSymbolAddress and kept in g_scratch_ptr.
constexpr int kNoAllocMaxAtoms = 1024;  // 8 MiB of scratch per device
constexpr int kNoAllocMaxDevices = 64;
static __device__ __align__(256) double scratch[(size_t)kNoAllocMaxAtoms * kNoAllocMaxAtoms];
static std::mutex g_scratch_mu;
static double *g_scratch_ptr[kNoAllocMaxDevices];
static int free_fail(int code, const char *msg) {
  if (code == PGXC_ERR_HIP) (void)hipGetLastError();
  snprintf(g_free_err, sizeof(g_free_err), "%s", msg);
  return code;
}

int pgxc_becke_weights_noalloc(int32_t n_atoms, const double *atom_xyz, int64_t npts,
                               const double *pts, const int32_t *owner, const double *w_atomic,
                               double *w_out, void *stream) {
  if (n_atoms <= 0 || npts < 0 || !atom_xyz ||
      (npts > 0 && (!pts || !owner || !w_atomic || !w_out)))
    return free_fail(PGXC_ERR_ARG, "pgxc_becke_weights_noalloc: null pointer or negative size");
  if (n_atoms > kNoAllocMaxAtoms)
    return free_fail(PGXC_ERR_ARG, "pgxc_becke_weights_noalloc: more than 1024 atoms (the scratch "
                                   "table holds 1024 x 1024 inverse distances)");
  if (npts == 0) return PGXC_OK;
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kNoAllocMaxDevices)
    return free_fail(PGXC_ERR_HIP, "pgxc_becke_weights_noalloc: no usable current device");
  double *ptr = nullptr;
  {
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (!g_scratch_ptr[dev]) {
      void *a = nullptr;
      if (hipGetSymbolAddress(&a, HIP_SYMBOL(scratch)) != hipSuccess || !a)
        return free_fail(PGXC_ERR_HIP, "pgxc_becke_weights_noalloc: hipGetSymbolAddress(scratch)");
      g_scratch_ptr[dev] = (double *)a;
    }
    ptr = g_scratch_ptr[dev];
  }
  hipStream_t s = (hipStream_t)stream;
  launch_inv_dist(s, n_atoms, atom_xyz, ptr);  // every entry rewritten: nothing to clear
  launch_becke(s, n_atoms, atom_xyz, ptr, (long)npts, (long)npts, pts, owner, w_atomic, w_out);
  if (hipGetLastError() != hipSuccess)
    return free_fail(PGXC_ERR_HIP, "pgxc_becke_weights_noalloc: kernel launch failed");
  return PGXC_OK;
}

}  // extern "C"
