// Internal declarations shared by the HIP kernels and the C-ABI layer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

struct pgxc_costmodel;

namespace pgxc {

typedef double d4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

constexpr int kLMax = 4;      // highest angular momentum of a shell
constexpr int kMaxContr = 8;  // contracted functions per shell
// per atom at most: shells, primitives and contraction coefficients
constexpr int kAtomShells = 16, kAtomPrims = 256, kAtomContr = 1024;
// A basis item evaluates one 256-point block against a range of atoms,
// consecutive in shell order: at most kRangeAtoms atoms and kRangeShells shells
// (a word of flags; an atom of the per-atom maximum fits).
constexpr int kRangeAtoms = 8, kRangeShells = 32;
constexpr int kPB = 4;  // rows of a shell's table are padded to this many primitives
constexpr int kThreads = 256; // 4 wave64 per workgroup everywhere
constexpr double kFar = 1.0e6;  // coordinate of padding points (all exps cut off)

// One shell = one (atom, l) block of unique_atom_basis_type.
struct ShellD {
  int atom, l, n_exp, n_unc, n_contr, exp_off, tab, func_off;  // tab: its table in tabd / tabf
};

// One centre with the contiguous shell range it carries.
struct AtomD {
  double x, y, z;
  int shell_begin, shell_end, lmax, pad;
};

// A range of atoms for the basis stage: ratoms[atom_begin .. +n_atoms) are
// its atoms, in shell order; their shells (shell_begin, n_shells) are contiguous.
struct RangeD {
  int atom_begin, n_atoms, shell_begin, n_shells;
};

// Per-point state kept across builds (incremental mode), SoA of length npad.
enum StateSlot { S_RHO = 0, S_GX, S_GY, S_GZ, S_A, S_BX, S_BY, S_BZ, S_NSLOT };

// ---- work lists ----------------------------------------------------------
// A unit is one grid chunk of one molecule: Mc points (multiple of 256) with
// the molecule's basis, its density operand and the chunk's work buffers.
struct UnitD {
  const double *gx, *gy, *gz, *gw;  // grid of the unit's points (offset to its first point)
  const AtomD *atoms;
  const ShellD *shells;
  const double *tabd;  // the shells' exponents, norms and coefficients, in FP64
  const float *tabf;   // and in FP32
  const RangeD *ranges;  // the basis stage's atom ranges
  const int *ratoms;     // atoms in shell order (the ranges index it)
  void *phi;        // [4][NP][Mc] values, d/dx, d/dy, d/dz (T)
  void *W;          // [NP][Mc] (T); split-BF16 builds: bf16 hi / lo planes [2][NP][Mc]
  const void *D;    // [NP][NP] density operand (T); split-BF16: transposed hi / lo planes
  double *part;     // [shares of the columns][4][Mc] density partials
  double *coef;     // [4][Mc] potential coefficients a, b
  double *state;    // [S_NSLOT][npad] molecule state, offset to the unit's first point
  double *epart;    // [Mc/256][2] block sums of w f and w rho (offset to the unit)
  // open-shell (ispin = 2) molecules: the alpha spin's unit also points at
  // the beta spin's partials, coefficients and state (the spin functional
  // reads both); nullptr otherwise
  const double *part2;
  double *coef2, *state2;
  void *W2;         // and the beta spin's W, written by the same W pass
  double *eterm;    // [Mc/256][5] block sums of the energy terms and the charge
  double *Hc;       // potential partials of the unit's splits, split s at ho[s]:
  const long *ho;   // its functions x its functions (padded to blocks of 16)
  // Work of the contractions, over gathered runs of 8 functions and gathered
  // functions (all of them when screening is off).  ditems / pitems: the
  // unit's density items (tile << 8 | share of its columns) and potential
  // items (split << 20 | row chunk << 10 | column chunk).  tl_off / tl: per
  // 128-point tile of the unit, its ascending run list, the density's K
  // (tl_off offset to the unit's first tile, values index tl); tf_off / tfl:
  // the same for its functions (those of the shells not cut off on the
  // tile), the density's output columns.
  // su_off / su: per point split of the unit, the union of its tiles'
  // functions, the potential's rows and columns in chunks of tile functions.
  const uint32_t *ditems, *pitems;
  const int *tl_off, *su_off, *tf_off;
  const uint16_t *tl, *su, *tfl;
  const uint32_t *tfb;  // the tiles' functions as bitmaps, nwf words per tile
  // per entry of tl: its run's functions in the tile's list (bit j: function
  // 8 r + j); the density contraction stages zeros for the others, which the
  // basis stage does not write
  const uint8_t *tlm;
  // per entry of su: bit t set when its function is in the list of the
  // split's tile t (a split has at most 32), else W and Phi are not written
  // there and count as 0
  const uint32_t *sumask;
  int nwf, pad_f;
  // Basis stage over the blocks the other stages read.  bitems: basis items
  // (256-point block << 16 | atom range) that write some block, block by block,
  // with bflags: per item a word for each of the block's two tiles, bit j: the
  // values and gradients of the range's shell j are read there.
  const uint32_t *bitems, *bflags;
  long nbi;
  long Mc, npad;
  int n_atoms, n_ranges, NP, nsplit, incremental, pad_n;
  uint32_t mask;
  int icols, dcols;  // most columns of a density item, and of a partial: kPartCols or (split-BF16) icols
  long ndi, npi;  // density / potential items of the unit
};

// Per-molecule descriptors of the operand preparation and the final packing.
struct PackD {
  const double *HS;  // [nseg][NP][NP] symmetric sums of partials (lower 32 x 32 tiles)
  double *Vout, *Vstate;
  const double *P;
  double *Pref;
  void *D;
  const int *fpos;  // internal position of each basis function (caller order)
  long n, NP;
  int nseg, incremental;
};

// Sums of a molecule's potential partials (k_fold): chunks chunk0, chunk0 +
// step, ... (nchunks of them), of their mask bytes the share seg of nseg, into
// out[NP][NP] (added to it when acc is set).  Split s's partial lies at ho[s]
// of Hc.  pos[split][NP]: a
// function's place in the split's list (0xffff: absent); rbits[row block of 32
// functions][nbytes]: a bit per split, whether it has any of the block's
// functions (bytes_c bytes per chunk).
struct FoldD {
  const double *Hc;
  const long *ho;
  const int *su_off;
  const uint16_t *pos;
  const uint8_t *rbits;
  double *out;
  long NP;
  int nsplit, bytes_c, nbytes, chunk0, step, nchunks, seg, nseg, acc, pad;
};

// One launch's items: prefix offsets base[0..nu] over units, optional order.
// Queues (ctr != nullptr, contraction stages only): positions are split into
// kQueues contiguous ranges qbeg[q] .. qbeg[q+1]-1 of about equal predicted
// cost; workgroup b drains queue b % kQueues (the XCD it runs on), taking the
// next position from the counter ctr[q], then helps with the queues after
// it.  tlog (optional): per item, the
// workgroup's wall-clock ticks spent on it.
constexpr int kQueues = 8;
struct StageList {
  const UnitD *units;
  int nu;
  const long *base;
  const int *order;
  long total;
  int *ctr;
  const long *qbeg;
  uint32_t *tlog;
  int lmax;  // basis lists: the largest angular momentum of their atoms
};

// ---- launchers (kernels: xc_kernels.hip; the contractions' xc_contract.h and
// xc_bf16x3.hip) --------------------------------------------------------------
template <typename T>
void launch_basis(hipStream_t s, bool grad, const StageList &L);
// W over the basis items, the basis evaluated again (split: stored as bf16 hi / lo
// planes; two: both spins of open-shell units)
template <typename T>
void launch_wbasis(hipStream_t s, bool grad, bool split, bool two, const StageList &L);
// var = contraction variant: 0 (K step 16, 2 LDS stages), 1 (32, 1), 2 (32, 2);
// tf = chunk of functions of the potential (64, 96 or 128) and icols = columns of
// the split-BF16 density's items (128 or 256), the same for every unit of a list
constexpr int kNumVariants = 3;
template <typename T>
void launch_density(hipStream_t s, bool grad, int var, const StageList &L);
void launch_functional(hipStream_t s, bool gga, const StageList &L);
void launch_functional_spin(hipStream_t s, bool gga, const StageList &L);
// energy terms only (no coefficients, state untouched); spin: open-shell units
void launch_energy(hipStream_t s, bool gga, bool spin, const StageList &L);
// W from the stored basis values (two: both spins' W, W2 from coef, coef2, from
// one read)
template <typename T>
void launch_wmat(hipStream_t s, bool grad, bool split, bool two, const StageList &L);
template <typename T>
void launch_potential(hipStream_t s, int tf, int var, const StageList &L);
void launch_density_bf16x3(hipStream_t s, bool grad, int icols, const StageList &L);
void launch_potential_bf16x3(hipStream_t s, int tf, const StageList &L);
void launch_fold(hipStream_t s, const FoldD *folds, int n, const long *base, long total);
void launch_pack(hipStream_t s, const PackD *mols, int nm, const long *base, long total,
                 const long *prep_base, long prep_total);
unsigned contraction_grid(const StageList &L, int per_cu);

// cost model internals used by the planner (cost_model.hip)
long costmodel_version(const pgxc_costmodel *m);
int costmodel_features(const pgxc_costmodel *m);
// mode of the density operand: 0 FP64, 1 FP32, 2 split-BF16 planes of D^T; also
// clears the nctr queue counters of the plan
void launch_prep(hipStream_t s, const PackD *mols, int nm, const long *base, long total,
                 int mode, int *ctr, int nctr);

// item counts per unit, shared by the planner and the kernels' decoding
inline long items_functional(long Mc) { return Mc / kThreads; }
inline long items_wmat(long Mc, int NP) { return (Mc / (4 * kThreads)) * (NP / 16); }
// chunks are whole multiples of this many points; point splits of the
// potential contraction have kSplitPts or fewer (setup_screen picks), so at
// most 32 tiles
constexpr int kSplitPts = 2048;
constexpr int kMinSplitPts = 256;

// ---- screening ------------------------------------------------------------
// A radial factor is exactly zero where alpha r^2 >= 50 (the cut-off of
// ParaGauss's radial, modules/orbital_module.f90:1839-1855), so a shell is
// zero on a set of points when alpha_min r^2 >= 50 at every one of them.
// Granularity: 32-point groups x runs of 8 functions.  The contractions work
// on gathered runs: a 128-point tile contracts over the runs marked on any of
// its groups, a point split over the union of its groups' runs; the terms
// left out are exact zeros.
constexpr int kGroup = 32;
constexpr int kRun = 8;
constexpr int kScreenTile = 128;       // point tile of the density contraction
// A density item takes at most 128 or 256 of its tile's functions as columns (a
// context's choice, UnitD::icols); the FP64/FP32 kernels form them in chunks of
// kPartCols, a partial each.
constexpr int kPartCols = 64;
constexpr int kMaxRuns = 1024;         // runs of 8 functions per molecule (NP <= 8192)
constexpr int kMaxShells = 8192;       // shells per molecule
constexpr double kCutoff = 50.0 * (1.0 + 1.0e-6);  // margin: a superset in every precision
struct ScreenShell {
  double amin;                 // smallest exponent of the shell
  int atom, func_off, nfunc, pad;
};
void launch_screen(hipStream_t s, long ntiles_pts, const double *gx, const double *gy,
                   const double *gz, int n_atoms, const AtomD *atoms, int n_shells,
                   const ScreenShell *shells, int n8, int *nb, uint32_t *sig8,
                   uint32_t *smark);

// P = C diag(occ) C^T into an NP x NP padded array (C in caller order; finv:
// caller index of each internal function)
void launch_copy(hipStream_t s, const double *src, double *dst, long n);
void launch_form_density(hipStream_t s, const double *C, const double *occ, const int *finv, int n,
                         int nocc, int NP, double *P);

// Nuclear gradient.  launch_xz: X = Phi P (plane 0) and, for nplanes = 2, Z = W P
// (plane 1) into XZ[plane][f][p] over a density list's items (tile x function
// chunks), for the tiles' functions only; units u with u % nspin == spin.
void launch_xz(hipStream_t s, int var, const StageList &L, const double *P, double *XZ,
               int nplanes, int nspin, int spin);
// coef = 2 a, b from the per-point state; the W pass over it forms Z's operand
void launch_bracket_coef(hipStream_t s, long Mc, const double *st, long np, double *coef);
// the basis-centre term of one chunk added to grad[atom][3] (caller atoms), w
// grad f per point to pm when given; part: 96 doubles per basis item
void launch_bracket(hipStream_t s, bool gga, int lmax, const UnitD *unit, long Mc, int n_ranges,
                    const double *XZ, const double *st, long np, double *pm, double *part,
                    double *grad);
// With the grid moving: own = owner of each internal point; pm summed by owner;
// f per point from the state (st2: the beta spin's, spin builds); the Becke
// weight derivatives times w f (scr: 64 doubles, list: one entry per wave and
// atom; part: 3 doubles per wave and atom)
void launch_gather_owner(hipStream_t s, long npts, long np, const int *perm, const int *owner, int *own);
void launch_owner_sum(hipStream_t s, int na, long np, const int *owner, const double *pm, long waves,
                      double *part, double *grad);
void launch_point_f(hipStream_t s, bool gga, bool spin, uint32_t mask, long Mc, long npad,
                    const double *st, const double *st2, double *fp);
long becke_grad_waves(int na, long np);
void launch_becke_grad(hipStream_t s, int na, const AtomD *atoms, const double *inv_dist, long np,
                       const double *grid, const double *fp, const int *owner, long waves,
                       double *scr, int *list, double *part, double *grad);

// Becke partition weights of points owned by atoms (grid generation)
void launch_inv_dist(hipStream_t s, int na, const double *axyz, double *inv);
// up to kAllPairs centres every pair is formed: kernel on molecules' grids of 15 to
// 300 thousand points, all pairs / near centres first, 3 atoms 9 / 10.5 us, 8
// 19 / 24, 11 40 / 47, 12 46 / 49, 13 54 / 55, 14 73 / 69, 16 94 / 80, 24 263 / 172
constexpr int kAllPairs = 12;
// npts points with coordinates stride apart
void launch_becke(hipStream_t s, int na, const double *axyz, const double *inv_dist, long npts,
                  long stride, const double *pts, const int *owner, const double *wat, double *wout);

}  // namespace pgxc
