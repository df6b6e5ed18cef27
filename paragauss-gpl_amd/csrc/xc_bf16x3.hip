// Split-BF16 contractions ("bf16x3") for gfx950.
//
// Every FP32 operand x is split as
//   hi = bf16(x), lo = bf16(x - hi)
// and a product is formed from three v_mfma_f32_16x16x32_bf16 passes,
//   a*b ~ a_lo*b_hi + a_hi*b_lo + a_hi*b_hi,   FP32 accumulation,
// dropping a_lo*b_lo (relative 2^-16).  W (k_wbasis) and D^T (k_prep) are
// stored split and k-contiguous, so their staging is a copy of 16-byte
// vectors into LDS; the basis values are read in FP32 (as stored, points
// contiguous) and split while they are staged, k-contiguous for the
// potential and transposed for the density.
// Items, partials and lists as for the FP32 and FP64 contractions
// (xc_contract.h); K advances 32 per MFMA.
#include <type_traits>

#include "pgxc_internal.h"
#include "xc_device.h"

namespace pgxc {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

// 16x16x32 bf16 operand placement (wave64): A(i,k) in lane i + 16 (k / 8),
// element k % 8; B(k,j) in lane j + 16 (k / 8), element k % 8.  Result as the
// FP32 16x16x4 MFMA.
__device__ __forceinline__ f4 mfma_bf16(bf16x8 a, bf16x8 b, f4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

constexpr int kXBK = 32;       // K per stage
constexpr int kXBM = 128;
template <int BM, int BN>
struct XStage {
  static constexpr int n = 2 * BM * kXBK + 2 * BN * kXBK;
};
// Place (bf16 elements) of k run c (8 k, 16 bytes) of row r in a stage: the four
// runs of a row change places by (r / 4) % 4, so that the 16 rows an MFMA
// operand read touches lie on all banks without padding (64 KB for two stages
// of 128 x 128, so two workgroups share a CU).
__device__ __forceinline__ int lds_at(int r, int c) { return r * kXBK + 8 * (c ^ ((r >> 2) & 3)); }

typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef const u32x4 __attribute__((address_space(1))) *gvec;

// Staging of an operand stored split and k-contiguous (bf16 hi and lo planes
// at the same offsets); per stage R rows x 32 k x 2 planes, moved as 16-byte
// vectors (runs of 8).  A thread's vectors keep their rows for the whole
// item and all take k-run c = threadIdx.x & 3 of a step, so an element offset
// is row part + k part: the row pointers (plane included) are set once per
// item, and a step supplies one k offset.  Loads are unconditional global
// loads (a missing row or k run reads the plane's first vector instead) and
// the zeros are applied when the vector is written to LDS, so no load sits in
// a branch and the loads of later steps stay in flight.
template <int R, int NT = kThreads>
struct PSOperand {
  struct Src {
    const __bf16 *hi, *lo;
  };
  static constexpr int NV = R * (kXBK / 8) * 2;  // 16-byte vectors per stage
  static constexpr int PER = NV / NT;
  static_assert(PER * NT == NV, "whole vectors per thread");
  static_assert(NT % 4 == 0, "k run = threadIdx.x & 3");
  const __bf16 *row[PER];  // plane + row offset of vector e, nullptr: row absent
  const __bf16 *dummy;
  unsigned tm[PER];  // vector e's row: bit t set when it can be nonzero on tile t
  long kbase;        // k offset of tile 0
  u32x4 v[2][PER];
  unsigned ok[2];

  __device__ __forceinline__ static void place(int idx, int &plane, int &r, int &c) {
    plane = idx / (R * 4);
    const int rem = idx % (R * 4);
    r = rem >> 2;
    c = rem & 3;
  }
  // rowf(r): element offset of row r (k = 0), or -1; maskf(r): the 128-k
  // tiles from k = kb on where row r can be nonzero (bit t: tile t, at most
  // 32 tiles); a row's steps on other tiles stage zeros without reading it
  template <class RowF, class MaskF>
  __device__ __forceinline__ void init(const Src &S, const RowF &rowf, const MaskF &maskf, long kb) {
    dummy = S.hi;
    kbase = kb;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      int plane, r, c;
      place(threadIdx.x + NT * e, plane, r, c);
      const long o = rowf(r);
      row[e] = o >= 0 ? (plane ? S.lo : S.hi) + o : nullptr;
      tm[e] = maskf(r);
    }
  }
  // kofs(kt, c): element offset of k run c of step kt, or -1; steps past
  // ksteps load zeros
  template <int SL, class KOfs>
  __device__ __forceinline__ void load(const KOfs &kofs, int kt, int ksteps) {
    const long ko = kt < ksteps ? kofs(kt, (int)(threadIdx.x & 3)) : -1;
    const int tb = (int)((ko - kbase) >> 7) & 31;
    unsigned m = 0;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const bool g = row[e] != nullptr && ko >= 0 && ((tm[e] >> tb) & 1u);
      v[SL][e] = *(gvec)(g ? row[e] + ko : dummy);
      m |= (unsigned)g << e;
    }
    ok[SL] = m;
  }
  template <int SL>
  __device__ __forceinline__ void store(__bf16 *hi, __bf16 *lo) const {
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      int plane, r, c;
      place(threadIdx.x + NT * e, plane, r, c);
      const u32x4 x = ((ok[SL] >> e) & 1u) ? v[SL][e] : u32x4{0u, 0u, 0u, 0u};
      *(u32x4 *)((plane ? lo : hi) + lds_at(r, c)) = x;
    }
  }
};

// Staging of an FP32 operand stored k-contiguous, split into bf16 hi and lo
// planes on its way to LDS (split_bf16, the split every stored split operand
// gets, so the MFMA inputs are the same bits).  Per stage R rows x 32 k as
// k-quads: one 16-byte load of 4 values gives 8 bytes of hi and 8 of lo.  A
// thread's quads all take quad q = threadIdx.x & 7 of a step (k run q / 2,
// half q % 2); rows, zeros and the pipeline as PSOperand.
template <int R, int NT = kThreads>
struct PFOperand {
  static constexpr int NQ = R * (kXBK / 4);  // k-quads per stage
  static constexpr int PER = NQ / NT;
  static_assert(PER * NT == NQ, "whole quads per thread");
  static_assert(NT % 8 == 0, "k quad = threadIdx.x & 7");
  const float *row[PER];  // plane + row offset of quad e, nullptr: row absent
  const float *dummy;
  unsigned tm[PER];  // as PSOperand
  long kbase;
  f4 v[2][PER];
  unsigned ok[2];

  template <class RowF, class MaskF>
  __device__ __forceinline__ void init(const float *plane, const RowF &rowf, const MaskF &maskf,
                                       long kb) {
    dummy = plane;
    kbase = kb;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int r = (int)((threadIdx.x + NT * e) >> 3);
      const long o = rowf(r);
      row[e] = o >= 0 ? plane + o : nullptr;
      tm[e] = maskf(r);
    }
  }
  template <int SL, class KOfs>
  __device__ __forceinline__ void load(const KOfs &kofs, int kt, int ksteps) {
    const int q = (int)(threadIdx.x & 7);
    const long kr = kt < ksteps ? kofs(kt, q >> 1) : -1;
    const long ko = kr >= 0 ? kr + 4 * (q & 1) : -1;
    const int tb = (int)((ko - kbase) >> 7) & 31;
    unsigned m = 0;
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const bool g = row[e] != nullptr && ko >= 0 && ((tm[e] >> tb) & 1u);
      v[SL][e] = gld((const f4 *)(g ? row[e] + ko : dummy));
      m |= (unsigned)g << e;
    }
    ok[SL] = m;
  }
  template <int SL>
  __device__ __forceinline__ void store(__bf16 *hi, __bf16 *lo) const {
    typedef uint16_t u4v __attribute__((ext_vector_type(4)));
    const int q = (int)(threadIdx.x & 7);
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int r = (int)((threadIdx.x + NT * e) >> 3);
      const bool g = (ok[SL] >> e) & 1u;
      u4v h, l;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        __bf16 hh, ll;
        split_bf16(g ? v[SL][e][j] : 0.0f, hh, ll);
        h[j] = __builtin_bit_cast(uint16_t, hh);
        l[j] = __builtin_bit_cast(uint16_t, ll);
      }
      const int o = lds_at(r, q >> 1) + 4 * (q & 1);
      *(u4v *)(hi + o) = h;
      *(u4v *)(lo + o) = l;
    }
  }
};

// The MFMAs of one stage of 32 k for a wave's WM x WN tile.  AHEAD: every
// operand is read before the first MFMA (hides the reads' latency at one or two
// waves a SIMD), else a row block at a time (fewer registers).
template <int WM, int WN, bool AHEAD>
__device__ __forceinline__ void mma_stage(const __bf16 *ah, const __bf16 *al, const __bf16 *bh,
                                          const __bf16 *bl, int wm, int wn,
                                          f4 (&acc)[WM / 16][WN / 16]) {
  constexpr int TM = WM / 16, TN = WN / 16;
  const int lane = threadIdx.x & 63, kr = lane >> 4;  // kr: k run
  bf16x8 ahi[TM], alo[TM], bhi[TN], blo[TN];
  auto row = [&](int i) {
    const int o = lds_at(wm * WM + i * 16 + (lane & 15), kr);
    ahi[i] = *(const bf16x8 *)(ah + o);
    alo[i] = *(const bf16x8 *)(al + o);
  };
  if (AHEAD)
#pragma unroll
    for (int i = 0; i < TM; ++i) row(i);
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    const int o = lds_at(wn * WN + j * 16 + (lane & 15), kr);
    bhi[j] = *(const bf16x8 *)(bh + o);
    blo[j] = *(const bf16x8 *)(bl + o);
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    if (!AHEAD) row(i);
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      acc[i][j] = mfma_bf16(alo[i], bhi[j], acc[i][j]);
      acc[i][j] = mfma_bf16(ahi[i], blo[j], acc[i][j]);
      acc[i][j] = mfma_bf16(ahi[i], bhi[j], acc[i][j]);
    }
  }
}

// OA / OB: operand staging (PSOperand or PFOperand, rows set by
// init).  kofs(kt,
// c): element offset of k run c (8 k) of step kt, or -1 for zeros.  The NT
// threads form NT / 64 waves in a (NT / 64 / WGN) x WGN grid, each with a
// (BM / rows) x (BN / WGN) tile of 16x16 blocks; acc holds one wave's blocks.
// Pipeline: two LDS stages and two register slots; the global loads of step
// kt + 2 are issued before the MFMAs of step kt, so each load has two steps
// of MFMA work to arrive in.
template <int BM, int BN, int NT, int WGN, class OA, class OB, class KOfs>
__device__ __forceinline__ void gemm_tile_bf16x3(
    OA &A, OB &B, int ksteps, const KOfs &kofs, __bf16 *lds,
    f4 (&acc)[BM / (NT / 64 / WGN) / 16][BN / WGN / 16]) {
  constexpr int WGM = NT / 64 / WGN;
  constexpr int WM = BM / WGM, WN = BN / WGN, TM = WM / 16, TN = WN / 16;
  constexpr int SA = BM * kXBK, SB = BN * kXBK, STAGE = 2 * SA + 2 * SB;
  const int wave = threadIdx.x >> 6, wm = wave / WGN, wn = wave % WGN;
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f4{0, 0, 0, 0};

  if (ksteps <= 0) return;
  auto compute = [&](int cur) {
    const __bf16 *ah = lds + cur * STAGE, *al = ah + SA, *bh = al + SA, *bl = bh + SB;
    mma_stage<WM, WN, (BN < 128)>(ah, al, bh, bl, wm, wn, acc);
  };
  // Loads and stores run unconditionally (past the last step they move zeros),
  // so the loop body is straight-line code and the compiler's wait counts keep
  // the later steps' loads in flight while the next step is written to LDS.
  // With four waves a SIMD the registers hold one step's loads ahead, else two.
  auto store = [&](auto slot, int buf) {
    constexpr int SL = decltype(slot)::value;
    __bf16 *ah = lds + buf * STAGE, *al = ah + SA, *bh = al + SA, *bl = bh + SB;
    A.template store<SL>(ah, al);
    B.template store<SL>(bh, bl);
  };
  auto load = [&](auto slot, int kt) {
    constexpr int SL = decltype(slot)::value;
    A.template load<SL>(kofs, kt, ksteps);
    B.template load<SL>(kofs, kt, ksteps);
  };
  constexpr std::integral_constant<int, 0> s0{};
  constexpr std::integral_constant<int, 1> s1{};
  load(s0, 0);
  if constexpr (NT > kThreads) {
    store(s0, 0);
    __syncthreads();
    for (int kt = 0; kt < ksteps; ++kt) {
      load(s0, kt + 1);
      compute(kt & 1);
      store(s0, (kt & 1) ^ 1);
      __syncthreads();
    }
  } else {  // step kt in register slot kt & 1 and LDS stage kt & 1
    load(s1, 1);
    store(s0, 0);
    __syncthreads();
    auto step = [&](auto slot, auto next, int kt) {
      load(slot, kt + 2);  // the slot is free: step kt is in LDS
      compute(decltype(slot)::value);
      store(next, decltype(next)::value);
      __syncthreads();
    };
    int kt = 0;
    for (; kt + 1 < ksteps; kt += 2) {
      step(s0, s1, kt);
      step(s1, s0, kt + 1);
    }
    if (kt < ksteps) step(s0, s1, kt);
  }
}


// X = Phi D of one 128-point tile and CN = 64 TN columns, eight waves in 2 x 4,
// each 64 points x 16 TN columns, K the tile's c8 runs of 8 functions (kl, with
// their functions in the tile's list km), four runs a step.  A wave stages one
// run of Phi for 64 points (its index is uniform, so the rows' addresses are
// scalar): 8 loads of 256 contiguous bytes, split into hi and lo and written as
// 16 bytes of each, k-contiguous; functions outside the tile's list (not
// written by the basis stage) count as 0.  D^T is stored split and
// k-contiguous: a thread copies a run's 16 bytes of hi and of lo per 128
// columns.  Two LDS stages, the next step's loads in flight during the MFMAs.
constexpr int kDensThreads = 512;
template <int TN>
__device__ __forceinline__ void dens_x3(const float *__restrict__ phi, long Mc,
                                        const __bf16 *__restrict__ D, int NP, const uint16_t *kl,
                                        const uint8_t *km, int c8, const uint16_t *cl, int ncol,
                                        __bf16 *lds, f4 (&acc)[4][TN]) {
  constexpr int CN = 64 * TN, SA = kXBM * kXBK, SB = CN * kXBK, STAGE = 2 * SA + 2 * SB;
  typedef uint16_t u8v __attribute__((ext_vector_type(8)));
  constexpr int NB = (CN + 127) / 128;  // columns per thread
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int ac = wave >> 1, ar = 64 * (wave & 1) + lane;  // A: the wave's run of a step, the lane's point
  const int bc = tid & 3, br = tid >> 2;                  // B: the thread's run and column
  unsigned boff[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) boff[b] = (unsigned)cl[min(br + 128 * b, ncol - 1)] * (unsigned)NP;
  const long np2 = (long)NP * NP;
  const int ksteps = (c8 + 3) / 4;
  float va[8];
  u32x4 vh[NB], vl[NB];
  unsigned am = 0;
  bool bm = false;
  auto load = [&](int kt) {
    const int u = min(4 * kt + ac, c8 - 1), w = min(4 * kt + bc, c8 - 1);
    const long r = __builtin_amdgcn_readfirstlane((int)kl[u]);
    am = 4 * kt + ac < c8 ? (unsigned)__builtin_amdgcn_readfirstlane((int)km[u]) : 0u;
    const float *p = phi + r * kRun * Mc;
#pragma unroll
    for (int j = 0; j < 8; ++j) va[j] = gld(p + ((am >> j) & 1u ? j * Mc : 0) + ar);
    bm = 4 * kt + bc < c8;
    const unsigned ko = (unsigned)kl[w] * kRun;
#pragma unroll
    for (int b = 0; b < NB; ++b)
      if (128 * (b + 1) <= CN || br + 128 * b < CN) {
        vh[b] = *(gvec)(D + (boff[b] + ko));
        vl[b] = *(gvec)(D + np2 + (boff[b] + ko));
      }
  };
  auto store = [&](int buf) {
    __bf16 *ah = lds + buf * STAGE, *al = ah + SA, *bh = al + SA, *bl = bh + SB;
    u8v h, l;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      __bf16 hh, ll;
      split_bf16((am >> j) & 1u ? va[j] : 0.0f, hh, ll);
      h[j] = __builtin_bit_cast(uint16_t, hh);
      l[j] = __builtin_bit_cast(uint16_t, ll);
    }
    *(u8v *)(ah + lds_at(ar, ac)) = h;
    *(u8v *)(al + lds_at(ar, ac)) = l;
#pragma unroll
    for (int b = 0; b < NB; ++b)
      if (128 * (b + 1) <= CN || br + 128 * b < CN) {
        const bool g = bm && br + 128 * b < ncol;
        *(u32x4 *)(bh + lds_at(br + 128 * b, bc)) = g ? vh[b] : u32x4{0u, 0u, 0u, 0u};
        *(u32x4 *)(bl + lds_at(br + 128 * b, bc)) = g ? vl[b] : u32x4{0u, 0u, 0u, 0u};
      }
  };
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = f4{0, 0, 0, 0};
  load(0);
  store(0);
  __syncthreads();
  for (int kt = 0; kt < ksteps; ++kt) {
    load(kt + 1);  // past the end: the last run again, stored as zeros
    const __bf16 *ah = lds + (kt & 1) * STAGE, *al = ah + SA, *bh = al + SA, *bl = bh + SB;
    mma_stage<64, 16 * TN, (TN > 2)>(ah, al, bh, bl, wave >> 2, wave & 3, acc);
    store((kt & 1) ^ 1);
    __syncthreads();
  }
}

// Sums of X = Phi D over a share's ncol columns: part[0] = sum_n Phi X, part[c] =
// 2 sum_n d_c Phi X at the tile's 128 points.  X goes through LDS ([column]
// [point], rows padded by 16 bytes), so that the values are read as they lie in
// memory: half a wave takes one column's 128 points, 512 contiguous bytes per
// plane (an MFMA block's layout has 64 of 16 columns), the 16 half waves every
// 16th column; their sums meet in LDS.
constexpr int kXRow = kXBM + 4;
template <int TN, bool GRAD>
__device__ __forceinline__ void dens_sums_x3(const f4 (&acc)[4][TN], const float *__restrict__ phi,
                                             long Mc, long cs, const uint16_t *cl, int ncol, float *xs,
                                             double *__restrict__ part) {
  constexpr int NC = GRAD ? 4 : 1;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
      *(f4 *)(xs + ((wave & 3) * 16 * TN + 16 * j + (lane & 15)) * kXRow + 64 * (wave >> 2) + 16 * i +
              4 * (lane >> 4)) = acc[i][j];
  __syncthreads();
  const int q = 4 * (lane & 31);  // the lane's four points
  double s[NC][4];
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) s[c][r] = 0.0;
#pragma unroll 2
  for (int n = 2 * wave + (lane >> 5); n < ncol; n += 16) {
    const float *p = phi + (long)cl[n] * Mc + q;
    f4 v[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) v[c] = gld((const f4 *)(p + c * cs));
    const f4 x = *(const f4 *)(xs + n * kXRow + q);
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int r = 0; r < 4; ++r) s[c][r] += (double)v[c][r] * (double)x[r];
  }
#pragma unroll
  for (int c = 0; c < NC; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r) s[c][r] += __shfl_xor(s[c][r], 32);
  __syncthreads();  // every wave has read its columns
  double *red = (double *)xs;  // [8 waves][NC][128]
  if (lane < 32)
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        typedef double d2 __attribute__((ext_vector_type(2)));
        *(d2 *)(red + (wave * NC + c) * kXBM + q + r) = d2{s[c][r], s[c][r + 1]};
      }
  __syncthreads();
  for (int e = tid; e < NC * kXBM; e += kDensThreads) {
    double v = 0.0;
#pragma unroll
    for (int w = 0; w < 8; ++w) v += red[w * NC * kXBM + e];
    gst(part + (long)(e / kXBM) * Mc + e % kXBM, e < kXBM ? v : 2.0 * v);
  }
}

// item = (128-point tile, up to IC of its functions as columns, shared out evenly
// over the tile's items).  IC = 128 (tiles of few functions): two LDS stages of
// 64 KB and 128 registers, so two workgroups share a CU and one's K loop runs
// during the other's sums.  IC = 256 (setup_screen: many functions): the K loop
// is most of the time, and twice the columns halve its LDS traffic per MFMA and
// the staging of Phi.  Bound by the sums' HBM reads (16 bytes per point and
// function) and, for many functions, by LDS.  Stage of an (H2O)32 build, one
// lane, 228 functions a tile: 3.48 ms with one workgroup of 192 columns per CU
// and the values read in the MFMA blocks' layout, 3.38 with two of 128, 2.8
// with the values read by column; (H2O)128 and solute, 916 a tile: 171 ms of
// two-lane stage time at IC = 128, 150 at 256.  At IC = 128 the 128 registers of
// four waves a SIMD are 9 too few (32 bytes of scratch a lane).
template <bool GRAD, int IC>
__global__ __launch_bounds__(kDensThreads) __attribute__((amdgpu_waves_per_eu(IC == 128 ? 4 : 2))) void k_density_bf16x3(const StageList S) {
  // the sums' X and reduction reuse the staging LDS
  constexpr int BM = kXBM, NT = kDensThreads;
  constexpr int kBytes = sizeof(float) * IC * kXRow;
  static_assert(kBytes >= (int)sizeof(__bf16) * 2 * XStage<BM, IC>::n && kBytes >= 8 * 4 * BM * 8, "LDS");
  __shared__ __attribute__((aligned(16))) char lds[kBytes];
  __shared__ uint16_t kl[kMaxRuns];
  __shared__ uint8_t km[kMaxRuns];  // per run of kl: its functions in the tile's list
  __shared__ uint16_t cl[IC];
  __shared__ long slot;
  static_assert(kXBK == 4 * kRun, "four runs per K step");
  for (long L = walk_next(S, -1, &slot); L < S.total;) {
    const uint64_t t0 = S.tlog ? wall_clock64() : 0;
    const long it = walk_item(S, L);
    const int u = find_unit(S.base, S.nu, it);
    const UnitD &U = S.units[u];
    const uint32_t e = U.ditems[it - S.base[u]];
    const int tile = (int)(e >> 8), item = (int)(e & 255);
    const long m0 = (long)tile * BM, Mc = U.Mc;
    const int off = U.tl_off[tile], c8 = U.tl_off[tile + 1] - off;
    const int nf = U.tf_off[tile + 1] - U.tf_off[tile], cc = share_cols(nf, IC);
    const int foff = U.tf_off[tile] + item * cc, ncol = min(cc, nf - item * cc);
    __syncthreads();  // the previous item's readers of kl, cl and the LDS are done
    for (int i = threadIdx.x; i < ncol; i += NT) cl[i] = gld(U.tfl + foff + i);
    for (int i = threadIdx.x; i < c8; i += NT) km[i] = gld(U.tlm + off + i);
    lds_list(U.tl + off, c8, kl);
    int ahead = 0;
    const float *phi = (const float *)U.phi + m0;
    double *part = U.part + (long)item * 4 * Mc + m0;
    auto go = [&](auto tn) {
      constexpr int TN = decltype(tn)::value;
      f4 acc[4][TN];
      dens_x3<TN>(phi, Mc, (const __bf16 *)U.D, U.NP, kl, km, c8, cl, ncol, (__bf16 *)lds, acc);
      ahead = walk_ahead(S);
      dens_sums_x3<TN, GRAD>(acc, phi, Mc, (long)U.NP * Mc, cl, ncol, (float *)lds, part);
    };
    if (ncol <= 64) go(std::integral_constant<int, 1>{});
    else if (IC == 128 || ncol <= 128) go(std::integral_constant<int, 2>{});
    else if (ncol <= 192) go(std::integral_constant<int, IC == 128 ? 2 : 3>{});
    else go(std::integral_constant<int, IC / 64>{});
    item_log(S, it, t0);
    L = walk_take(S, L, ahead, &slot);
  }
}

template <int IC>
static void density_x3(hipStream_t s, bool grad, const StageList &L) {
  dim3 g(contraction_grid(L, IC == 128 ? 2 : 1));
  if (grad)
    hipLaunchKernelGGL((k_density_bf16x3<true, IC>), g, dim3(kDensThreads), 0, s, L);
  else
    hipLaunchKernelGGL((k_density_bf16x3<false, IC>), g, dim3(kDensThreads), 0, s, L);
}

void launch_density_bf16x3(hipStream_t s, bool grad, int icols, const StageList &L) {
  if (!L.total) return;
  if (icols == 128) density_x3<128>(s, grad, L);
  else density_x3<256>(s, grad, L);
}

// item = (point split, function tile pair), as k_potential (chunks of 128: four
// waves a SIMD, 20 registers spilled, 84 bytes a lane)
constexpr int pot_threads(int BT) { return BT == 128 ? 512 : 256; }
template <int BT>
__global__ __launch_bounds__(pot_threads(BT))
__attribute__((amdgpu_waves_per_eu(BT == 128 ? 4 : 2))) void k_potential_bf16x3(const StageList S) {
  constexpr int NT = pot_threads(BT), WGN = NT / 128, WM = BT / 2, WN = BT / WGN;
  __shared__ __attribute__((aligned(16))) __bf16 lds[2 * XStage<BT, BT>::n];
  __shared__ uint16_t ul[2 * BT];  // the functions of the row chunk, then of the column chunk
  __shared__ int rb[32], cb[32], nt;
  __shared__ uint8_t tl[32];
  __shared__ long slot;
  static_assert(kXBK == kGroup, "one K step per 32-point group");
  for (long L = walk_next(S, -1, &slot); L < S.total;) {
    const uint64_t t0 = S.tlog ? wall_clock64() : 0;
    const long it = walk_item(S, L);
    const int u = find_unit(S.base, S.nu, it);
    const UnitD &U = S.units[u];
    const uint32_t e = U.pitems[it - S.base[u]];
    const int sl = (int)(e >> 20), ci = (int)((e >> 10) & 1023), cj = (int)(e & 1023);
    const long Mc = U.Mc;
    const int so = U.su_off[sl], nu = U.su_off[sl + 1] - so;
    const long kb = (long)sl * (Mc / U.nsplit);
    const int nri = min(BT, nu - ci * BT), nrj = min(BT, nu - cj * BT);
    __syncthreads();  // the previous item's readers of ul / gl are done
    for (int i = threadIdx.x; i < 2 * BT; i += NT)
      if (i < BT ? i < nri : i - BT < nrj) ul[i] = gld(U.su + so + (i < BT ? ci * BT + i : cj * BT + i - BT));
    const uint32_t *tmi = U.sumask + so + ci * BT, *tmj = U.sumask + so + cj * BT;
    const int ng = 4 * potential_tiles<BT, NT>(tmi, nri, tmj, nrj, rb, cb, tl, &nt);
    const uint16_t *ri = ul, *rj = ul + BT;
    const __bf16 *wh = (const __bf16 *)U.W;
    const long pn = (long)U.NP * Mc;
    // A(m, k) = W[f_i(m)][kb + p(k)] (stored split), B(k, n) =
    // Phi[f_j(n)][kb + p(k)] (FP32 values, split while staged)
    PSOperand<BT, NT> opa;
    PFOperand<BT, NT> opb;
    // rows and columns skip the tiles whose list lacks their function (W and
    // Phi are 0 there)
    opa.init({wh, wh + pn}, [&](int m) -> long { return m < nri ? (long)ri[m] * Mc : -1; },
             [&](int m) -> unsigned { return m < nri ? gld(tmi + m) : 0u; }, kb);
    opb.init((const float *)U.phi, [&](int n) -> long { return n < nrj ? (long)rj[n] * Mc : -1; },
             [&](int n) -> unsigned { return n < nrj ? gld(tmj + n) : 0u; }, kb);
    auto kofs = [&](int kt, int c) -> long { return kb + 32 * (4 * (int)tl[kt >> 2] + (kt & 3)) + 8 * c; };
    f4 acc[WM / 16][WN / 16];
    gemm_tile_bf16x3<BT, BT, NT, WGN>(opa, opb, ng, kofs, lds, acc);
    const int ahead = walk_ahead(S);
    {
      const int ld = split_ld(nu), wave = threadIdx.x >> 6;
      const int r0 = (wave / WGN) * WM, c0 = (wave % WGN) * WN;
      double *H = U.Hc + U.ho[sl] + (long)(ci * BT + r0) * ld + cj * BT + c0;
#pragma unroll
      for (int i = 0; i < WM / 16; ++i)
#pragma unroll
        for (int j = 0; j < WN / 16; ++j)
          if (r0 + 16 * i < nri && c0 + 16 * j < nrj) put_block<float>(acc[i][j], H + (long)16 * i * ld + 16 * j, ld);
    }
    item_log(S, it, t0);
    L = walk_take(S, L, ahead, &slot);
  }
}

void launch_potential_bf16x3(hipStream_t s, int tf, const StageList &L) {
  if (!L.total) return;
  dim3 g(contraction_grid(L, 2));
  switch (tf) {
    case 64: hipLaunchKernelGGL((k_potential_bf16x3<64>), g, dim3(pot_threads(64)), 0, s, L); break;
    case 96: hipLaunchKernelGGL((k_potential_bf16x3<96>), g, dim3(pot_threads(96)), 0, s, L); break;
    default: hipLaunchKernelGGL((k_potential_bf16x3<128>), g, dim3(pot_threads(128)), 0, s, L); break;
  }
}

}  // namespace pgxc
