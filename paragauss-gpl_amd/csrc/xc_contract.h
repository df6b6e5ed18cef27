// FP64 and FP32 contractions of the XC build on MFMA, for gfx950 (kernel
// templates; xc_contract_f64.hip and xc_contract_f32.hip instantiate them).
//
//   k_density    X = Phi D per 128-point tile, fused rho = sum Phi X,
//                grad rho = 2 sum dPhi X
//                (ParaGauss modules/density_calc_module.f90:1478-1577)
//   k_potential  H = W^T Phi per point split (modules/xc_hamiltonian.f90:1528-1531)
//
// A 16x16x4 FP64 MFMA holds its SIMD's matrix core for 64 cycles (FP32: 32), so
// the time is the number of MFMAs: K and the output columns are the tile's own
// functions, one by one, not runs of 8 or whole column chunks, and 16-column
// blocks past the last function are skipped.  The operands' loads and LDS
// traffic are a small share of it and only have to stay ahead.
#pragma once
#include <algorithm>
#include <type_traits>

#include "pgxc_internal.h"
#include "xc_device.h"

namespace pgxc {

template <typename T>
struct V2 {
  typedef T type __attribute__((ext_vector_type(2)));
};

// Point of a 16-point block that MFMA row i stands for: chosen so that a
// lane's four results are four consecutive points 4 (lane / 16) + r (the FP64
// result has rows lane / 16 + 4 r, the FP32 result those already).
template <typename T>
__device__ __forceinline__ int row_point(int i) {
  return MF<T>::kQuadRows ? i : 4 * (i & 3) + (i >> 2);
}

constexpr int kDBM = 128;  // points of a density tile
constexpr int kLPad = 16;  // LDS row padding: the four k rows an MFMA operand
                           // read touches lie on different banks

// X(m, n) = sum_k Phi[f(k)][m0 + m] D[f(k)][c(n)] for one tile and one chunk of
// NB 16-column blocks, f and c entries of the tile's function list: four waves,
// each 32 points x all columns.  Both operands are staged [k][row] as they lie
// in memory: a wave takes whole k rows (its index is uniform, so their addresses
// are scalar), a lane two points of Phi and one column of D (symmetric, so row
// f(k) is read along the columns).  Rows past the list repeat its last
// function, and their D is 0; columns past it repeat its last one and are not
// used.  The list entries of a step are read a step ahead of its loads.
//
// ST = 2: two LDS stages, one barrier per step; ST = 1: one stage.
template <typename T, int BN, int VAR>
struct DensTile {
  static_assert(BN <= 64, "a column per lane");
  static constexpr int BK = Var<VAR>::BK, ST = Var<VAR>::ST;
  static constexpr int SA = kDBM + kLPad, SB = BN + kLPad, R = BK / 4;
  static constexpr int kLds = ST * BK * (SA + SB);
  typedef typename V2<T>::type v2;
  typedef typename MF<T>::acc acc_t;

  template <int NB>
  __device__ static __forceinline__ void run(const T *__restrict__ phi, long Mc,
                                             const T *__restrict__ D, long NP,
                                             const uint16_t *__restrict__ fl, int K,
                                             const uint16_t *__restrict__ cf, int ncol, T *lds,
                                             acc_t (&acc)[2][NB]) {
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int ksteps = (K + BK - 1) / BK;
    const int c0 = gld(cf + min(lane, ncol - 1));
    v2 ra[R];
    T rb[R];
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < NB; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
    auto list = [&](int kt) { return (int)gld(fl + min(kt * BK + (lane & (BK - 1)), K - 1)); };
    auto load = [&](int fk) {
#pragma unroll
      for (int e = 0; e < R; ++e) {
        const long f = __builtin_amdgcn_readlane(fk, wave + 4 * e);
        ra[e] = gld((const v2 *)(phi + f * Mc) + lane);
        rb[e] = gld(D + f * NP + c0);
      }
    };
    auto store = [&](int buf, int kt) {
      T *as = lds + buf * BK * (SA + SB), *bs = as + BK * SA;
#pragma unroll
      for (int e = 0; e < R; ++e) {
        const int r = wave + 4 * e;
        const bool live = kt * BK + r < K;
        *(v2 *)(as + r * SA + 2 * lane) = ra[e];
        bs[r * SB + lane] = live ? rb[e] : T(0);
      }
    };
    const int ar = 32 * wave + row_point<T>(lane & 15), br = lane & 15, kg = lane >> 4;
    auto compute = [&](int buf) {
      const T *as = lds + buf * BK * (SA + SB) + kg * SA + ar;
      const T *bs = lds + buf * BK * (SA + SB) + BK * SA + kg * SB + br;
#pragma unroll
      for (int k4 = 0; k4 < BK / 4; ++k4) {
        T a[2], b[NB];
        a[0] = as[4 * k4 * SA];
        a[1] = as[4 * k4 * SA + 16];
#pragma unroll
        for (int j = 0; j < NB; ++j) b[j] = bs[4 * k4 * SB + 16 * j];
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int i = 0; i < 2; ++i) acc[i][j] = MF<T>::mma(a[i], b[j], acc[i][j]);
      }
    };
    int fn = list(0);
    load(fn);
    fn = list(1);
    if constexpr (ST == 2) {
      store(0, 0);
      __syncthreads();
      for (int kt = 0; kt < ksteps; ++kt) {
        load(fn);  // step kt + 1 (past the end: the last function again, D 0)
        fn = list(kt + 2);
        compute(kt & 1);
        store((kt & 1) ^ 1, kt + 1);
        __syncthreads();
      }
    } else {
      for (int kt = 0; kt < ksteps; ++kt) {
        store(0, kt);
        __syncthreads();
        load(fn);
        fn = list(kt + 2);
        compute(0);
        __syncthreads();
      }
    }
  }
};

// Sums of a wave's 32 points over a chunk's columns: part[0] = sum_n Phi X,
// part[c] = 2 sum_n d_c Phi X.  A lane holds four consecutive points of one
// column per block: 16-byte loads; the 16 lanes of a block's columns are summed
// by group_reduce, and the wave holds every column, so nothing crosses waves.
// Absent columns read the chunk's first function and add nothing.
template <typename T, int NB, bool GRAD>
__device__ __forceinline__ void density_sums(typename MF<T>::acc (&acc)[2][NB],
                                             const T *__restrict__ phi, long Mc, long cs,
                                             const uint16_t *__restrict__ cf, int ncol,
                                             double *__restrict__ part) {
  constexpr int NC = GRAD ? 4 : 1, NV = 4 * (int)sizeof(T) / 16, E = 16 / (int)sizeof(T);
  typedef T vec __attribute__((ext_vector_type(16 / sizeof(T))));
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int p0 = 32 * wave + 4 * (lane >> 4);
  const T *ph[NB];
#pragma unroll
  for (int j = 0; j < NB; ++j) {
    const int n = 16 * j + (lane & 15);
    ph[j] = phi + (long)gld(cf + (n < ncol ? n : 0)) * Mc + p0;
    if (n >= ncol)
#pragma unroll
      for (int i = 0; i < 2; ++i) acc[i][j] = typename MF<T>::acc{0, 0, 0, 0};
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll 1  // one plane's loads in flight at a time: more would spill
    for (int c = 0; c < NC; ++c) {
      vec v[NB][NV];
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int q = 0; q < NV; ++q) v[j][q] = gld((const vec *)(ph[j] + c * cs + 16 * i) + q);
      double t[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
      for (int j = 0; j < NB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) t[r] += (double)v[j][r / E][r % E] * (double)acc[i][j][r];
      int idx;
      const double tot = group_reduce(t, lane, idx);
      if ((lane & 3) == 0) gst(part + (long)c * Mc + p0 + 16 * i + idx, c ? 2.0 * tot : tot);
    }
}

// item = (128-point tile, share of its functions as columns).  Bound by
// the matrix cores and, about equally, the sums' reads of Phi and d Phi (32
// bytes per point and function, 14 GB at (H2O)32 in FP64).  The kernel before
// walked whole runs of 8 functions and 96-column chunks (1.4 times the MFMAs)
// and looked every operand vector up in the run list as it loaded it: FP64
// density stage of an (H2O)32 build, one lane, 10.8 ms; now 6.3 (variant 1 6.6,
// 2 8.5).
template <typename T, int BN, int VAR, bool GRAD>
__global__ __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(VAR == 2 ? 1 : 2))) void k_density(const StageList S) {
  typedef DensTile<T, BN, VAR> G;
  __shared__ __attribute__((aligned(16))) T lds[G::kLds];
  __shared__ long slot;
  for (long L = walk_next(S, -1, &slot); L < S.total;) {
    const uint64_t t0 = S.tlog ? wall_clock64() : 0;
    const long it = walk_item(S, L);
    const int u = find_unit(S.base, S.nu, it);
    const UnitD &U = S.units[u];
    const uint32_t e = U.ditems[it - S.base[u]];
    const int tile = (int)(e >> 8), item = (int)(e & 255);
    const long m0 = (long)tile * kDBM, Mc = U.Mc, NP = U.NP;
    const int off = U.tf_off[tile], nf = U.tf_off[tile + 1] - off;
    const uint16_t *fl = U.tfl + off;
    const int cc = share_cols(nf, BN), per = U.icols / BN, ch1 = min((item + 1) * per, (nf + BN - 1) / BN);
    const T *phi = (const T *)U.phi + m0, *D = (const T *)U.D;
    int ahead = 0;
    for (int ch = item * per; ch < ch1; ++ch) {
      const bool last = ch + 1 == ch1;
      const uint16_t *cf = fl + ch * cc;
      const int ncol = min(cc, nf - ch * cc);
      auto go = [&](auto nb) {
        constexpr int NB = decltype(nb)::value;
        typename MF<T>::acc acc[2][NB];
        __syncthreads();  // the previous chunk's readers of the LDS stages are done
        G::template run<NB>(phi, Mc, D, NP, fl, nf, cf, ncol, lds, acc);
        if (last) ahead = walk_ahead(S);
        density_sums<T, NB, GRAD>(acc, phi, Mc, NP * Mc, cf, ncol, U.part + (long)ch * 4 * Mc + m0);
      };
      const int nb = (ncol + 15) / 16;
      if (nb <= 1) go(std::integral_constant<int, 1>{});
      else if (nb == 2) go(std::integral_constant<int, 2>{});
      else if (nb == 3) go(std::integral_constant<int, 3>{});
      else go(std::integral_constant<int, 4>{});
    }
    item_log(S, it, t0);
    L = walk_take(S, L, ahead, &slot);
  }
}

// The nuclear gradient's products over the density's items, P for D, stored
// instead of summed: plane 0 X = Phi P, plane 1 Z = W P, at the tile's functions.
// Bound by the matrix cores: 0.98 ms per (H2O)16 chunk of 245 760 points (X and
// the three products of the gradient planes on whole runs: 2.8 ms).
template <int BN, int VAR>
__global__ __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(VAR == 2 ? 1 : 2))) void k_xz(const StageList S, const double *__restrict__ P,
                                                                  double *__restrict__ XZ, int nplanes,
                                                                  int nspin, int spin) {
  typedef DensTile<double, BN, VAR> G;
  __shared__ __attribute__((aligned(16))) double lds[G::kLds];
  for (long L = blockIdx.x; L < S.total; L += gridDim.x) {
    const long it = (long)xcd_remap((int)L, (int)S.total);
    const int u = find_unit(S.base, S.nu, it);
    if (u % nspin != spin) continue;  // uniform over the workgroup
    const UnitD &U = S.units[u];
    const uint32_t e = U.ditems[it - S.base[u]];
    const int tile = (int)(e >> 8), item = (int)(e & 255);
    const long m0 = (long)tile * kDBM, Mc = U.Mc, NP = U.NP;
    const int off = U.tf_off[tile], nf = U.tf_off[tile + 1] - off;
    const uint16_t *fl = U.tfl + off;
    const int cc = share_cols(nf, BN), per = U.icols / BN, ch1 = min((item + 1) * per, (nf + BN - 1) / BN);
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    for (int ch = item * per; ch < ch1; ++ch) {
      const uint16_t *cf = fl + ch * cc;
      const int ncol = min(cc, nf - ch * cc);
      for (int pl = 0; pl < nplanes; ++pl) {
        const double *A = (const double *)(pl ? U.W : U.phi) + m0;
        double *out = XZ + pl * NP * Mc + m0 + 32 * wave + 4 * (lane >> 4);
        auto go = [&](auto nb) {
          constexpr int NB = decltype(nb)::value;
          d4 acc[2][NB];
          __syncthreads();  // the previous product's readers of the LDS stages are done
          G::template run<NB>(A, Mc, P, NP, fl, nf, cf, ncol, lds, acc);
#pragma unroll
          for (int j = 0; j < NB; ++j) {
            const int n = 16 * j + (lane & 15);
            if (n >= ncol) continue;
            double *o = out + (long)gld(cf + n) * Mc;
#pragma unroll
            for (int i = 0; i < 2; ++i) {  // four consecutive points
              gst((V2<double>::type *)(o + 16 * i), V2<double>::type{acc[i][j][0], acc[i][j][1]});
              gst((V2<double>::type *)(o + 16 * i) + 1, V2<double>::type{acc[i][j][2], acc[i][j][3]});
            }
          }
        };
        const int nb = (ncol + 15) / 16;
        if (nb <= 2) go(std::integral_constant<int, 2>{});
        else if (nb == 3) go(std::integral_constant<int, 3>{});
        else go(std::integral_constant<int, 4>{});
      }
    }
  }
}

inline void launch_xz_impl(hipStream_t s, int var, const StageList &L, const double *P, double *XZ, int np,
                           int ns, int sp) {
  if (!L.total) return;
  dim3 g((unsigned)std::min<long>(L.total, 512));
  switch (var) {
    case 1: hipLaunchKernelGGL((k_xz<kPartCols, 1>), g, dim3(kThreads), 0, s, L, P, XZ, np, ns, sp); break;
    case 2: hipLaunchKernelGGL((k_xz<kPartCols, 2>), g, dim3(kThreads), 0, s, L, P, XZ, np, ns, sp); break;
    default: hipLaunchKernelGGL((k_xz<kPartCols, 0>), g, dim3(kThreads), 0, s, L, P, XZ, np, ns, sp); break;
  }
}

template <typename T, int VAR>
static void density_var(hipStream_t s, bool grad, const StageList &L) {
  dim3 g(contraction_grid(L, 2));
  if (grad)
    hipLaunchKernelGGL((k_density<T, kPartCols, VAR, true>), g, dim3(kThreads), 0, s, L);
  else
    hipLaunchKernelGGL((k_density<T, kPartCols, VAR, false>), g, dim3(kThreads), 0, s, L);
}

template <typename T>
void launch_density(hipStream_t s, bool grad, int var, const StageList &L) {
  if (!L.total) return;
  switch (var) {
    case 1: density_var<T, 1>(s, grad, L); break;
    case 2: density_var<T, 2>(s, grad, L); break;
    default: density_var<T, 0>(s, grad, L); break;
  }
}

// H(m, n) += sum_p W[f(m)][p] Phi[f(n)][p] over the tiles of one split where
// both chunks have a function: 256 threads, waves 2 x 2, wave (wm, wn) holding
// the 16 x 16 blocks (2 i + wm, 2 j + wn), so that the rows and columns past the
// last function, and the blocks without a function on a tile, are shared
// evenly.  On a tile only the blocks that have one on both sides are multiplied
// (a uniform branch over the MFMAs of 16 points).  Both operands are kept
// [row][k] with rows padded by 16 bytes; a lane reads 16 bytes, E consecutive k,
// for E MFMAs (MFMA e of a chunk takes k = 4 E c + E g + e in lane group g).
// Functions not in a tile's list are staged as zeros (their values are not
// written).
template <typename T, int BT, int VAR>
struct PotTile {
  static constexpr int BK = Var<VAR>::BK, ST = Var<VAR>::ST, E = 16 / (int)sizeof(T);
  static constexpr int BKP = BK + E, SO = BT * BKP, kLds = 2 * ST * SO, TT = BT / 32;
  // vectors a row is loaded in: 16 bytes where they share out evenly
  static constexpr int VE = BT * (BK / E) % kThreads == 0 ? E : E / 2;
  static constexpr int NV = BK / VE, PER = BT * NV / kThreads, RS = kThreads / NV;
  static constexpr int SPT = kScreenTile / BK;  // K steps per tile
  static_assert(PER * kThreads == BT * NV && PER * RS == BT, "whole vectors per thread");
  typedef T vec __attribute__((ext_vector_type(VE)));
  typedef T rd __attribute__((ext_vector_type(E)));
  typedef typename MF<T>::acc acc_t;

  __device__ static __forceinline__ void run(const T *__restrict__ W, const T *__restrict__ phi,
                                             long Mc, const uint16_t *__restrict__ fr,
                                             const uint32_t *__restrict__ mr, int nr,
                                             const uint16_t *__restrict__ fc,
                                             const uint32_t *__restrict__ mc, int nc,
                                             const int *rb, const int *cb, const uint8_t *tl,
                                             int ntl, T *lds, acc_t (&acc)[TT][TT]) {
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wave >> 1, wn = wave & 1, kv = tid % NV, r0 = tid / NV;
    const T *pa[PER], *pb[PER];
    unsigned ma[PER], mb[PER];
#pragma unroll
    for (int e = 0; e < PER; ++e) {
      const int r = r0 + RS * e;
      pa[e] = W + (long)gld(fr + min(r, nr - 1)) * Mc + VE * kv;
      pb[e] = phi + (long)gld(fc + min(r, nc - 1)) * Mc + VE * kv;
      ma[e] = r < nr ? gld(mr + r) : 0u;
      mb[e] = r < nc ? gld(mc + r) : 0u;
    }
#pragma unroll
    for (int i = 0; i < TT; ++i)
#pragma unroll
      for (int j = 0; j < TT; ++j) acc[i][j] = acc_t{0, 0, 0, 0};
    vec ra[PER], rb_[PER];
    unsigned ok = 0;  // bits 2 e, 2 e + 1: vector e of W, of Phi is live
    const int ksteps = ntl * SPT;
    if (!ksteps) return;
    auto load = [&](int kt) {
      const int t = tl[min(kt / SPT, ntl - 1)];
      const long k = kScreenTile * t + (kt % SPT) * BK;
      ok = 0;
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        const bool ga = (ma[e] >> t) & 1u, gb = (mb[e] >> t) & 1u;
        ra[e] = gld((const vec *)(ga ? pa[e] + k : W));
        rb_[e] = gld((const vec *)(gb ? pb[e] + k : W));
        ok |= (unsigned)ga << (2 * e) | (unsigned)gb << (2 * e + 1);
      }
    };
    auto store = [&](int buf) {
      T *as = lds + 2 * buf * SO, *bs = as + SO;
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        const int o = (r0 + RS * e) * BKP + VE * kv;
        *(vec *)(as + o) = (ok >> (2 * e)) & 1u ? ra[e] : vec{};
        *(vec *)(bs + o) = (ok >> (2 * e + 1)) & 1u ? rb_[e] : vec{};
      }
    };
    auto compute = [&](int buf, int kt) {
      const int t = __builtin_amdgcn_readfirstlane((int)tl[kt / SPT]);
      const int la = __builtin_amdgcn_readfirstlane(rb[t]) >> wm, lb = __builtin_amdgcn_readfirstlane(cb[t]) >> wn;
      const T *as = lds + 2 * buf * SO + (16 * wm + (lane & 15)) * BKP + E * (lane >> 4);
      const T *bs = lds + 2 * buf * SO + SO + (16 * wn + (lane & 15)) * BKP + E * (lane >> 4);
      constexpr int CH = 1;  // reads per branch
#pragma unroll
      for (int c0 = 0; c0 < BK / (4 * E); c0 += CH) {
        rd a[TT][CH], b[TT][CH];
#pragma unroll
        for (int i = 0; i < TT; ++i)
#pragma unroll
          for (int c = 0; c < CH; ++c) {
            a[i][c] = *(const rd *)(as + 32 * i * BKP + 4 * E * (c0 + c));
            b[i][c] = *(const rd *)(bs + 32 * i * BKP + 4 * E * (c0 + c));
          }
#pragma unroll
        for (int i = 0; i < TT; ++i)
#pragma unroll
          for (int j = 0; j < TT; ++j)
            if ((la >> (2 * i)) & (lb >> (2 * j)) & 1) {
#pragma unroll
              for (int c = 0; c < CH; ++c)
#pragma unroll
                for (int e = 0; e < E; ++e) acc[i][j] = MF<T>::mma(a[i][c][e], b[j][c][e], acc[i][j]);
            }
      }
    };
    load(0);
    if constexpr (ST == 2) {
      store(0);
      __syncthreads();
      for (int kt = 0; kt < ksteps; ++kt) {
        load(kt + 1);  // past the end: the last tile again, not used
        compute(kt & 1, kt);
        store((kt & 1) ^ 1);
        __syncthreads();
      }
    } else {
      for (int kt = 0; kt < ksteps; ++kt) {
        store(0);
        __syncthreads();
        load(kt + 1);
        compute(0, kt);
        __syncthreads();
      }
    }
  }
};

// item = (point split, pair of chunks of its functions); writes its blocks of
// the split's partial (zeros where no tile has both).  Bound by the matrix
// cores: the blocks multiplied are 1.25 times sum n^2 at (H2O)32 (whole chunks
// on the groups where both had a function: 1.83).  FP64 stage of an (H2O)32
// build, one lane: 10.1 -> 6.1 ms; 23-atom molecule (233 000 points) 852 -> 150
// us, its 57 splits of 4096 points now 456 of 512.  Variants 0 and 1 keep
// their LDS stages under 80 KB: two workgroups share a CU and hide each other's
// waits.  With FP64 chunks of 128, 16 result blocks and a step's operands pass the
// 256 registers: variant 0 spills 13 (56 bytes of scratch a lane), variant 1 103.
template <typename T, int BT, int VAR>
__global__ __launch_bounds__(kThreads)
__attribute__((amdgpu_waves_per_eu(VAR == 2 ? 1 : 2))) void k_potential(const StageList S) {
  typedef PotTile<T, BT, VAR> G;
  __shared__ __attribute__((aligned(16))) T lds[G::kLds];
  __shared__ int rb[32], cb[32], nt;
  __shared__ uint8_t tl[32];
  __shared__ long slot;
  for (long L = walk_next(S, -1, &slot); L < S.total;) {
    const uint64_t t0 = S.tlog ? wall_clock64() : 0;
    const long it = walk_item(S, L);
    const int u = find_unit(S.base, S.nu, it);
    const UnitD &U = S.units[u];
    const uint32_t e = U.pitems[it - S.base[u]];
    const int sl = (int)(e >> 20), ci = (int)((e >> 10) & 1023), cj = (int)(e & 1023);
    const long Mc = U.Mc, kb = (long)sl * (Mc / U.nsplit);
    const int so = U.su_off[sl], nu = U.su_off[sl + 1] - so;
    const int nr = min(BT, nu - ci * BT), nc = min(BT, nu - cj * BT);
    const uint32_t *mr = U.sumask + so + ci * BT, *mc = U.sumask + so + cj * BT;
    const int n = potential_tiles<BT>(mr, nr, mc, nc, rb, cb, tl, &nt);
    typename MF<T>::acc acc[G::TT][G::TT];
    G::run((const T *)U.W + kb, (const T *)U.phi + kb, Mc, U.su + so + ci * BT, mr, nr,
           U.su + so + cj * BT, mc, nc, rb, cb, tl, n, lds, acc);
    const int ahead = walk_ahead(S);
    const int ld = split_ld(nu), wave = threadIdx.x >> 6, wm = wave >> 1, wn = wave & 1;
    double *H = U.Hc + U.ho[sl] + (long)ci * BT * ld + cj * BT;
#pragma unroll
    for (int i = 0; i < G::TT; ++i)
#pragma unroll
      for (int j = 0; j < G::TT; ++j) {
        const int r = 16 * (2 * i + wm), c = 16 * (2 * j + wn);
        if (r < nr && c < nc) put_block<T>(acc[i][j], H + (long)r * ld + c, ld);
      }
    item_log(S, it, t0);
    L = walk_take(S, L, ahead, &slot);
  }
}

template <typename T, int VAR>
static void potential_var(hipStream_t s, int tf, const StageList &L) {
  dim3 g(contraction_grid(L, 2));
  switch (tf) {
    case 64: hipLaunchKernelGGL((k_potential<T, 64, VAR>), g, dim3(kThreads), 0, s, L); break;
    case 96: hipLaunchKernelGGL((k_potential<T, 96, VAR>), g, dim3(kThreads), 0, s, L); break;
    default: hipLaunchKernelGGL((k_potential<T, 128, VAR>), g, dim3(kThreads), 0, s, L); break;
  }
}

template <typename T>
void launch_potential(hipStream_t s, int tf, int var, const StageList &L) {
  if (!L.total) return;
  switch (var) {
    case 1: potential_var<T, 1>(s, tf, L); break;
    case 2: potential_var<T, 2>(s, tf, L); break;
    default: potential_var<T, 0>(s, tf, L); break;
  }
}

}  // namespace pgxc
