// Basis evaluation on the device, shared by the basis and W stages and the
// nuclear gradient: solid harmonics, a range of atoms' data staged in LDS, and
// the walk over a staged range.
#pragma once
#include "pgxc_internal.h"
#include "xc_device.h"

namespace pgxc {

// --------------------------------------------------------- solid harmonics
// Racah-normalised real solid harmonics up to L and their gradients, by the
// reference's recursion in l (m = 1 is z-like, then (2m, 2m+1) pairs, top
// pair by the (x, y) rotation); gradients by differentiating the recursion.
template <int L, typename R>
__device__ __forceinline__ void sh_eval(R x, R y, R z, R *C, R *Cx, R *Cy, R *Cz) {
  const R r2 = x * x + y * y + z * z;
  C[0] = R(1);
  Cx[0] = Cy[0] = Cz[0] = R(0);
  if constexpr (L >= 1) {
    C[1] = z; C[2] = x; C[3] = y;
    Cx[1] = R(0); Cy[1] = R(0); Cz[1] = R(1);
    Cx[2] = R(1); Cy[2] = R(0); Cz[2] = R(0);
    Cx[3] = R(0); Cy[3] = R(1); Cz[3] = R(0);
  }
  const R dr2x = R(2) * x, dr2y = R(2) * y, dr2z = R(2) * z;
#pragma unroll
  for (int l = 2; l <= L; ++l) {
    const int o = l * l, o1 = (l - 1) * (l - 1), o2 = (l - 2) * (l - 2);
    const R lr = l, l1r = l - 1, ll1r = 2 * l - 1;
    C[o] = (ll1r * z * C[o1] - l1r * r2 * C[o2]) / lr;
    Cx[o] = (ll1r * z * Cx[o1] - l1r * (dr2x * C[o2] + r2 * Cx[o2])) / lr;
    Cy[o] = (ll1r * z * Cy[o1] - l1r * (dr2y * C[o2] + r2 * Cy[o2])) / lr;
    Cz[o] = (ll1r * (C[o1] + z * Cz[o1]) - l1r * (dr2z * C[o2] + r2 * Cz[o2])) / lr;
#pragma unroll
    for (int im = 1; im <= l - 2; ++im) {
      const R sim = (R)(im * im);
      const R rlm = R(1) / sqrt(lr * lr - sim);
      const R rl1m = sqrt(l1r * l1r - sim);
      const R a = ll1r * z * rlm, b = rl1m * r2 * rlm;
      const R daz = ll1r * rlm, db = rl1m * rlm;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int m = 2 * im + k - 1;
        C[o + m] = a * C[o1 + m] - b * C[o2 + m];
        Cx[o + m] = a * Cx[o1 + m] - b * Cx[o2 + m] - db * dr2x * C[o2 + m];
        Cy[o + m] = a * Cy[o1 + m] - b * Cy[o2 + m] - db * dr2y * C[o2 + m];
        Cz[o + m] = a * Cz[o1 + m] + daz * C[o1 + m] - b * Cz[o2 + m] - db * dr2z * C[o2 + m];
      }
    }
    {
      const R sim = (R)((l - 1) * (l - 1));
      const R rlm = R(1) / sqrt(lr * lr - sim);
      const R a = ll1r * z * rlm, daz = ll1r * rlm;
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int m = 2 * l - 3 + k;
        C[o + m] = a * C[o1 + m];
        Cx[o + m] = a * Cx[o1 + m];
        Cy[o + m] = a * Cy[o1 + m];
        Cz[o + m] = a * Cz[o1 + m] + daz * C[o1 + m];
      }
    }
    {
      const R rll = sqrt(ll1r / (R(2) * lr));
      const int i2 = o1 + 2 * l - 3, i1 = o1 + 2 * l - 2;
      C[o + 2 * l - 1] = (x * C[i2] - y * C[i1]) * rll;
      C[o + 2 * l] = (y * C[i2] + x * C[i1]) * rll;
      Cx[o + 2 * l - 1] = (C[i2] + x * Cx[i2] - y * Cx[i1]) * rll;
      Cy[o + 2 * l - 1] = (x * Cy[i2] - C[i1] - y * Cy[i1]) * rll;
      Cz[o + 2 * l - 1] = (x * Cz[i2] - y * Cz[i1]) * rll;
      Cx[o + 2 * l] = (y * Cx[i2] + C[i1] + x * Cx[i1]) * rll;
      Cy[o + 2 * l] = (C[i2] + y * Cy[i2] + x * Cy[i1]) * rll;
      Cz[o + 2 * l] = (y * Cz[i2] + x * Cz[i1]) * rll;
    }
  }
}

// ------------------------------------------------------------------- basis
// Evaluation in the output precision T: FP64 for the plain build, FP32 for
// the mixed builds (whose low-precision error is proportional to ||dP||).
// Value and gradient of function m of a shell of angular momentum L at one
// point (r0, r1: the contracted radial factor and its derivative factor);
// every consumer of basis values forms them with this one expression.
template <int L, bool GRAD, typename T>
__device__ __forceinline__ void fn_values(int m, T r0, T r1, T x, T y, T z, const T *C,
                                          const T *Cx, const T *Cy, const T *Cz, T &v, T &gx,
                                          T &gy, T &gz) {
  constexpr int o = L * L;
  const T sv = C[o + m];
  v = sv * r0;
  if (GRAD) {
    const T hv = sv * r1;
    gx = x * hv + Cx[o + m] * r0;
    gy = y * hv + Cy[o + m] * r0;
    gz = z * hv + Cz[o + m] * r0;
  }
}

// Emitter of the basis stage: stores a shell's values (and gradients) at
// point p of the [4][NP][Mc] planes.  Global (not flat) stores: a flat
// store also counts against the LDS wait counter, so every wait for the
// staged shell data would wait for the stores issued before it.
template <typename T>
struct StorePhi {
  T *phi;
  long Mc, cs;
  int p;
  template <int L, bool GRAD>
  __device__ __forceinline__ void emit(long f0, int nf, T r0, T r1, T x, T y, T z, const T *C,
                                       const T *Cx, const T *Cy, const T *Cz) const {
#pragma unroll
    for (int m = 0; m < 2 * L + 1; ++m) {
      const long q = (f0 + (long)m * nf) * Mc + p;
      T v, gx = T(0), gy = T(0), gz = T(0);
      fn_values<L, false>(m, r0, r1, x, y, z, C, Cx, Cy, Cz, v, gx, gy, gz);
      gst(phi + q, v);
      if (GRAD) {
        fn_values<L, true>(m, r0, r1, x, y, z, C, Cx, Cy, Cz, v, gx, gy, gz);
        gst(phi + cs + q, gx);
        gst(phi + 2 * cs + q, gy);
        gst(phi + 3 * cs + q, gz);
      }
    }
  }
};

// A range of atoms' basis data staged in LDS for a basis item: the shells,
// their exponents, norms and contraction coefficients in the evaluation
// precision, per atom its centre, shell range (relative to the range's
// first shell) and largest l, and per (shell, 32-point group of the item)
// whether to write its values (and gradients).
template <typename T>
struct RangeLds {
  ShellD sh[kRangeShells];
  T ex[kRangePrims], nm[kRangePrims], ct[kRangeContr];
  double ax[kRangeAtoms], ay[kRangeAtoms], az[kRangeAtoms];
  int s0[kRangeAtoms], s1[kRangeAtoms], lm[kRangeAtoms];
  uint8_t fl[kRangeShells][kThreads / kGroup];
};

// ex, nm: the shell's primitives; ct: its n_exp x n_contr coefficients.
// Primitives go in blocks of kPB: the block's exponents, norms and
// coefficients are read from LDS together (one wait, not one per read), its
// radial factors formed without a branch per primitive (a block whose
// primitives are all cut off on the wave's points skips the exponentials),
// then added into the contractions in primitive order.
constexpr int kPB = 4;
template <int L, bool GRAD, typename T, class Put>
__device__ __forceinline__ void shell_emit(const ShellD &sh, const T *ex, const T *nm, const T *ct,
                                           T x, T y, T z, T r2, const T *C, const T *Cx,
                                           const T *Cy, const T *Cz, const Put &put) {
  const int ne = sh.n_exp, nu = sh.n_unc, nc = sh.n_contr, nf = nu + nc;
  T rc0[kMaxContr], rc1[kMaxContr];
#pragma unroll
  for (int k = 0; k < kMaxContr; ++k) rc0[k] = rc1[k] = T(0);
  for (int e0 = 0; e0 < ne; e0 += kPB) {
    T al[kPB], ar2[kPB], nv[kPB], r0[kPB], r1[kPB];
    bool any = false;
#pragma unroll
    for (int i = 0; i < kPB; ++i) {
      const int e = min(e0 + i, ne - 1);  // past the shell: a repeat, never used
      al[i] = ex[e];
      nv[i] = nm[e];
      ar2[i] = al[i] * r2;
      any = any || (e0 + i < ne && ar2[i] < T(50));
    }
    if (__ballot(any)) {
#pragma unroll
      for (int i = 0; i < kPB; ++i) {
        const T v = nv[i] * exp(-ar2[i]);
        r0[i] = (e0 + i < ne && ar2[i] < T(50)) ? v : T(0);  // primitive cut-off of radial1()
        r1[i] = (T(-2) * al[i]) * r0[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < kPB; ++i) r0[i] = r1[i] = T(0);
    }
#pragma unroll
    for (int i = 0; i < kPB; ++i)
      if (e0 + i < nu)
        put.template emit<L, GRAD>(sh.func_off + e0 + i, nf, r0[i], r1[i], x, y, z, C, Cx, Cy, Cz);
#pragma unroll
    for (int k = 0; k < kMaxContr; ++k)
      if (k < nc) {
        T c[kPB];
#pragma unroll
        for (int i = 0; i < kPB; ++i) c[i] = ct[k * ne + min(e0 + i, ne - 1)];
#pragma unroll
        for (int i = 0; i < kPB; ++i)
          if (e0 + i < ne) {
            rc0[k] += r0[i] * c[i];
            rc1[k] += r1[i] * c[i];
          }
      }
  }
#pragma unroll
  for (int k = 0; k < kMaxContr; ++k)
    if (k < nc)
      put.template emit<L, GRAD>(sh.func_off + nu + k, nf, rc0[k], rc1[k], x, y, z, C, Cx, Cy, Cz);
}

// One atom's shells sb .. se-1 of the LDS image A at one point (e0, c0: the
// range's first primitive and coefficient); grp: the point's group in the
// item.
template <int LA, bool GRAD, typename T, class Put>
__device__ __forceinline__ void basis_atom(const RangeLds<T> &A, int sb, int se, int e0, int c0,
                                           T x, T y, T z, const Put &put, int grp) {
  constexpr int NLM = (LA + 1) * (LA + 1);
  T C[NLM], Cx[NLM], Cy[NLM], Cz[NLM];
  sh_eval<LA, T>(x, y, z, C, Cx, Cy, Cz);
  const T r2 = x * x + y * y + z * z;
  for (int s = sb; s < se; ++s) {
    if (!(A.fl[s][grp] & 1)) continue;  // no stage reads the shell's values on this group
    // every lane reads the same shell: its fields are uniform over the wave,
    // so the loops over its primitives and functions run on scalar counters
    ShellD sh = A.sh[s];
    sh.l = __builtin_amdgcn_readfirstlane(sh.l);
    sh.n_exp = __builtin_amdgcn_readfirstlane(sh.n_exp);
    sh.n_unc = __builtin_amdgcn_readfirstlane(sh.n_unc);
    sh.n_contr = __builtin_amdgcn_readfirstlane(sh.n_contr);
    sh.exp_off = __builtin_amdgcn_readfirstlane(sh.exp_off);
    sh.contr_off = __builtin_amdgcn_readfirstlane(sh.contr_off);
    sh.func_off = __builtin_amdgcn_readfirstlane(sh.func_off);
    const T *ex = A.ex + (sh.exp_off - e0), *nm = A.nm + (sh.exp_off - e0);
    const T *ct = A.ct + (sh.contr_off - c0);
    switch (sh.l) {
      case 0: shell_emit<0, GRAD>(sh, ex, nm, ct, x, y, z, r2, C, Cx, Cy, Cz, put); break;
      case 1: if constexpr (LA >= 1) shell_emit<1, GRAD>(sh, ex, nm, ct, x, y, z, r2, C, Cx, Cy, Cz, put); break;
      case 2: if constexpr (LA >= 2) shell_emit<2, GRAD>(sh, ex, nm, ct, x, y, z, r2, C, Cx, Cy, Cz, put); break;
      case 3: if constexpr (LA >= 3) shell_emit<3, GRAD>(sh, ex, nm, ct, x, y, z, r2, C, Cx, Cy, Cz, put); break;
      case 4: if constexpr (LA >= 4) shell_emit<4, GRAD>(sh, ex, nm, ct, x, y, z, r2, C, Cx, Cy, Cz, put); break;
    }
  }
}

// A basis item staged: its first point, the range's first primitive and
// coefficient, its atom count, and the point's coordinates.
struct BasisItem {
  long p;
  int e0, c0, n_atoms;
  double gx, gy, gz;
};

// Stages basis item `local` of unit U in A (every thread calls it; starts
// and ends with a barrier).
template <typename T>
__device__ __forceinline__ BasisItem stage_basis_item(const UnitD &U, long local, RangeLds<T> &A) {
  const int tid = threadIdx.x;
  const uint32_t e = U.bitems[local];
  const long blk = e >> 16;
  const int rng = (int)(e & 0xffffu);
  const RangeD R = U.ranges[rng];
  BasisItem it;
  it.e0 = R.exp_begin;
  it.c0 = R.contr_begin;
  it.n_atoms = R.n_atoms;
  it.p = blk * kThreads + tid;
  // the point's coordinates in FP64, loads in flight across the staging
  it.gx = gld(U.gx + it.p);
  it.gy = gld(U.gy + it.p);
  it.gz = gld(U.gz + it.p);
  __syncthreads();  // the previous item's reads of A are done
  for (int i = tid; i < R.n_shells; i += kThreads) A.sh[i] = U.shells[R.shell_begin + i];
  for (int i = tid; i < R.n_exp; i += kThreads) {
    A.ex[i] = (T)gld(U.exps + it.e0 + i);
    A.nm[i] = (T)gld(U.norms + it.e0 + i);
  }
  for (int i = tid; i < R.n_contr; i += kThreads) A.ct[i] = (T)gld(U.contr + it.c0 + i);
  if (tid < R.n_atoms) {
    const AtomD at = U.atoms[gld(U.ratoms + R.atom_begin + tid)];
    A.ax[tid] = at.x;
    A.ay[tid] = at.y;
    A.az[tid] = at.z;
    A.s0[tid] = at.shell_begin - R.shell_begin;
    A.s1[tid] = at.shell_end - R.shell_begin;
    A.lm[tid] = at.lmax;
  }
  if (tid < R.n_shells * (kThreads / kGroup))  // flag of (shell tid / 8, group tid % 8)
    A.fl[tid / (kThreads / kGroup)][tid % (kThreads / kGroup)] =
        (uint8_t)((U.bflags[8 * local + (tid >> 5)] >> (tid & 31)) & 1u);
  __syncthreads();
  return it;
}

// The staged range's atoms in turn at the thread's point, each shell written
// on the point's group handed to put.
template <bool GRAD, int LMAX, typename T, class Put>
__device__ __forceinline__ void eval_basis_item(const RangeLds<T> &A, const BasisItem &it,
                                                const Put &put) {
  const int grp = threadIdx.x / kGroup;
  const int na = __builtin_amdgcn_readfirstlane(it.n_atoms);
  for (int a = 0; a < na; ++a) {
    const int sb = __builtin_amdgcn_readfirstlane(A.s0[a]), se = __builtin_amdgcn_readfirstlane(A.s1[a]);
    bool any = false;
    for (int s = sb; s < se; ++s) any = any || (A.fl[s][grp] & 1);
    if (!any) continue;  // no stage reads this atom's values on the point's group
    const T x = (T)(it.gx - A.ax[a]), y = (T)(it.gy - A.ay[a]), z = (T)(it.gz - A.az[a]);
    // the kernel holds the registers of its largest case, so it is built
    // for the largest angular momentum of the list (every atom's lmax <= LMAX)
    switch (__builtin_amdgcn_readfirstlane(A.lm[a])) {
      case 0: basis_atom<0, GRAD>(A, sb, se, it.e0, it.c0, x, y, z, put, grp); break;
      case 1: if constexpr (LMAX >= 1) basis_atom<1, GRAD>(A, sb, se, it.e0, it.c0, x, y, z, put, grp); break;
      case 2: if constexpr (LMAX >= 2) basis_atom<2, GRAD>(A, sb, se, it.e0, it.c0, x, y, z, put, grp); break;
      case 3: if constexpr (LMAX >= 3) basis_atom<3, GRAD>(A, sb, se, it.e0, it.c0, x, y, z, put, grp); break;
      default: if constexpr (LMAX >= 4) basis_atom<4, GRAD>(A, sb, se, it.e0, it.c0, x, y, z, put, grp); break;
    }
  }
}

}  // namespace pgxc
