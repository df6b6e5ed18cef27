// Basis evaluation on the device, shared by the basis and W stages and the
// nuclear gradient: solid harmonics, the shells' radial parts from scalar
// tables, and the walk over a basis item.
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
// point p of the [4][NP][Mc] planes: the row's address is the wave's (scalar, a
// step per function), the lane adds its point's 32-bit offset in the store.
template <typename T>
struct StorePhi {
  T *phi;
  long Mc, cs;
  unsigned p;
  template <int L, bool GRAD>
  __device__ __forceinline__ void emit(long f0, int nf, T r0, T r1, T x, T y, T z, const T *C,
                                       const T *Cx, const T *Cy, const T *Cz) const {
    T *row = phi + f0 * Mc;
    const long step = nf * Mc;
#pragma unroll
    for (int m = 0; m < 2 * L + 1; ++m, row += step) {
      T v, gx = T(0), gy = T(0), gz = T(0);
      fn_values<L, false>(m, r0, r1, x, y, z, C, Cx, Cy, Cz, v, gx, gy, gz);
      gst_row(row, p, v);
      if (GRAD) {
        fn_values<L, true>(m, r0, r1, x, y, z, C, Cx, Cy, Cz, v, gx, gy, gz);
        gst_row(row + cs, p, gx);
        gst_row(row + 2 * cs, p, gy);
        gst_row(row + 3 * cs, p, gz);
      }
    }
  }
};

// Reads of tables that no kernel writes, at addresses that are the same for the
// whole wave: scalar loads into scalar registers (the constant address space
// says so; through an ordinary pointer from a descriptor the compiler has to
// expect the stores in between to change them).
template <typename T>
__device__ __forceinline__ T cld(const T *p) {
  return *(const __attribute__((address_space(4))) T *)p;
}

// The units' shell tables in T: per shell its primitives in blocks of kPB (padded
// with the last exponent, norm and coefficients 0), a block's exponents, norms and
// the coefficients of each contraction in turn.
template <typename T>
__device__ __forceinline__ const T *shell_tables(const UnitD &U);
template <>
__device__ __forceinline__ const double *shell_tables<double>(const UnitD &U) { return U.tabd; }
template <>
__device__ __forceinline__ const float *shell_tables<float>(const UnitD &U) { return U.tabf; }

__device__ __forceinline__ ShellD shell_at(const ShellD *p) {
  ShellD s;
  s.atom = cld(&p->atom);
  s.l = cld(&p->l);
  s.n_exp = cld(&p->n_exp);
  s.n_unc = cld(&p->n_unc);
  s.n_contr = cld(&p->n_contr);
  s.tab = cld(&p->tab);
  s.func_off = cld(&p->func_off);
  return s;
}

// A block of a shell's table: loaded at once, so that a wave waits once for it
// (scalar loads return out of order: each wait is for all of them), with the
// first two contractions (the table ends with as much room); the others as used.
template <typename T>
struct PrimBlock {
  const T *p;
  T al[kPB], nv[kPB], c[2][kPB];
  __device__ __forceinline__ PrimBlock(const T *tab, int nc, int e0) : p(tab + (2 + nc) * e0) {
#pragma unroll
    for (int i = 0; i < kPB; ++i) {
      al[i] = cld(p + i);
      nv[i] = cld(p + kPB + i);
      c[0][i] = cld(p + 2 * kPB + i);
      c[1][i] = cld(p + 3 * kPB + i);
    }
  }
  __device__ __forceinline__ T coeff(int k, int i) const { return k < 2 ? c[k][i] : cld(p + (2 + k) * kPB + i); }
};

// tab: the shell's table.  Primitives go in blocks of kPB: radial factors formed
// without a branch per primitive (a block whose primitives are all cut off on
// the wave's points skips the exponentials and adds nothing), then added into
// the contractions in primitive order.
template <int L, bool GRAD, typename T, class Put>
__device__ __forceinline__ void shell_emit(const ShellD &sh, const T *tab, T x, T y, T z, T r2,
                                           const T *C, const T *Cx, const T *Cy, const T *Cz,
                                           const Put &put) {
  const int ne = sh.n_exp, nu = sh.n_unc, nc = sh.n_contr, nf = nu + nc;
  T rc0[kMaxContr], rc1[kMaxContr];
#pragma unroll
  for (int k = 0; k < kMaxContr; ++k) rc0[k] = rc1[k] = T(0);
  for (int e0 = 0; e0 < ne; e0 += kPB) {
    const PrimBlock<T> q(tab, nc, e0);
    T r0[kPB], r1[kPB];
    bool any = false;
#pragma unroll
    for (int i = 0; i < kPB; ++i) any = any || q.al[i] * r2 < T(50);
    const bool live = __ballot(any) != 0;
    if (live) {
#pragma unroll
      for (int i = 0; i < kPB; ++i) {
        const T ar2 = q.al[i] * r2, v = q.nv[i] * exp(-ar2);
        r0[i] = ar2 < T(50) ? v : T(0);  // primitive cut-off of radial1()
        r1[i] = (T(-2) * q.al[i]) * r0[i];
      }
    } else {
#pragma unroll
      for (int i = 0; i < kPB; ++i) r0[i] = r1[i] = T(0);
    }
#pragma unroll
    for (int i = 0; i < kPB; ++i)
      if (e0 + i < nu)
        put.template emit<L, GRAD>(sh.func_off + e0 + i, nf, r0[i], r1[i], x, y, z, C, Cx, Cy, Cz);
    if (!live) continue;
#pragma unroll
    for (int k = 0; k < kMaxContr; ++k)
      if (k < nc) {
#pragma unroll
        for (int i = 0; i < kPB; ++i) {
          const T c = q.coeff(k, i);
          rc0[k] += r0[i] * c;
          rc1[k] += r1[i] * c;
        }
      }
  }
#pragma unroll
  for (int k = 0; k < kMaxContr; ++k)
    if (k < nc)
      put.template emit<L, GRAD>(sh.func_off + nu + k, nf, rc0[k], rc1[k], x, y, z, C, Cx, Cy, Cz);
}

// The shells `live` (bits, from shell s0 on) of one atom at the thread's point.
template <int LA, bool GRAD, typename T, class Put>
__device__ __forceinline__ void basis_atom(const UnitD &U, int s0, unsigned live, T x, T y, T z,
                                           const Put &put) {
  constexpr int NLM = (LA + 1) * (LA + 1);
  T C[NLM], Cx[NLM], Cy[NLM], Cz[NLM];
  sh_eval<LA, T>(x, y, z, C, Cx, Cy, Cz);
  const T r2 = x * x + y * y + z * z;
  for (; live; live &= live - 1) {
    const ShellD sh = shell_at(U.shells + s0 + __builtin_ctz(live));
    const T *tab = shell_tables<T>(U) + sh.tab;
    switch (sh.l) {
      case 0: shell_emit<0, GRAD>(sh, tab, x, y, z, r2, C, Cx, Cy, Cz, put); break;
      case 1: if constexpr (LA >= 1) shell_emit<1, GRAD>(sh, tab, x, y, z, r2, C, Cx, Cy, Cz, put); break;
      case 2: if constexpr (LA >= 2) shell_emit<2, GRAD>(sh, tab, x, y, z, r2, C, Cx, Cy, Cz, put); break;
      case 3: if constexpr (LA >= 3) shell_emit<3, GRAD>(sh, tab, x, y, z, r2, C, Cx, Cy, Cz, put); break;
      case 4: if constexpr (LA >= 4) shell_emit<4, GRAD>(sh, tab, x, y, z, r2, C, Cx, Cy, Cz, put); break;
    }
  }
}

// One atom of a basis item on the wave's tile: its centre, first shell, largest
// l, and its shells that are not cut off there (bits from the first shell on).
struct ItemAtom {
  double x, y, z;
  int s0, lmax;
  unsigned live;
};
__device__ __forceinline__ ItemAtom item_atom(const UnitD &U, int rng, int a, unsigned mask) {
  const RangeD *R = U.ranges + rng;
  const AtomD *at = U.atoms + cld(U.ratoms + cld(&R->atom_begin) + a);
  ItemAtom q;
  q.s0 = cld(&at->shell_begin);
  const int n = cld(&at->shell_end) - q.s0;  // at most kAtomShells
  q.live = (mask >> (q.s0 - cld(&R->shell_begin))) & ((1u << n) - 1u);
  q.x = cld(&at->x);
  q.y = cld(&at->y);
  q.z = cld(&at->z);
  q.lmax = cld(&at->lmax);
  return q;
}

// The basis items' walk: item `local` of unit U is a 256-point block and a range
// of atoms; the shells of the range not cut off on a tile of the block are the
// bits of bflags[2 local + tile].  A wave's 64 points lie in one tile, so which
// shells it evaluates, and every table read, is uniform: scalar registers, no
// LDS, and waves that wait for no other.
__device__ __forceinline__ long item_point(const UnitD &U, long local) {
  return (long)(cld(U.bitems + local) >> 16) * kThreads + threadIdx.x;
}
__device__ __forceinline__ unsigned item_mask(const UnitD &U, long local) {
  return cld(U.bflags + 2 * local + (__builtin_amdgcn_readfirstlane(threadIdx.x >> 6) >> 1));
}
template <bool GRAD, int LMAX, typename T, class Put>
__device__ __forceinline__ void eval_basis_item(const UnitD &U, long local, long p, const Put &put) {
  const unsigned mask = item_mask(U, local);
  if (!mask) return;
  const int rng = (int)(cld(U.bitems + local) & 0xffffu), na = cld(&U.ranges[rng].n_atoms);
  const double gx = gld(U.gx + p), gy = gld(U.gy + p), gz = gld(U.gz + p);
  for (int a = 0; a < na; ++a) {
    const ItemAtom q = item_atom(U, rng, a, mask);
    if (!q.live) continue;  // no stage reads this atom's values on the wave's tile
    const T x = (T)(gx - q.x), y = (T)(gy - q.y), z = (T)(gz - q.z);
    // the kernel holds the registers of its largest case, so it is built
    // for the largest angular momentum of the list (every atom's lmax <= LMAX)
    switch (q.lmax) {
      case 0: basis_atom<0, GRAD>(U, q.s0, q.live, x, y, z, put); break;
      case 1: if constexpr (LMAX >= 1) basis_atom<1, GRAD>(U, q.s0, q.live, x, y, z, put); break;
      case 2: if constexpr (LMAX >= 2) basis_atom<2, GRAD>(U, q.s0, q.live, x, y, z, put); break;
      case 3: if constexpr (LMAX >= 3) basis_atom<3, GRAD>(U, q.s0, q.live, x, y, z, put); break;
      default: if constexpr (LMAX >= 4) basis_atom<4, GRAD>(U, q.s0, q.live, x, y, z, put); break;
    }
  }
}

}  // namespace pgxc
