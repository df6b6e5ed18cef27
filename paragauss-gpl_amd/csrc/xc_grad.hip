// Nuclear gradient of E_xc for gfx950: ParaGauss's F1 (basis centres,
// modules/post_scf_module.f90:150-185, grad_xc when weight_grads is off) and,
// with the grid moving, F2 (points and Becke weights).  Per spin
//
//   dE/dR_A = -2 sum_p sum_{i on A} t_i(p),
//   t_i     = grad phi_i (2 a X_i + b . Y_i) + X_i (b . grad) grad phi_i,
//
// X = Phi P, Y_c = (d/dc Phi) P, a = w dF/drho / 2, b = w (2 dF/dg_ss grad rho_s
// + dF/dg_ab grad rho_s') of the build (the second term only for GGA).  The
// bracket's Z = 2 a X + b . Y is one product, Z = W P with W = 2 a Phi + b .
// grad Phi per point, so a GGA gradient takes two products (X and Z) where X
// and the three Y_c are four.  The basis functions' second derivatives are
// formed along b where they are used, never stored.
#include <algorithm>
#include <type_traits>

#include "xc_basis.h"

namespace pgxc {
namespace {

// A value and its derivative along the point's b.
struct Du {
  double v, d;
};
__device__ __forceinline__ Du operator+(Du a, Du b) { return {a.v + b.v, a.d + b.d}; }
__device__ __forceinline__ Du operator-(Du a, Du b) { return {a.v - b.v, a.d - b.d}; }
__device__ __forceinline__ Du operator*(Du a, Du b) { return {a.v * b.v, a.d * b.v + a.v * b.d}; }
__device__ __forceinline__ Du operator*(double s, Du a) { return {s * a.v, s * a.d}; }

// Solid harmonics up to L and their gradients as such pairs: the recursion of
// the value evaluation (m = 1 z-like, (2m, 2m+1) pairs, top pair by the (x, y)
// rotation) and its derivatives, carried out on values with a derivative along b.
template <int L>
__device__ __forceinline__ void sh_along(Du x, Du y, Du z, Du *C, Du *Cx, Du *Cy, Du *Cz) {
  const Du zero = {0.0, 0.0}, one = {1.0, 0.0};
  const Du r2 = x * x + y * y + z * z;
  C[0] = one;
  Cx[0] = Cy[0] = Cz[0] = zero;
  if constexpr (L >= 1) {
    C[1] = z; C[2] = x; C[3] = y;
    Cx[1] = zero; Cy[1] = zero; Cz[1] = one;
    Cx[2] = one; Cy[2] = zero; Cz[2] = zero;
    Cx[3] = zero; Cy[3] = one; Cz[3] = zero;
  }
  // u = s z p - t r2 q and its derivatives
  auto two = [&](int o, double s, int p, double t, int q) {
    C[o] = s * (z * C[p]) - t * (r2 * C[q]);
    Cx[o] = s * (z * Cx[p]) - t * (2.0 * (x * C[q]) + r2 * Cx[q]);
    Cy[o] = s * (z * Cy[p]) - t * (2.0 * (y * C[q]) + r2 * Cy[q]);
    Cz[o] = s * (C[p] + z * Cz[p]) - t * (2.0 * (z * C[q]) + r2 * Cz[q]);
  };
#pragma unroll
  for (int l = 2; l <= L; ++l) {
    const int o = l * l, o1 = (l - 1) * (l - 1), o2 = (l - 2) * (l - 2);
    const double lr = l, l1r = l - 1, ll1r = 2 * l - 1;
    two(o, ll1r / lr, o1, l1r / lr, o2);
#pragma unroll
    for (int im = 1; im <= l - 2; ++im) {
      const double sim = (double)(im * im);
      const double rlm = 1.0 / sqrt(lr * lr - sim), rl1m = sqrt(l1r * l1r - sim);
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int m = 2 * im + k - 1;
        two(o + m, ll1r * rlm, o1 + m, rl1m * rlm, o2 + m);
      }
    }
    const double rlm = ll1r / sqrt(lr * lr - l1r * l1r);
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int m = 2 * l - 3 + k;
      C[o + m] = rlm * (z * C[o1 + m]);
      Cx[o + m] = rlm * (z * Cx[o1 + m]);
      Cy[o + m] = rlm * (z * Cy[o1 + m]);
      Cz[o + m] = rlm * (C[o1 + m] + z * Cz[o1 + m]);
    }
    const double rll = sqrt(ll1r / (2.0 * lr));
    const int i2 = o1 + 2 * l - 3, i1 = o1 + 2 * l - 2, a = o + 2 * l - 1, b = o + 2 * l;
    C[a] = rll * (x * C[i2] - y * C[i1]);
    Cx[a] = rll * (C[i2] + x * Cx[i2] - y * Cx[i1]);
    Cy[a] = rll * (x * Cy[i2] - C[i1] - y * Cy[i1]);
    Cz[a] = rll * (x * Cz[i2] - y * Cz[i1]);
    C[b] = rll * (y * C[i2] + x * C[i1]);
    Cx[b] = rll * (y * Cx[i2] + C[i1] + x * Cx[i1]);
    Cy[b] = rll * (C[i2] + y * Cy[i2] + x * Cy[i1]);
    Cz[b] = rll * (y * Cz[i2] + x * Cz[i1]);
  }
}

// One point's inputs of the bracket: X and Z (rows of Mc, read at column p;
// LDA: Z = 2 a X) and b.
struct Bracket {
  const double *X, *Z;
  long Mc;
  unsigned p;
  double a2, b[3];
};

// t += sum over the 2 L + 1 functions of a shell's radial function R (at f0,
// nf apart) of the bracket, with r0 = R, r1 = R'/r, r2 = (R'/r)'/r and bx = b . x
template <int L, bool GGA>
__device__ __forceinline__ void bracket_fn(const Bracket &B, long f0, int nf, double r0, double r1,
                                           double r2, double x, double y, double z, double bx,
                                           const Du *C, const Du *Cx, const Du *Cy, const Du *Cz,
                                           double (&t)[3]) {
  constexpr int o = L * L;
  double X[2 * L + 1], Z[2 * L + 1];
#pragma unroll
  for (int m = 0; m < 2 * L + 1; ++m) {
    const long q = (f0 + (long)m * nf) * B.Mc;
    X[m] = gld_row(B.X + q, B.p);
    Z[m] = GGA ? gld_row(B.Z + q, B.p) : B.a2 * X[m];
  }
  double u0[3] = {0.0, 0.0, 0.0}, u1[3] = {0.0, 0.0, 0.0}, zs = 0.0, xs = 0.0, xg = 0.0;
#pragma unroll
  for (int m = 0; m < 2 * L + 1; ++m) {
    const Du g[3] = {Cx[o + m], Cy[o + m], Cz[o + m]};
    zs += Z[m] * C[o + m].v;
#pragma unroll
    for (int d = 0; d < 3; ++d) u0[d] += Z[m] * g[d].v;
    if (GGA) {
      xs += X[m] * C[o + m].v;
      xg += X[m] * C[o + m].d;
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        u0[d] += X[m] * g[d].d;
        u1[d] += X[m] * g[d].v;
      }
    }
  }
  const double xx[3] = {x, y, z};
  double s = r1 * zs;
  if (GGA) s += r1 * xg + r2 * bx * xs;
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    t[d] += r0 * u0[d] + s * xx[d];
    if (GGA) t[d] += r1 * (bx * u1[d] + B.b[d] * xs);
  }
}

template <int L, bool GGA>
__device__ __forceinline__ void bracket_shell(const Bracket &B, const ShellD &sh, const double *tab,
                                              double x, double y, double z, const Du *C, const Du *Cx,
                                              const Du *Cy, const Du *Cz, double (&t)[3]) {
  const int ne = sh.n_exp, nu = sh.n_unc, nc = sh.n_contr, nf = nu + nc;
  const double rr = x * x + y * y + z * z, bx = GGA ? B.b[0] * x + B.b[1] * y + B.b[2] * z : 0.0;
  double s0[kMaxContr], s1[kMaxContr], s2[kMaxContr];
#pragma unroll
  for (int k = 0; k < kMaxContr; ++k) s0[k] = s1[k] = s2[k] = 0.0;
  for (int e0 = 0; e0 < ne; e0 += kPB) {  // as shell_emit
    const PrimBlock<double> q(tab, nc, e0);
    double r0[kPB], r1[kPB], r2[kPB];
    bool any = false;
#pragma unroll
    for (int i = 0; i < kPB; ++i) any = any || q.al[i] * rr < 50.0;
    const bool live = __ballot(any) != 0;
#pragma unroll
    for (int i = 0; i < kPB; ++i) r0[i] = 0.0;
    if (live) {
#pragma unroll
      for (int i = 0; i < kPB; ++i) {
        const double ar2 = q.al[i] * rr, v = q.nv[i] * exp(-ar2);
        r0[i] = ar2 < 50.0 ? v : 0.0;  // the value evaluation's cut-off
      }
    }
#pragma unroll
    for (int i = 0; i < kPB; ++i) {
      r1[i] = -2.0 * q.al[i] * r0[i];
      r2[i] = -2.0 * q.al[i] * r1[i];
      if (e0 + i < nu)
        bracket_fn<L, GGA>(B, sh.func_off + e0 + i, nf, r0[i], r1[i], r2[i], x, y, z, bx, C, Cx, Cy, Cz, t);
    }
    if (!live) continue;
#pragma unroll
    for (int k = 0; k < kMaxContr; ++k)
      if (k < nc) {
#pragma unroll
        for (int i = 0; i < kPB; ++i) {
          const double c = q.coeff(k, i);
          s0[k] += r0[i] * c;
          s1[k] += r1[i] * c;
          s2[k] += r2[i] * c;
        }
      }
  }
#pragma unroll
  for (int k = 0; k < kMaxContr; ++k)
    if (k < nc)
      bracket_fn<L, GGA>(B, sh.func_off + nu + k, nf, s0[k], s1[k], s2[k], x, y, z, bx, C, Cx, Cy, Cz, t);
}

// The brackets of one atom's live shells at the thread's point.
template <int LA, bool GGA>
__device__ __forceinline__ void bracket_atom(const UnitD &U, int s0, unsigned live, const Bracket &B,
                                             double x, double y, double z, double (&t)[3]) {
  constexpr int NLM = (LA + 1) * (LA + 1);
  Du C[NLM], Cx[NLM], Cy[NLM], Cz[NLM];
  sh_along<LA>({x, B.b[0]}, {y, B.b[1]}, {z, B.b[2]}, C, Cx, Cy, Cz);
  for (; live; live &= live - 1) {
    const ShellD sh = shell_at(U.shells + s0 + __builtin_ctz(live));
    const double *tab = U.tabd + sh.tab;
    switch (sh.l) {
      case 0: bracket_shell<0, GGA>(B, sh, tab, x, y, z, C, Cx, Cy, Cz, t); break;
      case 1: if constexpr (LA >= 1) bracket_shell<1, GGA>(B, sh, tab, x, y, z, C, Cx, Cy, Cz, t); break;
      case 2: if constexpr (LA >= 2) bracket_shell<2, GGA>(B, sh, tab, x, y, z, C, Cx, Cy, Cz, t); break;
      case 3: if constexpr (LA >= 3) bracket_shell<3, GGA>(B, sh, tab, x, y, z, C, Cx, Cy, Cz, t); break;
      case 4: if constexpr (LA >= 4) bracket_shell<4, GGA>(B, sh, tab, x, y, z, C, Cx, Cy, Cz, t); break;
    }
  }
}

// Sum of v over the wave's 64 lanes, in every lane, in a fixed order.
__device__ __forceinline__ double wave_sum(double v) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
  return v;
}

// item = 256-point block of a chunk's unit: its basis items (block, atom range)
// in turn, the brackets of every atom's functions that are not cut off summed
// over each wave's points into part[item][atom of the range][wave][3], and over
// functions into pm[d][p] += 2 t (w grad f at the point: its motion with its
// atom) when pm is given.  XZ = [2][NP][Mc] at the tiles' functions; st: the
// build's coefficients a, b (planes stride np apart).  Bound by the reads of X
// and Z and the registers of their use (two waves a SIMD; one: 0.80 ms; with f and
// g shells one, 14 registers spilled in the GGA kernel).  Per
// (H2O)16 chunk of 245 760 points 0.38 ms (0.48 with a range staged in LDS and a
// branch per primitive; 0.67 when the items came through loads the compiler takes
// for different lanes' and everything after them went per lane); storing the six
// second-derivative planes of every function and point and reading 13 planes back
// twice, once per sum, took 2.7 ms.
template <bool GGA, int LMAX>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(LMAX <= 2 ? 2 : 1))) void k_bracket(const UnitD *__restrict__ unit,
                                                      const double *__restrict__ XZ,
                                                      const double *__restrict__ st, long np,
                                                      double *__restrict__ pm,
                                                      double *__restrict__ part) {
  const UnitD &U = *unit;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const long Mc = U.Mc, cs = (long)U.NP * Mc;
  for (long blk = blockIdx.x; blk < Mc / kThreads; blk += gridDim.x) {
    long i0 = 0, hi = U.nbi;  // the block's items: they are listed block by block
    while (i0 < hi) {
      const long mid = (i0 + hi) >> 1;
      if ((long)(cld(U.bitems + mid) >> 16) < blk) i0 = mid + 1; else hi = mid;
    }
    const long p = blk * kThreads + tid;
    Bracket B;
    B.X = XZ;
    B.Z = XZ + cs;
    B.Mc = Mc;
    B.p = (unsigned)p;
    B.a2 = 2.0 * st[(S_A)*np + p];
    for (int d = 0; d < 3; ++d) B.b[d] = GGA ? st[(S_BX + d) * np + p] : 0.0;
    const double r[3] = {gld(U.gx + p), gld(U.gy + p), gld(U.gz + p)};
    double tp[3] = {0.0, 0.0, 0.0};
    for (long item = i0; item < U.nbi && (long)(cld(U.bitems + item) >> 16) == blk; ++item) {
      const unsigned mask = item_mask(U, item);
      const int rng = (int)(cld(U.bitems + item) & 0xffffu), na = cld(&U.ranges[rng].n_atoms);
      for (int a = 0; a < na; ++a) {
        const ItemAtom q = item_atom(U, rng, a, mask);
        double t[3] = {0.0, 0.0, 0.0};
        if (!q.live) {
          if (lane < 3) part[((item * kRangeAtoms + a) * 4 + wave) * 3 + lane] = 0.0;
          continue;
        }
        const double x = r[0] - q.x, y = r[1] - q.y, z = r[2] - q.z;
        switch (q.lmax) {
          case 0: bracket_atom<0, GGA>(U, q.s0, q.live, B, x, y, z, t); break;
          case 1: bracket_atom<1, GGA>(U, q.s0, q.live, B, x, y, z, t); break;
          case 2: if constexpr (LMAX >= 2) bracket_atom<2, GGA>(U, q.s0, q.live, B, x, y, z, t); break;
          default: if constexpr (LMAX >= 4) bracket_atom<4, GGA>(U, q.s0, q.live, B, x, y, z, t); break;
        }
        for (int d = 0; d < 3; ++d) {
          tp[d] += t[d];
          const double s = wave_sum(t[d]);
          if (lane == 0) part[((item * kRangeAtoms + a) * 4 + wave) * 3 + d] = s;
        }
      }
    }
    if (pm)
      for (int d = 0; d < 3; ++d) pm[d * np + p] += 2.0 * tp[d];
  }
}

// item = atom of a range: grad[atom][d] -= 2 x the sum of part over the chunk's
// basis items of the range, in a fixed order (a thread takes every 256th item,
// then the lanes and the waves are summed).  Bound by the walk over the item
// list: four codes are read at a time; 21 us for an (H2O)16 chunk.  One workgroup
// per range instead, 24 sums a thread, filled 6 CUs there and 12 for (H2O)32 (246
// us): energies and gradient of (H2O)16, four chunks, 15.0 ms against 14.5.
__global__ __launch_bounds__(kThreads) void k_bracket_sum(const UnitD *__restrict__ unit,
                                                          const double *__restrict__ part,
                                                          double *__restrict__ grad) {
  __shared__ double sh[kThreads / 64][3];
  const UnitD &U = *unit;
  const unsigned rng = blockIdx.x / kRangeAtoms;
  const int a = blockIdx.x % kRangeAtoms, tid = threadIdx.x;
  const RangeD R = U.ranges[rng];
  if (a >= R.n_atoms) return;
  double s[3] = {0.0, 0.0, 0.0};
  for (long i0 = tid; i0 < U.nbi; i0 += 4 * kThreads) {
    unsigned code[4];
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      const long i = i0 + t * kThreads;
      code[t] = i < U.nbi ? gld(U.bitems + i) & 0xffffu : ~0u;
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      if (code[t] != rng) continue;
      const double *q = part + ((i0 + t * kThreads) * kRangeAtoms + a) * 12;
      for (int w = 0; w < 4; ++w)
        for (int d = 0; d < 3; ++d) s[d] += q[3 * w + d];
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const double t = wave_sum(s[d]);
    if ((tid & 63) == 0) sh[tid >> 6][d] = t;
  }
  __syncthreads();
  if (tid < 3)
    grad[3 * U.ratoms[R.atom_begin + a] + tid] -=
        2.0 * ((sh[0][tid] + sh[1][tid]) + (sh[2][tid] + sh[3][tid]));
}

// coef = 2 a, b of the build (planes stride np apart): the W pass over them
// gives 2 a Phi + b . grad Phi
__global__ __launch_bounds__(kThreads) void k_bracket_coef(long Mc, const double *__restrict__ st,
                                                           long np, double *__restrict__ coef) {
  for (long p = (long)blockIdx.x * kThreads + threadIdx.x; p < Mc; p += (long)gridDim.x * kThreads) {
    coef[p] = 2.0 * st[S_A * np + p];
    for (int d = 0; d < 3; ++d) coef[(1 + d) * Mc + p] = st[(S_BX + d) * np + p];
  }
}

// out[j] += sum_i part[i][j], j < m: one workgroup per j, fixed order
__global__ __launch_bounds__(kThreads) void k_column_sum(long n, int m, const double *__restrict__ part,
                                                         double *__restrict__ out) {
  __shared__ double sh[kThreads];
  const int j = blockIdx.x, tid = threadIdx.x;
  double s = 0.0;
  for (long i = tid; i < n; i += kThreads) s += part[i * m + j];
  sh[tid] = s;
  __syncthreads();
  for (int o = kThreads / 2; o > 0; o >>= 1) {
    if (tid < o) sh[tid] += sh[tid + o];
    __syncthreads();
  }
  if (tid == 0) out[j] += sh[0];
}

// Adds a wave's three values to the three of atom `a`, kept per wave (only this
// wave touches them).
__device__ __forceinline__ void wave_add(double *acc, int a, double v0, double v1, double v2) {
  const int lane = threadIdx.x & 63;
  const double s0 = wave_sum(v0), s1 = wave_sum(v1), s2 = wave_sum(v2);
  if (lane < 3) acc[3 * a + lane] += lane == 0 ? s0 : lane == 1 ? s1 : s2;
}

// One wave per workgroup: the wave's points in groups of 64, pm summed by owner
// (the owners of a group in order of first appearance) into part[wave][na][3].
__global__ __launch_bounds__(64) void k_owner_sum(int na, long np, const int *__restrict__ owner,
                                                  const double *__restrict__ pm,
                                                  double *__restrict__ part) {
  double *acc = part + (long)blockIdx.x * na * 3;
  const int lane = threadIdx.x;
  for (int j = lane; j < 3 * na; j += 64) acc[j] = 0.0;
  __syncthreads();
  for (long g = blockIdx.x; g < np / 64; g += gridDim.x) {
    const long p = g * 64 + lane;
    const int own = owner[p];
    const double v[3] = {pm[p], pm[np + p], pm[2 * np + p]};
    unsigned long long left = __ballot(own >= 0);
    while (left) {
      const int a = __builtin_amdgcn_readlane(own, __builtin_ctzll(left));
      const bool mine = own == a;
      wave_add(acc, a, mine ? v[0] : 0.0, mine ? v[1] : 0.0, mine ? v[2] : 0.0);
      left &= ~__ballot(mine);
    }
  }
}

// ------------------------------------------------- Becke weight derivatives
// w_p = w_atomic P_A(r_p) / Z, P_C = prod_{D != C} s(mu_CD), Z = sum_C P_C,
// mu_CD = (|r - R_C| - |r - R_D|) / |R_C - R_D|, s = (1 - f3(mu)) / 2 with f3
// the three-fold iterated polynomial x (3 - x^2) / 2 (no atomic-size
// adjustment); the point moves with its owner A.  With sigma = s'/s:
//   d log P_C / dR_B = sum_{D != C} sigma(mu_CD) d mu_CD / dR_B
//   dw / dR_B = w sum_C (delta_CA - P_C / Z) d log P_C / dR_B.
// s = 0 only at mu = +-1, where s' = 0 too: sigma is taken as 0 there.
__device__ __forceinline__ void becke_sigma(double mu, double &s, double &sig) {
  const double f1 = mu * (3.0 - mu * mu) / 2.0, f2 = f1 * (3.0 - f1 * f1) / 2.0,
               f3 = f2 * (3.0 - f2 * f2) / 2.0;
  const double d = 1.5 * (1.0 - f2 * f2) * 1.5 * (1.0 - f1 * f1) * 1.5 * (1.0 - mu * mu);
  s = 0.5 * (1.0 - f3);
  sig = s > 0.0 ? -0.5 * d / s : 0.0;
}
__device__ __forceinline__ double becke_cell(double mu) {
  const double f1 = mu * (3.0 - mu * mu) / 2.0, f2 = f1 * (3.0 - f1 * f1) / 2.0;
  return 0.5 * (1.0 - f2 * (3.0 - f2 * f2) / 2.0);
}

struct Pt {
  double x, y, z;
};
// distance of the point from a centre, and the unit vector from the centre
__device__ __forceinline__ double dist(const AtomD &A, Pt r, double (&e)[3]) {
  e[0] = r.x - A.x;
  e[1] = r.y - A.y;
  e[2] = r.z - A.z;
  const double d = sqrt(e[0] * e[0] + e[1] * e[1] + e[2] * e[2]);
  const double id = d > 0.0 ? 1.0 / d : 0.0;
  e[0] *= id;
  e[1] *= id;
  e[2] *= id;
  return d;
}
__device__ __forceinline__ double dist(const AtomD &A, Pt r) {
  const double x = r.x - A.x, y = r.y - A.y, z = r.z - A.z;
  return sqrt(x * x + y * y + z * z);
}

// One wave per workgroup, a point per lane, groups of 64 points in turn: the
// wave's sums over its points of w f d log w / dR into part[wave][na][3].  As the
// weights themselves, only the centres C whose P_C can matter to a point of the
// wave (above becke_negligible of the nearest centre's, or the owner) are formed and
// differentiated: their P in scr[wave][listed centre][64], their indices in
// list[wave][na].  For each of them every other centre D takes
// k_C sigma d mu_CD / dR_D, C the same with d mu_CD / dR_C, and the owner
// d mu_CD / dr through the point's motion.  Bound by FP64 arithmetic; (H2O)16,
// 48 centres, 966 000 points: 4.9 ms, every pair of centres for every point (in
// two kernels) 21 ms.
// LDS: the wave's sums are kept there (na up to kLdsAtoms), else in part.
constexpr int kNearQ = 8, kFormQ = 4, kLdsAtoms = 1024;
template <bool LDS>
__global__ __launch_bounds__(64) void k_becke_grad(int na, const AtomD *__restrict__ atoms,
                                                   const double *__restrict__ inv_dist, long np,
                                                   const double *__restrict__ grid,
                                                   const double *__restrict__ fp,
                                                   const int *__restrict__ owner,
                                                   double *__restrict__ scr,
                                                   int *__restrict__ list,
                                                   double *__restrict__ part) {
  extern __shared__ double lacc[];  // 3 na
  double *acc = LDS ? lacc : part + (long)blockIdx.x * na * 3;
  double *P = scr + (long)blockIdx.x * na * 64;
  int *ls = list + (long)blockIdx.x * na;
  const int lane = threadIdx.x;
  for (int j = lane; j < 3 * na; j += 64) acc[j] = 0.0;
  __syncthreads();
  for (long g = blockIdx.x; g < np / 64; g += gridDim.x) {
    const long p = g * 64 + lane;
    const int own = owner[p];
    const double wf = own >= 0 ? grid[3 * np + p] * fp[p] : 0.0;
    const bool on = wf != 0.0;
    if (!__any(on)) continue;
    const Pt r = {grid[p], grid[np + p], grid[2 * np + p]};
    // the nearest centres and the nearest one's P, as in the weights
    double rn[kNearQ];
    int in[kNearQ];
#pragma unroll
    for (int t = 0; t < kNearQ; ++t) {
      rn[t] = __builtin_inf();
      in[t] = 0;
    }
    for (int i = 0; i < na; ++i) {
      double v = dist(atoms[i], r);
      int id = i;
      if (!__any(v < rn[kNearQ - 1])) continue;
#pragma unroll
      for (int t = 0; t < kNearQ; ++t)
        if (v < rn[t]) {
          const double tv = rn[t];
          const int ti = in[t];
          rn[t] = v;
          in[t] = id;
          v = tv;
          id = ti;
        }
    }
    double floor_p = 2.0 * becke_negligible(na);  // 2: a centre's cell with itself is 1/2
    for (int k = 0; k < na; ++k)
      floor_p *= becke_cell((rn[0] - dist(atoms[k], r)) * inv_dist[(long)in[0] * na + k]);
    int nl = 0;  // listed centres, the same for the wave
    for (int i = 0; i < na; ++i) {
      const double ri = dist(atoms[i], r);
      double pi = 2.0;
#pragma unroll
      for (int t = 0; t < kNearQ; ++t)
        if (t < na) pi *= becke_cell((ri - rn[t]) * inv_dist[(long)i * na + in[t]]);
      if (!__any(on && (!(pi <= floor_p) || i == own))) continue;
      if (lane == 0) ls[nl] = i;
      ++nl;
    }
    __syncthreads();
    double Z = 0.0;
    for (int c0 = 0; c0 < nl; c0 += kFormQ) {
      double ri[kFormQ], pi[kFormQ];
      int c[kFormQ];
#pragma unroll
      for (int m = 0; m < kFormQ; ++m) {
        c[m] = __builtin_amdgcn_readfirstlane(ls[min(c0 + m, nl - 1)]);
        ri[m] = dist(atoms[c[m]], r);
        pi[m] = 2.0;
      }
      for (int k = 0; k < na; ++k) {
        const double rk = dist(atoms[k], r);
#pragma unroll
        for (int m = 0; m < kFormQ; ++m) pi[m] *= becke_cell((ri[m] - rk) * inv_dist[(long)c[m] * na + k]);
      }
#pragma unroll
      for (int m = 0; m < kFormQ; ++m)
        if (c0 + m < nl) {
          P[(c0 + m) * 64 + lane] = pi[m];
          Z += pi[m];
        }
    }
    const double iz = 1.0 / Z;
    double rm[3] = {0.0, 0.0, 0.0};
    for (int c0 = 0; c0 < nl; c0 += kFormQ) {
      double rc[kFormQ], ec[kFormQ][3], kc[kFormQ], ac[kFormQ][3];
      int c[kFormQ];
#pragma unroll
      for (int m = 0; m < kFormQ; ++m) {
        const bool there = c0 + m < nl;
        c[m] = __builtin_amdgcn_readfirstlane(ls[min(c0 + m, nl - 1)]);
        rc[m] = dist(atoms[c[m]], r, ec[m]);
        kc[m] = on && there ? wf * ((c[m] == own ? 1.0 : 0.0) - P[min(c0 + m, nl - 1) * 64 + lane] * iz) : 0.0;
        ac[m][0] = ac[m][1] = ac[m][2] = 0.0;
      }
      for (int D = 0; D < na; ++D) {
        double eD[3], v[3] = {0.0, 0.0, 0.0};
        const AtomD &AD = atoms[D];
        const double rD = dist(AD, r, eD);
#pragma unroll
        for (int m = 0; m < kFormQ; ++m) {
          if (c[m] == D) continue;
          const double iR = inv_dist[(long)c[m] * na + D], mu = (rc[m] - rD) * iR;
          double s, sig;
          becke_sigma(mu, s, sig);
          const double T = kc[m] != 0.0 ? kc[m] * sig * iR : 0.0, M = T * mu * iR;
          const AtomD &AC = atoms[c[m]];
          const double dR[3] = {M * (AC.x - AD.x), M * (AC.y - AD.y), M * (AC.z - AD.z)};
#pragma unroll
          for (int d = 0; d < 3; ++d) {
            v[d] += T * eD[d] + dR[d];
            ac[m][d] -= T * ec[m][d] + dR[d];
            rm[d] += T * (ec[m][d] - eD[d]);
          }
        }
        wave_add(acc, D, v[0], v[1], v[2]);
      }
#pragma unroll
      for (int m = 0; m < kFormQ; ++m)
        if (c0 + m < nl) wave_add(acc, c[m], ac[m][0], ac[m][1], ac[m][2]);
    }
    // through the points' motion with their owners
    unsigned long long left = __ballot(on);
    while (left) {
      const int a = __builtin_amdgcn_readlane(own, __builtin_ctzll(left));
      const bool mine = on && own == a;
      wave_add(acc, a, mine ? rm[0] : 0.0, mine ? rm[1] : 0.0, mine ? rm[2] : 0.0);
      left &= ~__ballot(mine);
    }
    __syncthreads();  // ls is written again
  }
  if (LDS)
    for (int j = lane; j < 3 * na; j += 64) part[(long)blockIdx.x * na * 3 + j] = acc[j];
}

// own[internal point] = owner[caller point], -1 for padding
__global__ __launch_bounds__(kThreads) void k_gather_owner(long npts, long np, const int *__restrict__ perm,
                                                           const int *__restrict__ owner,
                                                           int *__restrict__ own) {
  for (long p = (long)blockIdx.x * kThreads + threadIdx.x; p < np; p += (long)gridDim.x * kThreads)
    own[p] = p < npts ? owner[perm[p]] : -1;
}

unsigned grid_of(long items, long cap) { return (unsigned)std::max<long>(1, std::min(items, cap)); }

}  // namespace

void launch_bracket_coef(hipStream_t s, long Mc, const double *st, long np, double *coef) {
  hipLaunchKernelGGL(k_bracket_coef, dim3(grid_of(Mc / kThreads, 2048)), dim3(kThreads), 0, s, Mc, st, np, coef);
}

void launch_bracket(hipStream_t s, bool gga, int lmax, const UnitD *unit, long Mc, int n_ranges,
                    const double *XZ, const double *st, long np, double *pm, double *part,
                    double *grad) {
  if (n_ranges <= 0) return;
  const dim3 g(grid_of(Mc / kThreads, 2048));
  auto go = [&](auto l) {
    constexpr int LM = decltype(l)::value;
    if (gga)
      hipLaunchKernelGGL((k_bracket<true, LM>), g, dim3(kThreads), 0, s, unit, XZ, st, np, pm, part);
    else
      hipLaunchKernelGGL((k_bracket<false, LM>), g, dim3(kThreads), 0, s, unit, XZ, st, np, pm, part);
  };
  if (lmax <= 2) go(std::integral_constant<int, 2>{});
  else go(std::integral_constant<int, 4>{});
  hipLaunchKernelGGL(k_bracket_sum, dim3((unsigned)(n_ranges * kRangeAtoms)), dim3(kThreads), 0, s, unit, part, grad);
}

long becke_grad_waves(int na, long np) {
  // one wave each, as many as fill the device a few times over and 256 MiB of
  // scratch allow
  const long per = (long)na * (64 * 8 + 4 + 24);
  return std::max<long>(1, std::min<long>({np / 64, 4096L, (256L << 20) / per}));
}

void launch_owner_sum(hipStream_t s, int na, long np, const int *owner, const double *pm, long waves,
                      double *part, double *grad) {
  hipLaunchKernelGGL(k_owner_sum, dim3((unsigned)waves), dim3(64), 0, s, na, np, owner, pm, part);
  hipLaunchKernelGGL(k_column_sum, dim3((unsigned)(3 * na)), dim3(kThreads), 0, s, waves, 3 * na, part, grad);
}

void launch_becke_grad(hipStream_t s, int na, const AtomD *atoms, const double *inv_dist, long np,
                       const double *grid, const double *fp, const int *owner, long waves,
                       double *scr, int *list, double *part, double *grad) {
  auto k = na <= kLdsAtoms ? k_becke_grad<true> : k_becke_grad<false>;
  hipLaunchKernelGGL(k, dim3((unsigned)waves), dim3(64), na <= kLdsAtoms ? 24 * na : 0, s, na, atoms, inv_dist,
                     np, grid, fp, owner, scr, list, part);
  hipLaunchKernelGGL(k_column_sum, dim3((unsigned)(3 * na)), dim3(kThreads), 0, s, waves, 3 * na, part, grad);
}

void launch_gather_owner(hipStream_t s, long npts, long np, const int *perm, const int *owner, int *own) {
  hipLaunchKernelGGL(k_gather_owner, dim3(grid_of(np / kThreads, 2048)), dim3(kThreads), 0, s, npts, np, perm,
                     owner, own);
}

}  // namespace pgxc
