// HIP kernels of the XC build for gfx950 (CDNA4, wave64).  All stage kernels
// run over work lists of units (a unit = one grid chunk of one molecule), so one
// launch per stage serves a single molecule or a batch of many.
//
//   k_basis       basis values and gradients  (ParaGauss modules/orbital_module.f90:1742-1932,
//                 2421-2619; solid harmonics modules/solid_harmonics_module.f90:369-568)
//   k_functional  Slater + PW92 + PBE-x + PBE-c in FP64, closed-form derivatives
//                 (modules/xc_func.f90:187-305 and the term modules)
//   k_wbasis      W = a Phi + b . grad Phi  (modules/xc_hamiltonian.f90:1429-1483)
//   k_pack        V = H + H^T into the packed lower triangle (:1561-1567)
#include <algorithm>
#include <type_traits>

#include "pgxc_internal.h"
#include "xc_basis.h"
#include "xc_device.h"

namespace pgxc {

// -------------------------------------------------------------- functional
// Closed-shell terms; each returns F, dF/drho, dF/dgamma added into (f, fr, fg).
namespace xcf {
constexpr double PI = 3.14159265358979324;
constexpr double DEPS = 1.0e-30;

// Slater exchange: -(3/4)(3/pi)^(1/3) rho^(4/3), zero for rho <= 0
__device__ __forceinline__ void xalpha(double rho, double &f, double &fr) {
  const double xa = -(3.0 / 4.0) * cbrt(3.0 / PI);
  if (rho > 0.0) {
    const double c = cbrt(rho);
    f += xa * (rho * c);
    fr += xa * ((4.0 / 3.0) * c);
  }
}

// PW92 paramagnetic G(rs) and dG/drs
__device__ __forceinline__ void pw92_g(double rs, double &E, double &dE) {
  const double a = 0.031091, a1 = 0.21370, b1 = 7.5957, b2 = 3.5876, b3 = 1.6382,
               b4 = 0.49294;
  const double s = sqrt(rs);
  const double Q0 = -(2.0 * a * (1.0 + a1 * rs));
  const double Q1 = 2.0 * a * (b1 * s + b2 * rs + b3 * rs * s + b4 * rs * rs);
  const double Q2 = log(1.0 + 1.0 / Q1);
  const double dQ1 = 2.0 * a * (b1 * 0.5 / s + b2 + 1.5 * b3 * s + 2.0 * b4 * rs);
  const double dQ2 = (-dQ1 / (Q1 * Q1)) / (1.0 + 1.0 / Q1);
  E = Q0 * Q2;
  dE = (-2.0 * a * a1) * Q2 + Q0 * dQ2;
}

// n * eps_c^PW92(n, zeta = 0) with the n < DEPS clamp; value and dn
__device__ __forceinline__ void pw92_unpol(double n, double &F, double &dF) {
  const double crs = cbrt(3.0 / (4.0 * PI));
  double nn = n;
  bool fixed = false;
  if (nn < DEPS) { nn = DEPS; fixed = true; }
  const double rs = crs / cbrt(nn);
  double E, dE;
  pw92_g(rs, E, dE);
  F = nn * E;
  dF = fixed ? 0.0 : E + nn * dE * (-rs / (3.0 * nn));
}

__device__ __forceinline__ void pwldac(double rho, double &f, double &fr) {
  double F, dF;
  pw92_unpol(0.5 * rho + 0.5 * rho, F, dF);
  f += F;
  fr += dF;
}

// PBE exchange excess e_x G(s^2), G = kappa mu s2 / (kappa + mu s2)
__device__ __forceinline__ void pbex(double rho, double gam, double &f, double &fr,
                                     double &fg) {
  const double xa = -(3.0 / 4.0) * cbrt(3.0 / PI);
  const double kappa = 0.804, mu = 0.066725 * (PI * PI / 3.0);
  const double s2_fact = 1.0 / (4.0 * cbrt(3.0 * PI * PI) * cbrt(3.0 * PI * PI));
  double ex = 0.0, dex = 0.0;
  if (rho > 0.0) {
    const double c = cbrt(rho);
    ex = xa * (rho * c);
    dex = xa * ((4.0 / 3.0) * c);
  }
  double s2 = 0.0, s2r = 0.0, s2g = 0.0;
  if (rho >= 1.0e-20) {
    const double c = cbrt(rho);
    s2g = s2_fact / (rho * rho * c * c);
    s2 = gam * s2g;
    s2r = -(8.0 / 3.0) * s2 / rho;
  }
  const double den = kappa + mu * s2;
  const double G = kappa * mu * s2 / den;
  const double dG = (kappa * kappa * mu) / (den * den);
  f += ex * G;
  fr += dex * G + ex * dG * s2r;
  fg += ex * dG * s2g;
}

// PBE correlation gradient term n H(n, gamma), zeta = 0 (phi = 1)
__device__ __forceinline__ void pbec(double rho, double g2, double &f, double &fr,
                                     double &fg) {
  const double beta = 0.066725, gc = 0.03109069086965489503494086371;
  const double bg = beta / gc;
  const double K = PI / (16.0 * cbrt(3.0 * PI * PI));
  const double nv = 0.5 * rho + 0.5 * rho;
  if (nv <= 0.0) return;
  double Fl, dFl;
  pw92_unpol(nv, Fl, dFl);
  const double El = Fl / nv, dEl = dFl / nv - Fl / (nv * nv);
  // phi = (za^(2/3) + zb^(2/3)) / 2^(1/3) = 1 for za = zb = 1/2
  const double fi3 = 1.0;
  const double Ex = exp(-El / (gc * fi3));
  const double dd = Ex - 1.0 + DEPS;
  const double A = bg / dd;
  const double dA = (bg / (dd * dd)) * Ex * (dEl / (gc * fi3));
  const double c = cbrt(nv);
  const double n73 = nv * nv * c;
  const double D = n73 + DEPS;
  const double t2 = g2 / D * K;
  const double dt2n = -(g2 * K / (D * D)) * (7.0 / 3.0) * (nv * c);
  const double dt2g = K / D;
  const double x = A * t2;
  const double dxn = dA * t2 + A * dt2n, dxg = A * dt2g;
  const double q = 1.0 + x + x * x;
  const double rat = (1.0 + x) / q;
  const double drat = -x * (2.0 + x) / (q * q);
  const double arg = 1.0 + bg * t2 * rat;
  const double H = gc * fi3 * log(arg);
  const double pre = gc * fi3 / arg * bg;
  f += nv * H;
  fr += H + nv * pre * (dt2n * rat + t2 * drat * dxn);
  fg += nv * pre * (dt2g * rat + t2 * drat * dxg);
}

// The terms of mask in enum order (XAlpha, PWLDAc, PBEx, PBEc): each term's
// F into e[0..3] (zeroed by the caller), dF/drho and dF/dgamma summed over
// them; the functional's F is ((e0 + e1) + e2) + e3.
template <bool GGA>
__device__ __forceinline__ void terms(uint32_t mask, double rho, double gam, double (&e)[4],
                                      double &fr, double &fg) {
  if (mask & (1u << 1)) xalpha(rho, e[0], fr);
  if (mask & (1u << 3)) pwldac(rho, e[1], fr);
  if (GGA) {
    if (mask & (1u << 10)) pbex(rho, gam, e[2], fr, fg);
    if (mask & (1u << 18)) pbec(rho, gam, e[3], fr, fg);
  }
}
__device__ __forceinline__ double sum4(const double (&e)[4]) { return ((e[0] + e[1]) + e[2]) + e[3]; }
}  // namespace xcf

// ============================================================ work lists
// Every stage kernel is persistent: a grid of at most a few waves of
// workgroups walks the stage's item list (item = unit-local tile), in the
// order given by `order` (cost-model schedule) or, without one, in an
// XCD-blocked order so that neighbouring tiles share an XCD's L2.  Items write
// disjoint outputs, so the order never changes a result bit.

__device__ __forceinline__ long item_at(const int *__restrict__ order, long L, long total) {
  return order ? (long)order[L] : (long)xcd_remap((int)L, (int)total);
}

// ------------------------------------------------------------------- basis
// item = (256-point block, range of atoms) of a unit, of the pairs whose values a
// later stage reads; one thread per point, walking the range's atoms.  The tables
// are read by scalar loads (a shell's block of four primitives in one wait), rows
// addressed by the wave; staging a range in LDS behind two barriers, with row
// addresses per lane, took for an (H2O)32 build, one lane, 1.67 ms in FP32 (now
// 1.50: the writes, 7.0 GB a build, at 4.6 TB/s) and 3.06 in FP64 (2.88).
template <bool GRAD, typename T, int LMAX>
__global__ __launch_bounds__(kThreads) void k_basis(const UnitD *__restrict__ units, int nu,
                                                    const long *__restrict__ base,
                                                    const int *__restrict__ order, long total) {
  for (long L = blockIdx.x; L < total; L += gridDim.x) {
    const long item = item_at(order, L, total);
    const int u = find_unit(base, nu, item);
    const UnitD &U = units[u];
    const long local = item - base[u], p = item_point(U, local);
    const StorePhi<T> put{(T *)U.phi, U.Mc, (long)U.NP * U.Mc, (unsigned)p};
    eval_basis_item<GRAD, LMAX, T>(U, local, p, put);
  }
}

// Emitter of the W pass over basis items: W = a Phi + b . grad Phi of a shell's
// functions at point p (FP64 from the values in T, as a pass reading stored
// values forms it), stored in T or (SPLIT) as bf16 hi / lo planes for NS spins.
template <typename T, bool SPLIT, int NS>
struct StoreW {
  void *w[2];
  long Mc, cs;
  unsigned p;
  double a[2], b0[2], b1[2], b2[2];
  template <int L, bool GRAD>
  __device__ __forceinline__ void emit(long f0, int nf, T r0, T r1, T x, T y, T z, const T *C,
                                       const T *Cx, const T *Cy, const T *Cz) const {
    long row = f0 * Mc;  // rows' addresses are the wave's, the lane's point a 32-bit offset
    const long step = nf * Mc;
#pragma unroll
    for (int m = 0; m < 2 * L + 1; ++m, row += step) {
      T v, gx = T(0), gy = T(0), gz = T(0);
      fn_values<L, GRAD>(m, r0, r1, x, y, z, C, Cx, Cy, Cz, v, gx, gy, gz);
#pragma unroll
      for (int sp = 0; sp < NS; ++sp) {
        const double u = GRAD ? a[sp] * (double)v + b0[sp] * (double)gx + b1[sp] * (double)gy +
                                    b2[sp] * (double)gz
                              : a[sp] * (double)v;
        if constexpr (SPLIT) {
          __bf16 h, l;
          split_bf16((float)u, h, l);
          gst_row((uint16_t *)w[sp] + row, p, __builtin_bit_cast(uint16_t, h));
          gst_row((uint16_t *)w[sp] + row + cs, p, __builtin_bit_cast(uint16_t, l));
        } else {
          gst_row((T *)w[sp] + row, p, (T)u);
        }
      }
    }
  }
};

// W pass over the basis items: the basis functions evaluated again (the same
// expressions as the basis stage, so the same values) instead of read back, W
// written for the shells whose values the basis stage writes, the only ones the
// potential reads (TWO: both spins of an open-shell unit).  Trades the reads of
// four planes for the evaluation: functional and W of an (H2O)32 build, one
// lane, FP64 4.48 -> 2.64 ms, FP32 2.28 -> 1.77; 14-atom open shell 284 -> 140
// us, 23-atom LDA 127 -> 92; one water 23 -> 23.  Bound by vector instructions (50
// a wave and function, a third of them exponentials): with tables from scalar
// loads, rows addressed by the wave and one conversion to bf16 instead of an
// emulated one from FP64, FP64 1.69 ms, FP32 1.22, split BF16 2.02 -> 1.31.  With f
// and g shells (one or two waves a SIMD in FP64) it is the better one too where the
// stage takes time: functional and W of (H2O)16 with 784 functions, 391 000 points,
// evaluated / read in FP64 468 / 1296 us (LDA 291 / 492), FP32 306 / 629 (204 /
// 223), split BF16 370 / 659 (235 / 229); one water within 9 us, either way.
template <typename T, bool SPLIT, bool GRAD, bool TWO, int LMAX>
__global__ __launch_bounds__(kThreads) void k_wbasis(const UnitD *__restrict__ units, int nu,
                                                     const long *__restrict__ base,
                                                     const int *__restrict__ order, long total) {
  constexpr int NS = TWO ? 2 : 1;
  for (long L = blockIdx.x; L < total; L += gridDim.x) {
    const long item = item_at(order, L, total);
    const int u = find_unit(base, nu, item);
    const UnitD &U = units[u];
    const long local = item - base[u], p = item_point(U, local), Mc = U.Mc;
    StoreW<T, SPLIT, NS> put;
    put.Mc = Mc;
    put.cs = (long)U.NP * Mc;
    put.p = (unsigned)p;
#pragma unroll
    for (int sp = 0; sp < NS; ++sp) {
      const double *cf = sp ? U.coef2 : U.coef;
      put.w[sp] = sp ? U.W2 : U.W;
      put.a[sp] = gld(cf + p);
      put.b0[sp] = GRAD ? gld(cf + Mc + p) : 0.0;
      put.b1[sp] = GRAD ? gld(cf + 2 * Mc + p) : 0.0;
      put.b2[sp] = GRAD ? gld(cf + 3 * Mc + p) : 0.0;
    }
    eval_basis_item<GRAD, LMAX, T>(U, local, p, put);
  }
}

// item = 256-point block of a unit
template <bool GGA>
__global__ __launch_bounds__(kThreads) void k_functional(const UnitD *__restrict__ units, int nu,
                                                         const long *__restrict__ base,
                                                         const int *__restrict__ order,
                                                         long total) {
  __shared__ double se[kThreads], sq[kThreads];
  const int tid = threadIdx.x;
  for (long L = blockIdx.x; L < total; L += gridDim.x) {
    const long it = item_at(order, L, total);
    const int u = find_unit(base, nu, it);
    const UnitD &U = units[u];
    const long blk = it - base[u];
    const long p = blk * kThreads + tid, Mc = U.Mc, npad = U.npad;
    const double *part = U.part;
    double *state = U.state, *coef = U.coef;  // state is offset to the unit's first point
    double rho = 0.0, g0 = 0.0, g1 = 0.0, g2 = 0.0;
    // partial sums of the density items of this point's tile, one per chunk
    const int tile = (int)(p / kScreenTile);
    const int nch = (U.tf_off[tile + 1] - U.tf_off[tile] + U.dcols - 1) / U.dcols;
    for (int t = 0; t < nch; ++t) {
      rho += part[((long)t * 4 + 0) * Mc + p];
      if (GGA) {
        g0 += part[((long)t * 4 + 1) * Mc + p];
        g1 += part[((long)t * 4 + 2) * Mc + p];
        g2 += part[((long)t * 4 + 3) * Mc + p];
      }
    }
    if (U.incremental) {
      rho = state[S_RHO * npad + p] + rho;
      if (GGA) {
        g0 = state[S_GX * npad + p] + g0;
        g1 = state[S_GY * npad + p] + g1;
        g2 = state[S_GZ * npad + p] + g2;
      }
    }
    const double gam = g0 * g0 + g1 * g1 + g2 * g2;
    double e[4] = {0.0, 0.0, 0.0, 0.0}, fr = 0.0, fg = 0.0;
    xcf::terms<GGA>(U.mask, rho, gam, e, fr, fg);
    const double f = xcf::sum4(e);
    const double ww = U.gw[p];
    const double a = 0.5 * fr * ww;
    const double bq = ww * 2.0 * fg;
    const double b0 = bq * g0, b1 = bq * g1, b2 = bq * g2;
    if (U.incremental) {
      coef[0 * Mc + p] = a - state[S_A * npad + p];
      if (GGA) {
        coef[1 * Mc + p] = b0 - state[S_BX * npad + p];
        coef[2 * Mc + p] = b1 - state[S_BY * npad + p];
        coef[3 * Mc + p] = b2 - state[S_BZ * npad + p];
      }
    } else {
      coef[0 * Mc + p] = a;
      if (GGA) {
        coef[1 * Mc + p] = b0;
        coef[2 * Mc + p] = b1;
        coef[3 * Mc + p] = b2;
      }
    }
    state[S_RHO * npad + p] = rho;
    state[S_A * npad + p] = a;
    if (GGA) {
      state[S_GX * npad + p] = g0;
      state[S_GY * npad + p] = g1;
      state[S_GZ * npad + p] = g2;
      state[S_BX * npad + p] = b0;
      state[S_BY * npad + p] = b1;
      state[S_BZ * npad + p] = b2;
    }
    se[tid] = f * ww;
    sq[tid] = rho * ww;
    __syncthreads();
    for (int st = kThreads / 2; st > 0; st >>= 1) {
      if (tid < st) {
        se[tid] += se[tid + st];
        sq[tid] += sq[tid + st];
      }
      __syncthreads();
    }
    if (tid == 0) {
      U.epart[2 * blk + 0] = se[0];
      U.epart[2 * blk + 1] = sq[0];
    }
    __syncthreads();
  }
}

// ------------------------------------------------------- functional, ispin = 2
// Spin-polarised correlation on values with first derivatives in
// (n_a, n_b, g2): PW92 c_lda (modules/pw_ldac_module.f90:127-195) and PBE
// c_gga (modules/pbe_ggcxc_module.f90:96-140); exchange by spin scaling
// (modules/exchange.f90:253-288, :511-601) through the closed-shell terms.
namespace xcs {
using xcf::PI;
using xcf::DEPS;
struct Dv {
  double v, d0, d1, d2;
};
__device__ __forceinline__ Dv cst(double v) { return {v, 0.0, 0.0, 0.0}; }
__device__ __forceinline__ Dv operator+(Dv a, Dv b) { return {a.v + b.v, a.d0 + b.d0, a.d1 + b.d1, a.d2 + b.d2}; }
__device__ __forceinline__ Dv operator-(Dv a, Dv b) { return {a.v - b.v, a.d0 - b.d0, a.d1 - b.d1, a.d2 - b.d2}; }
__device__ __forceinline__ Dv operator*(Dv a, Dv b) {
  return {a.v * b.v, a.d0 * b.v + a.v * b.d0, a.d1 * b.v + a.v * b.d1, a.d2 * b.v + a.v * b.d2};
}
__device__ __forceinline__ Dv operator*(Dv a, double c) { return {a.v * c, a.d0 * c, a.d1 * c, a.d2 * c}; }
__device__ __forceinline__ Dv operator/(Dv a, Dv b) {
  const double q = a.v / b.v, r = 1.0 / b.v;
  return {q, (a.d0 - q * b.d0) * r, (a.d1 - q * b.d1) * r, (a.d2 - q * b.d2) * r};
}
__device__ __forceinline__ Dv chain(Dv a, double v, double g) { return {v, g * a.d0, g * a.d1, g * a.d2}; }
// the powers the formulas take, through sqrt / cbrt (arguments > 0 here)
__device__ __forceinline__ Dv sqrtd(Dv a) {
  const double t = sqrt(a.v);
  return chain(a, t, 0.5 / t);
}
__device__ __forceinline__ Dv cbrtd(Dv a) {  // a^(1/3)
  const double t = cbrt(a.v);
  return chain(a, t, t / (3.0 * a.v));
}
__device__ __forceinline__ Dv p23(Dv a) {  // a^(2/3)
  const double t = cbrt(a.v);
  return chain(a, t * t, (2.0 / 3.0) / t);
}
__device__ __forceinline__ Dv p43(Dv a) {  // a^(4/3)
  const double t = cbrt(a.v);
  return chain(a, a.v * t, (4.0 / 3.0) * t);
}
__device__ __forceinline__ Dv p73(Dv a) {  // a^(7/3)
  const double t = cbrt(a.v);
  return chain(a, a.v * a.v * t, (7.0 / 3.0) * a.v * t);
}
__device__ __forceinline__ Dv logd(Dv a) { return chain(a, log(a.v), 1.0 / a.v); }
__device__ __forceinline__ Dv expd(Dv a) {
  const double e = exp(a.v);
  return chain(a, e, e);
}

// PW92 G(rs) for the parameter sets of eps_c(zeta = 0), eps_c(zeta = 1) and
// -alpha_c (p = 1)
__device__ __forceinline__ Dv pw92_gs(Dv rs, int set) {
  const double A[3] = {0.031091, 0.015545, 0.016887};
  const double A1[3] = {0.21370, 0.20548, 0.11125};
  const double B1[3] = {7.5957, 14.1189, 10.357};
  const double B2[3] = {3.5876, 6.1977, 3.6231};
  const double B3[3] = {1.6382, 3.3662, 0.88026};
  const double B4[3] = {0.49294, 0.62517, 0.49671};
  const double a = A[set];
  const Dv s = sqrtd(rs);
  const Dv Q0 = (cst(1.0) + rs * A1[set]) * (-2.0 * a);
  const Dv Q1 = (s * B1[set] + rs * B2[set] + rs * s * B3[set] + rs * rs * B4[set]) * (2.0 * a);
  const Dv Q2 = logd(cst(1.0) + cst(1.0) / Q1);
  return Q0 * Q2;
}

// n eps_c^PW92(n_a, n_b)
__device__ __forceinline__ Dv pw92_spin(Dv na, Dv nb) {
  const double c13 = 1.0 / 3.0, c43 = 4.0 / 3.0;
  const double crs = cbrt(3.0 / (4.0 * PI));
  const double cf = 1.0 / (2.0 * cbrt(2.0) - 2.0);
  const double cfzz = 2.0 * c43 * c13 * cf;
  Dv n = na + nb;
  if (n.v < DEPS) n = cst(DEPS);
  const Dv rs = cst(crs) / cbrtd(n);
  const Dv eu = pw92_gs(rs, 0), ep = pw92_gs(rs, 1), ma = pw92_gs(rs, 2);
  const Dv z = (na - nb) / n, z2 = z * z, z4 = z2 * z2;
  const Dv fz = (p43(cst(1.0) + z + cst(DEPS)) + p43(cst(1.0) - z + cst(DEPS)) - cst(2.0)) * cf;
  const Dv ec = eu + (ep - eu) * fz * z4 - ma * fz * (cst(1.0) - z4) * (1.0 / cfzz);
  return n * ec;
}

// n H(n_a, n_b, g2), g2 = |grad n|^2, on lda = pw92_spin(n_a, n_b) (the
// PW92 term PBE-c is built on, computed once for both)
__device__ __forceinline__ Dv pbec_spin(Dv na, Dv nb, Dv g2, Dv lda) {
  const double beta = 0.066725, gc = 0.03109069086965489503494086371;
  const Dv n = na + nb;
  if (n.v <= 0.0) return cst(0.0);
  const Dv el = lda / n;
  Dv za = na / n, zb = nb / n;
  if (za.v < DEPS) za = cst(DEPS);
  if (zb.v < DEPS) zb = cst(DEPS);
  const Dv fi = (p23(za) + p23(zb)) * (1.0 / cbrt(2.0));
  const Dv fi2 = fi * fi, fi3 = fi2 * fi;
  const Dv A = cst(beta / gc) / (expd(el * (-1.0) / (fi3 * gc)) - cst(1.0) + cst(DEPS));
  const Dv t2 = g2 / (fi2 * p73(n) + cst(DEPS)) * (PI / (16.0 * cbrt(3.0 * PI * PI)));
  const Dv x = A * t2;
  const Dv rat = (cst(1.0) + x) / (cst(1.0) + x + x * x);
  const Dv H = fi3 * gc * logd(cst(1.0) + t2 * (beta / gc) * rat);
  return n * H;
}

// The spin-polarised terms of mask in enum order: exchange by spin scaling,
// PW92 once (its own term and the base of PBE-c, which needs it); each
// term's F into e[0..3], dF/drho_s into fr[s], dF/dg_ss into fgs[s] and
// dF/dg_ab into fab (all zeroed by the caller).
template <bool GGA>
__device__ __forceinline__ void terms(uint32_t mask, const double (&rho)[2], const double (&gss)[2],
                                      double gab, double (&e)[4], double (&fr)[2],
                                      double (&fgs)[2], double &fab) {
  if (mask & (1u << 1))
    for (int sp = 0; sp < 2; ++sp) {
      double x = 0.0, xr = 0.0;
      xcf::xalpha(2.0 * rho[sp], x, xr);
      e[0] += 0.5 * x;
      fr[sp] += xr;
    }
  Dv lda = cst(0.0);
  if (mask & (1u << 3)) {
    lda = pw92_spin({rho[0], 1.0, 0.0, 0.0}, {rho[1], 0.0, 1.0, 0.0});
    e[1] += lda.v;
    fr[0] += lda.d0;
    fr[1] += lda.d1;
  }
  if (GGA) {
    if (mask & (1u << 10))
      for (int sp = 0; sp < 2; ++sp) {
        double x = 0.0, xr = 0.0, xg = 0.0;
        xcf::pbex(2.0 * rho[sp], 4.0 * gss[sp], x, xr, xg);
        e[2] += 0.5 * x;
        fr[sp] += xr;
        fgs[sp] += 2.0 * xg;
      }
    if (mask & (1u << 18)) {
      const Dv F = pbec_spin({rho[0], 1.0, 0.0, 0.0}, {rho[1], 0.0, 1.0, 0.0},
                             {gss[0] + gss[1] + 2.0 * gab, 0.0, 0.0, 1.0}, lda);
      e[3] += F.v;
      fr[0] += F.d0;
      fr[1] += F.d1;
      fgs[0] += F.d2;
      fgs[1] += F.d2;
      fab += 2.0 * F.d2;
    }
  }
}
}  // namespace xcs

// item = 256-point block of an open-shell unit (the alpha spin's unit, which
// carries the beta spin's partials, coefficients and state in part2, coef2,
// state2).  Per point: rho_s, grad rho_s from the partials, f, dF/drho_s,
// dF/dg_aa, dF/dg_bb, dF/dg_ab, then a_s = w dF/drho_s / 2 and
// b_s = w (2 dF/dg_ss grad rho_s + dF/dg_ab grad rho_s')
// (modules/xc_hamiltonian.f90:1428-1445).
template <bool GGA>
__global__ __launch_bounds__(kThreads) void k_functional_spin(const UnitD *__restrict__ units, int nu,
                                                              const long *__restrict__ base,
                                                              const int *__restrict__ order,
                                                              long total) {
  __shared__ double se[kThreads], sq[kThreads];
  const int tid = threadIdx.x;
  for (long L = blockIdx.x; L < total; L += gridDim.x) {
    const long it = item_at(order, L, total);
    const int u = find_unit(base, nu, it);
    const UnitD &U = units[u];
    const long blk = it - base[u];
    const long p = blk * kThreads + tid, Mc = U.Mc, npad = U.npad;
    const double *part[2] = {U.part, U.part2};
    double *state[2] = {U.state, U.state2};
    double *coef[2] = {U.coef, U.coef2};
    double rho[2], g[2][3];
    const int tile = (int)(p / kScreenTile);
    const int nch = (U.tf_off[tile + 1] - U.tf_off[tile] + U.dcols - 1) / U.dcols;
    for (int sp = 0; sp < 2; ++sp) {
      double r = 0.0, g0 = 0.0, g1 = 0.0, g2 = 0.0;
      for (int t = 0; t < nch; ++t) {
        r += part[sp][((long)t * 4 + 0) * Mc + p];
        if (GGA) {
          g0 += part[sp][((long)t * 4 + 1) * Mc + p];
          g1 += part[sp][((long)t * 4 + 2) * Mc + p];
          g2 += part[sp][((long)t * 4 + 3) * Mc + p];
        }
      }
      if (U.incremental) {
        r = state[sp][S_RHO * npad + p] + r;
        if (GGA) {
          g0 = state[sp][S_GX * npad + p] + g0;
          g1 = state[sp][S_GY * npad + p] + g1;
          g2 = state[sp][S_GZ * npad + p] + g2;
        }
      }
      rho[sp] = r;
      g[sp][0] = g0;
      g[sp][1] = g1;
      g[sp][2] = g2;
    }
    const double gaa = g[0][0] * g[0][0] + g[0][1] * g[0][1] + g[0][2] * g[0][2];
    const double gbb = g[1][0] * g[1][0] + g[1][1] * g[1][1] + g[1][2] * g[1][2];
    const double gab = g[0][0] * g[1][0] + g[0][1] * g[1][1] + g[0][2] * g[1][2];
    const double gss[2] = {gaa, gbb};
    double e[4] = {0.0, 0.0, 0.0, 0.0}, fr[2] = {0.0, 0.0}, fgs[2] = {0.0, 0.0}, fab = 0.0;
    xcs::terms<GGA>(U.mask, rho, gss, gab, e, fr, fgs, fab);
    const double f = xcf::sum4(e);
    const double ww = U.gw[p];
    for (int sp = 0; sp < 2; ++sp) {
      const double a = 0.5 * fr[sp] * ww;
      double b[3];
      for (int c = 0; c < 3; ++c) b[c] = ww * (2.0 * fgs[sp] * g[sp][c] + fab * g[1 - sp][c]);
      double *cf = coef[sp], *st = state[sp];
      if (U.incremental) {
        cf[0 * Mc + p] = a - st[S_A * npad + p];
        if (GGA) {
          cf[1 * Mc + p] = b[0] - st[S_BX * npad + p];
          cf[2 * Mc + p] = b[1] - st[S_BY * npad + p];
          cf[3 * Mc + p] = b[2] - st[S_BZ * npad + p];
        }
      } else {
        cf[0 * Mc + p] = a;
        if (GGA) {
          cf[1 * Mc + p] = b[0];
          cf[2 * Mc + p] = b[1];
          cf[3 * Mc + p] = b[2];
        }
      }
      st[S_RHO * npad + p] = rho[sp];
      st[S_A * npad + p] = a;
      if (GGA) {
        st[S_GX * npad + p] = g[sp][0];
        st[S_GY * npad + p] = g[sp][1];
        st[S_GZ * npad + p] = g[sp][2];
        st[S_BX * npad + p] = b[0];
        st[S_BY * npad + p] = b[1];
        st[S_BZ * npad + p] = b[2];
      }
    }
    se[tid] = f * ww;
    sq[tid] = (rho[0] + rho[1]) * ww;
    __syncthreads();
    for (int st = kThreads / 2; st > 0; st >>= 1) {
      if (tid < st) {
        se[tid] += se[tid + st];
        sq[tid] += sq[tid + st];
      }
      __syncthreads();
    }
    if (tid == 0) {
      U.epart[2 * blk + 0] = se[0];
      U.epart[2 * blk + 1] = sq[0];
    }
    __syncthreads();
  }
}

// Each term's F at a point from rho and grad rho (per spin when SPIN)
template <bool GGA, bool SPIN>
__device__ __forceinline__ void point_terms(uint32_t mask, const double (&rho)[2],
                                            const double (&g)[2][3], double (&e)[4]) {
  if (!SPIN) {
    const double gam = g[0][0] * g[0][0] + g[0][1] * g[0][1] + g[0][2] * g[0][2];
    double fr = 0.0, fg = 0.0;
    xcf::terms<GGA>(mask, rho[0], gam, e, fr, fg);
  } else {
    const double gss[2] = {g[0][0] * g[0][0] + g[0][1] * g[0][1] + g[0][2] * g[0][2],
                           g[1][0] * g[1][0] + g[1][1] * g[1][1] + g[1][2] * g[1][2]};
    const double gab = g[0][0] * g[1][0] + g[0][1] * g[1][1] + g[0][2] * g[1][2];
    double fr[2] = {0.0, 0.0}, fgs[2] = {0.0, 0.0}, fab = 0.0;
    xcs::terms<GGA>(mask, rho, gss, gab, e, fr, fgs, fab);
  }
}

// ------------------------------------------------------- energy terms
// item = 256-point block of a unit (SPIN: an open-shell molecule's alpha unit):
// the XC energy of each functional term and the charge on the block, without
// potential coefficients and without touching the per-point state
// (post_scf_calc_xc_energy, modules/post_scf_module.f90:2204-2420).  Block
// sums go to eterm[blk][5]: XAlpha, PWLDAc, PBEx, PBEc, charge.
template <bool GGA, bool SPIN>
__global__ __launch_bounds__(kThreads) void k_energy(const UnitD *__restrict__ units, int nu,
                                                     const long *__restrict__ base,
                                                     const int *__restrict__ order, long total) {
  __shared__ double sh[5][kThreads];
  const int tid = threadIdx.x;
  for (long L = blockIdx.x; L < total; L += gridDim.x) {
    const long it = item_at(order, L, total);
    const int u = find_unit(base, nu, it);
    const UnitD &U = units[u];
    const long blk = it - base[u];
    const long p = blk * kThreads + tid, Mc = U.Mc;
    const int tile = (int)(p / kScreenTile);
    const int nch = (U.tf_off[tile + 1] - U.tf_off[tile] + U.dcols - 1) / U.dcols;
    double rho[2] = {0.0, 0.0}, g[2][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
    for (int sp = 0; sp < (SPIN ? 2 : 1); ++sp) {
      const double *part = sp ? U.part2 : U.part;
      for (int t = 0; t < nch; ++t) {
        rho[sp] += part[((long)t * 4 + 0) * Mc + p];
        if (GGA)
          for (int c = 0; c < 3; ++c) g[sp][c] += part[((long)t * 4 + 1 + c) * Mc + p];
      }
    }
    const double ww = U.gw[p];
    double e[4] = {0.0, 0.0, 0.0, 0.0};
    point_terms<GGA, SPIN>(U.mask, rho, g, e);
    for (int k = 0; k < 4; ++k) sh[k][tid] = e[k] * ww;
    sh[4][tid] = (rho[0] + rho[1]) * ww;
    __syncthreads();
    for (int st = kThreads / 2; st > 0; st >>= 1) {
      if (tid < st)
        for (int k = 0; k < 5; ++k) sh[k][tid] += sh[k][tid + st];
      __syncthreads();
    }
    if (tid < 5) U.eterm[5 * blk + tid] = sh[tid][0];
    __syncthreads();
  }
}

// ------------------------------------------------ energy density per point
// f at each point of a chunk from the per-point state of the last build
// (rho, grad rho per spin): the weight-derivative term of the nuclear
// gradient multiplies it by dw/dR.
template <bool GGA, bool SPIN>
__global__ __launch_bounds__(kThreads) void k_point_f(long Mc, long npad, uint32_t mask,
                                                      const double *__restrict__ st,
                                                      const double *__restrict__ st2,
                                                      double *__restrict__ fp) {
  for (long p = (long)blockIdx.x * kThreads + threadIdx.x; p < Mc; p += (long)gridDim.x * kThreads) {
    double rho[2] = {0.0, 0.0}, g[2][3] = {{0.0, 0.0, 0.0}, {0.0, 0.0, 0.0}};
    for (int sp = 0; sp < (SPIN ? 2 : 1); ++sp) {
      const double *S = sp ? st2 : st;
      rho[sp] = S[S_RHO * npad + p];
      if (GGA)
        for (int c = 0; c < 3; ++c) g[sp][c] = S[(S_GX + c) * npad + p];
    }
    double e[4] = {0.0, 0.0, 0.0, 0.0};
    point_terms<GGA, SPIN>(mask, rho, g, e);
    const double f = xcf::sum4(e);
    fp[p] = f;
  }
}

// -------------------------------------------------------------------- W
// item = (1024-point block, 16-function group), 4 consecutive points of one
// 32-point group per thread: W = a Phi + b . grad Phi for the functions of the
// point's tile (the potential contraction reads no others).  SPLIT (split-BF16
// builds, T = float): W stored as bf16 hi / lo planes.
template <typename T, bool GRAD, bool SPLIT, bool TWO>
__global__ __launch_bounds__(kThreads) void k_wmat(const UnitD *__restrict__ units, int nu,
                                                   const long *__restrict__ base,
                                                   const int *__restrict__ order, long total) {
  typedef T t4 __attribute__((ext_vector_type(4)));
  typedef uint16_t h4 __attribute__((ext_vector_type(4)));
  constexpr int NS = TWO ? 2 : 1;  // spins written from one read of the basis values
  for (long L = blockIdx.x; L < total; L += gridDim.x) {
    const long it = item_at(order, L, total);
    const int u = find_unit(base, nu, it);
    const UnitD &U = units[u];
    const long local = it - base[u];
    const int ng = U.NP / 16;
    const long p = (local / ng) * (4 * kThreads) + 4 * threadIdx.x;
    const long f0 = (local % ng) * 16;
    const long Mc = U.Mc, cs = (long)U.NP * Mc;
    const T *phi = (const T *)U.phi;
    void *Wout[2] = {U.W, TWO ? U.W2 : U.W};
    const double *cf[2] = {U.coef, TWO ? U.coef2 : U.coef};
    auto put = [&](int sp, long q, const double (&v)[4]) {
      if constexpr (SPLIT) {
        uint16_t *Wh = (uint16_t *)Wout[sp], *Wl = Wh + cs;
        h4 hi, lo;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          __bf16 h, l;
          split_bf16((float)v[j], h, l);
          hi[j] = __builtin_bit_cast(uint16_t, h);
          lo[j] = __builtin_bit_cast(uint16_t, l);
        }
        gst((h4 *)(Wh + q), hi);
        gst((h4 *)(Wl + q), lo);
      } else {
        t4 w;
#pragma unroll
        for (int j = 0; j < 4; ++j) w[j] = (T)v[j];
        gst((t4 *)((T *)Wout[sp] + q), w);
      }
    };
    const uint32_t *fb = U.tfb + (p / kScreenTile) * U.nwf;
#pragma unroll
    for (int h = 0; h < 2; ++h) {  // the item's two runs of 8 functions
      const long fr = f0 + h * kRun;
      const uint32_t fm = gld(fb + (fr >> 5)) >> (fr & 31);  // the run's functions in the tile's list
      if (!(fm & 0xffu)) continue;
      double a[NS][4], b0[NS][4] = {}, b1[NS][4] = {}, b2[NS][4] = {};
#pragma unroll
      for (int sp = 0; sp < NS; ++sp)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          a[sp][j] = gld(cf[sp] + p + j);
          if (GRAD) {
            b0[sp][j] = gld(cf[sp] + Mc + p + j);
            b1[sp][j] = gld(cf[sp] + 2 * Mc + p + j);
            b2[sp][j] = gld(cf[sp] + 3 * Mc + p + j);
          }
        }
#pragma unroll 4
      for (int k = 0; k < kRun; ++k) {
        if (!((fm >> k) & 1u)) continue;
        const long q = (fr + k) * Mc + p;
        const t4 v0 = gld((const t4 *)(phi + q));
        t4 v1 = {}, v2 = {}, v3 = {};
        if (GRAD) {
          v1 = gld((const t4 *)(phi + cs + q));
          v2 = gld((const t4 *)(phi + 2 * cs + q));
          v3 = gld((const t4 *)(phi + 3 * cs + q));
        }
#pragma unroll
        for (int sp = 0; sp < NS; ++sp) {
          double v[4];
#pragma unroll
          for (int j = 0; j < 4; ++j)
            v[j] = GRAD ? a[sp][j] * (double)v0[j] + b0[sp][j] * (double)v1[j] +
                              b1[sp][j] * (double)v2[j] + b2[sp][j] * (double)v3[j]
                        : a[sp][j] * (double)v0[j];
          put(sp, q, v);
        }
      }
    }
  }
}

// -------------------------------------------------------------------- pack
// Fold, item = 32 x 32 tile (rb >= cb): S(r, c) = sum over the listed splits of
// H(r, c) + H(c, r), each split's H gathered from its partial through the
// functions' places in it (0 where a split lacks one).  Of every kFoldSplits
// splits those with functions of both blocks of 32 (their mask bits) are
// listed in LDS with the places of the two blocks' functions, so the loop over
// them has only the elements' loads, four splits' at a time, to wait for.  The
// mirror tile's sums change places through LDS.  Bound by the latency of those
// loads; a tile all splits hold sets the time, hence the segments, of at most 64
// splits while there are no more than 32 of them: (H2O)32, 960 splits, 500 MB,
// fold and packing 0.32 ms (0.65 with two segments).
constexpr int kFoldSplits = 64;
__global__ __launch_bounds__(kThreads) void k_fold(const FoldD *__restrict__ folds, int n,
                                                   const long *__restrict__ base, long total) {
  typedef uint16_t u8v __attribute__((ext_vector_type(8)));
  __shared__ double t[32][33];
  __shared__ __attribute__((aligned(16))) uint16_t pos[kFoldSplits][2][32];
  __shared__ const double *hp[kFoldSplits];
  __shared__ int ls[kFoldSplits], ld[kFoldSplits], cnt;
  const int tid = threadIdx.x, c = tid & 31, r0 = tid >> 5;
  for (long L = blockIdx.x; L < total; L += gridDim.x) {
    const int m = find_unit(base, n, L);
    const FoldD &F = folds[m];
    long e = L - base[m], rb = (long)((sqrt(8.0 * (double)e + 1.0) - 1.0) * 0.5);
    while (rb * (rb + 1) / 2 > e) --rb;
    while ((rb + 1) * (rb + 2) / 2 <= e) ++rb;
    const long cb = e - rb * (rb + 1) / 2, NP = F.NP;
    double sa[4] = {}, sb[4] = {};
    const uint8_t *br = F.rbits + rb * F.nbytes, *bc = F.rbits + cb * F.nbytes;
    const long ns = (long)F.nchunks * F.nsplit, s1 = ns * (F.seg + 1) / F.nseg;
    for (long s0 = ns * F.seg / F.nseg; s0 < s1; s0 += kFoldSplits) {
      if (tid < kFoldSplits) {  // one wave
        const long s = s0 + tid;
        const int k = F.chunk0 + (int)(s / F.nsplit) * F.step, sl = (int)(s % F.nsplit);
        const long at = (long)k * F.bytes_c + sl / 8;
        const bool live = s < s1 && ((gld(br + at) & gld(bc + at)) >> (sl & 7) & 1);
        const unsigned long long lv = __ballot(live);
        const int q = __popcll(lv & ((1ull << tid) - 1ull));
        if (live) {
          const long S = (long)k * F.nsplit + sl;
          ls[q] = (int)S;
          ld[q] = split_ld(F.su_off[S + 1] - F.su_off[S]);
          hp[q] = F.Hc + F.ho[S];
        }
        if (tid == 0) cnt = __popcll(lv);
      }
      __syncthreads();
      const int nl = cnt;
      for (int i = tid; i < nl * 8; i += kThreads) {  // 16 bytes: 8 places
        const int q = i >> 3, h = (i >> 2) & 1, v = i & 3;
        *(u8v *)&pos[q][h][8 * v] = gld((const u8v *)(F.pos + ls[q] * NP + (h ? cb : rb) * 32 + 8 * v));
      }
      __syncthreads();
      for (int q0 = 0; q0 < nl; q0 += 4) {
        double va[4][4], vb[4][4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int q = min(q0 + u, nl - 1);
          const double *H = hp[q];
          const int pc = q0 + u < nl ? pos[q][1][c] : 0xffff, qc = q0 + u < nl ? pos[q][0][c] : 0xffff;
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            const int pr = pos[q][0][r0 + 8 * i], qr = pos[q][1][r0 + 8 * i];
            const bool ga = pr != 0xffff && pc != 0xffff, gb = qr != 0xffff && qc != 0xffff;
            const double x = gld(H + (ga ? (long)pr * ld[q] + pc : 0));
            const double y = gld(H + (gb ? (long)qr * ld[q] + qc : 0));
            va[u][i] = ga ? x : 0.0;
            vb[u][i] = gb ? y : 0.0;
          }
        }
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            sa[i] += va[u][i];
            sb[i] += vb[u][i];
          }
      }
      __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) t[r0 + 8 * i][c] = sb[i];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = r0 + 8 * i;
      double *o = F.out + (rb * 32 + r) * NP + cb * 32 + c;
      const double v = sa[i] + t[c][r];
      *o = F.acc ? *o + v : v;
    }
    __syncthreads();
  }
}

// item = 256 packed elements of one molecule (caller's function order):
// V = base + S at the functions' internal rows (S folded above, symmetric,
// read from its lower tiles, summed over its segments); then the molecule's
// state for the next incremental build: V_state = V.  Items from total on: 256
// elements of P_ref = P (the density operand's list), in the same launch.
__global__ __launch_bounds__(kThreads) void k_pack(const PackD *__restrict__ mols, int nm,
                                                   const long *__restrict__ base, long total,
                                                   const long *__restrict__ prep_base,
                                                   long prep_total) {
  for (long L = blockIdx.x; L < total + prep_total; L += gridDim.x) {
    if (L >= total) {
      const int m = find_unit(prep_base, nm, L - total);
      const PackD &M = mols[m];
      const long i = (L - total - prep_base[m]) * kThreads + threadIdx.x;
      if (i < M.NP * M.NP) M.Pref[i] = M.P[i];
      continue;
    }
    const int m = find_unit(base, nm, L);
    const PackD &M = mols[m];
    const long idx = (L - base[m]) * kThreads + threadIdx.x;
    const long n = M.n, NP = M.NP, npk = n * (n + 1) / 2;
    if (idx >= npk) continue;
    long j = (long)((sqrt(8.0 * (double)idx + 1.0) - 1.0) * 0.5);
    while (j * (j + 1) / 2 > idx) --j;
    while ((j + 1) * (j + 2) / 2 <= idx) ++j;
    const long k = idx - j * (j + 1) / 2;
    const long pj = M.fpos[j], pk = M.fpos[k];  // internal rows of caller functions j, k
    const long r = pj > pk ? pj : pk, c = pj > pk ? pk : pj;
    double v = 0.0;
#pragma unroll 4
    for (int s = 0; s < M.nseg; ++s) v += M.HS[((long)s * NP + r) * NP + c];
    const double out = M.incremental ? M.Vstate[idx] + v : v;
    M.Vout[idx] = out;
    M.Vstate[idx] = out;
  }
}

// Density operand of one molecule: D = P - P_ref (incremental) or P, in the
// contraction precision.  item = 256 elements.  The first workgroup also clears
// the plan's queue counters.
__global__ __launch_bounds__(kThreads) void k_prep(const PackD *__restrict__ mols, int nm,
                                                   const long *__restrict__ base, long total,
                                                   int mode, int *__restrict__ ctr, int nctr) {
  if (blockIdx.x == 0)
    for (int i = threadIdx.x; i < nctr; i += kThreads) ctr[i] = 0;
  for (long L = blockIdx.x; L < total; L += gridDim.x) {
    const int m = find_unit(base, nm, L);
    const PackD &M = mols[m];
    const long i = (L - base[m]) * kThreads + threadIdx.x;
    if (i >= (long)M.NP * M.NP) continue;
    const double d = M.incremental ? M.P[i] - M.Pref[i] : M.P[i];
    if (mode == 2) {  // split planes of D^T: element (r, c) goes to (c, r)
      const long np2 = M.NP * M.NP, r = i / M.NP, c = i % M.NP;
      __bf16 hi, lo;
      split_bf16((float)d, hi, lo);
      ((__bf16 *)M.D)[c * M.NP + r] = hi;
      ((__bf16 *)M.D)[np2 + c * M.NP + r] = lo;
    } else if (mode == 1) {
      ((float *)M.D)[i] = (float)d;
    } else {
      ((double *)M.D)[i] = d;
    }
  }
}

// ---------------------------------------------------------------- launches
static unsigned persistent_grid(long total, int per_cu) {
  const long cap = 256L * per_cu;
  return (unsigned)(total < cap ? (total > 0 ? total : 1) : cap);
}

// grid of a contraction launch: with queues, whole workgroups per queue
unsigned contraction_grid(const StageList &L, int per_cu) {
  long g = persistent_grid(L.total, per_cu);
  if (L.ctr) g = std::max<long>(kQueues, (g + kQueues - 1) / kQueues * kQueues);
  return (unsigned)g;
}

template <typename T, int LMAX>
static void basis_l(hipStream_t s, bool grad, const StageList &L) {
  dim3 g(persistent_grid(L.total, 8));
  if (grad)
    hipLaunchKernelGGL((k_basis<true, T, LMAX>), g, dim3(kThreads), 0, s, L.units, L.nu, L.base, L.order, L.total);
  else
    hipLaunchKernelGGL((k_basis<false, T, LMAX>), g, dim3(kThreads), 0, s, L.units, L.nu, L.base, L.order, L.total);
}

template <typename T, bool SPLIT, int LMAX>
static void wbasis_l(hipStream_t s, bool grad, bool two, const StageList &L) {
  dim3 g(persistent_grid(L.total, 8));
  auto k = grad ? (two ? k_wbasis<T, SPLIT, true, true, LMAX> : k_wbasis<T, SPLIT, true, false, LMAX>)
                : (two ? k_wbasis<T, SPLIT, false, true, LMAX> : k_wbasis<T, SPLIT, false, false, LMAX>);
  hipLaunchKernelGGL(k, g, dim3(kThreads), 0, s, L.units, L.nu, L.base, L.order, L.total);
}

template <typename T, bool SPLIT>
static void wbasis_t(hipStream_t s, bool grad, bool two, const StageList &L) {
  switch (L.lmax) {
    case 0: case 1: wbasis_l<T, SPLIT, 1>(s, grad, two, L); break;
    case 2: wbasis_l<T, SPLIT, 2>(s, grad, two, L); break;
    case 3: wbasis_l<T, SPLIT, 3>(s, grad, two, L); break;
    default: wbasis_l<T, SPLIT, 4>(s, grad, two, L); break;
  }
}

template <typename T>
void launch_wbasis(hipStream_t s, bool grad, bool split, bool two, const StageList &L) {
  if (!L.total) return;
  if constexpr (std::is_same<T, float>::value)
    if (split) {
      wbasis_t<T, true>(s, grad, two, L);
      return;
    }
  wbasis_t<T, false>(s, grad, two, L);
}

template <typename T>
void launch_basis(hipStream_t s, bool grad, const StageList &L) {
  if (!L.total) return;
  switch (L.lmax) {
    case 0: case 1: basis_l<T, 1>(s, grad, L); break;
    case 2: basis_l<T, 2>(s, grad, L); break;
    case 3: basis_l<T, 3>(s, grad, L); break;
    default: basis_l<T, 4>(s, grad, L); break;
  }
}

void launch_functional(hipStream_t s, bool gga, const StageList &L) {
  if (!L.total) return;
  dim3 g(persistent_grid(L.total, 8));
  if (gga)
    hipLaunchKernelGGL((k_functional<true>), g, dim3(kThreads), 0, s, L.units, L.nu, L.base, L.order, L.total);
  else
    hipLaunchKernelGGL((k_functional<false>), g, dim3(kThreads), 0, s, L.units, L.nu, L.base, L.order, L.total);
}

void launch_point_f(hipStream_t s, bool gga, bool spin, uint32_t mask, long Mc, long npad,
                    const double *st, const double *st2, double *fp) {
  const unsigned g = (unsigned)std::min<long>((Mc + kThreads - 1) / kThreads, 256L * 8);
  auto k = spin ? (gga ? k_point_f<true, true> : k_point_f<false, true>)
                : (gga ? k_point_f<true, false> : k_point_f<false, false>);
  hipLaunchKernelGGL(k, dim3(g), dim3(kThreads), 0, s, Mc, npad, mask, st, st2, fp);
}

void launch_energy(hipStream_t s, bool gga, bool spin, const StageList &L) {
  if (!L.total) return;
  dim3 g(persistent_grid(L.total, 8));
  auto k = spin ? (gga ? k_energy<true, true> : k_energy<false, true>)
                : (gga ? k_energy<true, false> : k_energy<false, false>);
  hipLaunchKernelGGL(k, g, dim3(kThreads), 0, s, L.units, L.nu, L.base, L.order, L.total);
}

void launch_functional_spin(hipStream_t s, bool gga, const StageList &L) {
  if (!L.total) return;
  dim3 g(persistent_grid(L.total, 8));
  if (gga)
    hipLaunchKernelGGL((k_functional_spin<true>), g, dim3(kThreads), 0, s, L.units, L.nu, L.base, L.order, L.total);
  else
    hipLaunchKernelGGL((k_functional_spin<false>), g, dim3(kThreads), 0, s, L.units, L.nu, L.base, L.order, L.total);
}

template <typename T>
void launch_wmat(hipStream_t s, bool grad, bool split, bool two, const StageList &L) {
  if (!L.total) return;
  dim3 g(persistent_grid(L.total, 8));
#define PGXC_WMAT(SPLIT)                                                                           \
  {                                                                                                \
    if (two) {                                                                                     \
      if (grad)                                                                                    \
        hipLaunchKernelGGL((k_wmat<T, true, SPLIT, true>), g, dim3(kThreads), 0, s, L.units, L.nu, \
                           L.base, L.order, L.total);                                              \
      else                                                                                         \
        hipLaunchKernelGGL((k_wmat<T, false, SPLIT, true>), g, dim3(kThreads), 0, s, L.units,     \
                           L.nu, L.base, L.order, L.total);                                        \
    } else if (grad) {                                                                             \
      hipLaunchKernelGGL((k_wmat<T, true, SPLIT, false>), g, dim3(kThreads), 0, s, L.units, L.nu,  \
                         L.base, L.order, L.total);                                                \
    } else {                                                                                       \
      hipLaunchKernelGGL((k_wmat<T, false, SPLIT, false>), g, dim3(kThreads), 0, s, L.units, L.nu, \
                         L.base, L.order, L.total);                                                \
    }                                                                                              \
  }
  if constexpr (std::is_same<T, float>::value) {
    if (split) {
      PGXC_WMAT(true)
      return;
    }
  }
  PGXC_WMAT(false)
#undef PGXC_WMAT
}

void launch_fold(hipStream_t s, const FoldD *folds, int n, const long *base, long total) {
  if (!total) return;
  hipLaunchKernelGGL(k_fold, dim3(persistent_grid(total, 8)), dim3(kThreads), 0, s, folds, n, base, total);
}

void launch_pack(hipStream_t s, const PackD *mols, int nm, const long *base, long total,
                 const long *prep_base, long prep_total) {
  if (!total) return;
  hipLaunchKernelGGL(k_pack, dim3(persistent_grid(total + prep_total, 8)), dim3(kThreads), 0, s, mols, nm, base,
                     total, prep_base, prep_total);
}

void launch_prep(hipStream_t s, const PackD *mols, int nm, const long *base, long total,
                 int mode, int *ctr, int nctr) {
  if (!total) return;
  hipLaunchKernelGGL(k_prep, dim3(persistent_grid(total, 8)), dim3(kThreads), 0, s, mols, nm, base,
                     total, mode, ctr, nctr);
}

#define PGXC_INST(T)                                                                  \
  template void launch_basis<T>(hipStream_t, bool, const StageList &);               \
  template void launch_wmat<T>(hipStream_t, bool, bool, bool, const StageList &);    \
  template void launch_wbasis<T>(hipStream_t, bool, bool, bool, const StageList &);
PGXC_INST(double)
PGXC_INST(float)
#undef PGXC_INST

// ---------------------------------------------------------------- screening
// item = one 128-point tile (four 32-point groups).  The smallest r^2 of each
// group to each atom (FP64, reduced over the group's 32 lanes), then per
// shell and group alpha_min r^2_min < cut-off marks the shell's runs of 8
// functions.  Outputs per group: the run flags (nw8 words, sig8); per tile:
// n_b, the functions of the shells marked on any of its groups, and those
// shells (smark, one bit per shell).
__global__ __launch_bounds__(kThreads) void k_screen(long ntiles, const double *__restrict__ gx,
                                                     const double *__restrict__ gy,
                                                     const double *__restrict__ gz, int n_atoms,
                                                     const AtomD *__restrict__ atoms, int n_shells,
                                                     const ScreenShell *__restrict__ shells,
                                                     int n8, int *nb, uint32_t *sig8,
                                                     uint32_t *smark) {
  constexpr int AC = 512;  // atoms per pass
  constexpr int W8 = kMaxRuns / 32;
  constexpr int WS = kMaxShells / 32;
  __shared__ double r2g[4][AC];
  __shared__ unsigned bits[4][W8];
  __shared__ unsigned sb[WS];
  __shared__ int nbs;
  const int tid = threadIdx.x;
  const int nw8 = (n8 + 31) / 32, nws = (n_shells + 31) / 32;
  for (long t = blockIdx.x; t < ntiles; t += gridDim.x) {
    for (int i = tid; i < 4 * W8; i += kThreads) (&bits[0][0])[i] = 0u;
    for (int i = tid; i < WS; i += kThreads) sb[i] = 0u;
    if (tid == 0) nbs = 0;
    const long p = t * kScreenTile + (tid & 127);
    const double x = gx[p], y = gy[p], z = gz[p];
    for (int a0 = 0; a0 < n_atoms; a0 += AC) {
      const int na = min(AC, n_atoms - a0);
      __syncthreads();
      // threads 0..127 take even atoms, 128..255 odd ones (whole waves each)
      for (int a = tid >> 7; a < na; a += 2) {
        const AtomD A = atoms[a0 + a];
        const double dx = x - A.x, dy = y - A.y, dz = z - A.z;
        double r2 = dx * dx + dy * dy + dz * dz;
#pragma unroll
        for (int off = 16; off >= 1; off >>= 1) r2 = fmin(r2, __shfl_xor(r2, off));
        if ((tid & 31) == 0) r2g[(tid & 127) >> 5][a] = r2;
      }
      __syncthreads();
      for (int si = tid; si < n_shells; si += kThreads) {
        const ScreenShell S = shells[si];
        if (S.atom < a0 || S.atom >= a0 + na) continue;
        bool any = false;
        const int b0 = S.func_off / kRun, b1 = (S.func_off + S.nfunc - 1) / kRun;
        for (int q = 0; q < 4; ++q) {
          if (S.amin * r2g[q][S.atom - a0] < kCutoff) {
            any = true;
            for (int b = b0; b <= b1; ++b) atomicOr(&bits[q][b >> 5], 1u << (b & 31));
          }
        }
        if (any) {
          atomicAdd(&nbs, S.nfunc);
          atomicOr(&sb[si >> 5], 1u << (si & 31));
        }
      }
    }
    __syncthreads();
    if (tid == 0) nb[t] = nbs;
    for (int i = tid; i < 4 * nw8; i += kThreads) {
      const int q = i / nw8, w = i % nw8;
      sig8[(t * 4 + q) * nw8 + w] = bits[q][w];
    }
    for (int i = tid; i < nws; i += kThreads) smark[t * nws + i] = sb[i];
    __syncthreads();
  }
}

void launch_screen(hipStream_t s, long ntiles_pts, const double *gx, const double *gy,
                   const double *gz, int n_atoms, const AtomD *atoms, int n_shells,
                   const ScreenShell *shells, int n8, int *nb, uint32_t *sig8, uint32_t *smark) {
  if (ntiles_pts <= 0) return;
  hipLaunchKernelGGL(k_screen, dim3(persistent_grid(ntiles_pts, 8)), dim3(kThreads), 0, s,
                     ntiles_pts, gx, gy, gz, n_atoms, atoms, n_shells, shells, n8, nb, sig8, smark);
}

// ------------------------------------------------------------ small kernels
// P = C diag(occ) C^T in the internal function order, one 64 x 64 tile (rb >=
// cb) and its mirror per workgroup, on FP64 MFMA: K = the orbitals, 16 a step,
// both operands staged [orbital][function] from C as the caller has it (finv:
// caller index of each internal function; rows from n on are 0, so the padding
// of P is written too).  A lane's four results are consecutive rows, so the
// mirror is written as 32 contiguous bytes.  Bound by latency at a few hundred
// functions; (H2O)32, 160 orbitals, 142 us (a dot product per element) -> 34; 4982 functions, 640
// orbitals 10.4 -> 0.61 ms.
constexpr int kFT = 64, kFK = 16, kFRow = kFT + 16;
__global__ __launch_bounds__(kThreads) void k_form_density(const double *__restrict__ C,
                                                           const double *__restrict__ occ,
                                                           const int *__restrict__ finv, int n,
                                                           int nocc, int NP, double *__restrict__ P) {
  __shared__ double as[2][kFK][kFRow], bs[2][kFK][kFRow];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  long rb = (long)((sqrt(8.0 * (double)blockIdx.x + 1.0) - 1.0) * 0.5);
  while (rb * (rb + 1) / 2 > (long)blockIdx.x) --rb;
  while ((rb + 1) * (rb + 2) / 2 <= (long)blockIdx.x) ++rb;
  const long cb = (long)blockIdx.x - rb * (rb + 1) / 2;
  // staging: a wave takes whole orbitals, a lane one function of each operand
  const long i = rb * kFT + lane, j = cb * kFT + lane;
  const int ri = i < n ? finv[i] : -1, rj = j < n ? finv[j] : -1;
  double ra[4], rc[4];
  auto load = [&](int k0) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int k = k0 + wave + 4 * e;
      const bool on = k < nocc;
      const double o = on ? occ[k] : 0.0;
      ra[e] = on && ri >= 0 ? o * C[ri + (long)k * n] : 0.0;
      rc[e] = on && rj >= 0 ? C[rj + (long)k * n] : 0.0;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      as[buf][wave + 4 * e][lane] = ra[e];
      bs[buf][wave + 4 * e][lane] = rc[e];
    }
  };
  d4 acc[2][2] = {};
  const int wm = 32 * (wave >> 1), wn = 32 * (wave & 1), l = lane & 15, kg = lane >> 4;
  const int lp = 4 * (l & 3) + (l >> 2);  // MFMA row l stands for this row of a block
  load(0);
  store(0);
  __syncthreads();
  for (int k0 = 0, buf = 0; k0 < nocc; k0 += kFK, buf ^= 1) {
    load(k0 + kFK);
#pragma unroll
    for (int k4 = 0; k4 < kFK; k4 += 4)
#pragma unroll
      for (int x = 0; x < 2; ++x)
#pragma unroll
        for (int y = 0; y < 2; ++y)
          acc[x][y] = MF<double>::mma(as[buf][k4 + kg][wm + 16 * x + lp], bs[buf][k4 + kg][wn + 16 * y + l], acc[x][y]);
    store(buf ^ 1);
    __syncthreads();
  }
#pragma unroll
  for (int x = 0; x < 2; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      const long r = rb * kFT + wm + 16 * x + 4 * kg, c = cb * kFT + wn + 16 * y + l;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        if (r + q < NP && c < NP) {
          P[(r + q) * NP + c] = acc[x][y][q];
          if (rb != cb) P[c * NP + r + q] = acc[x][y][q];
        }
    }
}

void launch_form_density(hipStream_t s, const double *C, const double *occ, const int *finv, int n,
                         int nocc, int NP, double *P) {
  const long nt = (NP + kFT - 1) / kFT;
  hipLaunchKernelGGL(k_form_density, dim3((unsigned)(nt * (nt + 1) / 2)), dim3(kThreads), 0, s, C, occ, finv, n,
                     nocc, NP, P);
}

// n doubles from src to dst, one of them pinned host memory: bound by the link
// (1 MiB to the host in 49 us, 21 GB/s; 2 KiB in 3 us).
__global__ __launch_bounds__(kThreads) void k_copy(const double *__restrict__ src, double *__restrict__ dst,
                                                   long n) {
  for (long i = (long)blockIdx.x * kThreads + threadIdx.x; i < n; i += (long)gridDim.x * kThreads) dst[i] = src[i];
}

void launch_copy(hipStream_t s, const double *src, double *dst, long n) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_copy, dim3((unsigned)std::min<long>(512, (n + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                     s, src, dst, n);
}

}  // namespace pgxc
