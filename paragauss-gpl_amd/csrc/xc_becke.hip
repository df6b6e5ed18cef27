// Becke partition weights for gfx950: the cell weights of a molecular grid's
// points, FP64, from a table of inverse centre distances.
#include "pgxc_internal.h"
#include "xc_device.h"

namespace pgxc {
// Becke partition weight of the owning atom (J. Chem. Phys. 88, 2547 (1988)),
// as becke0 (ParaGauss modules/grid_module.f90:2442-2497) with the step
// function mu3 = p(p(p(mu))), p(m) = m (3 - m^2) / 2
// (autodiff/becke_step_func.f90:84-124), no atomic-size adjustment.
// s(mu) = (1 - mu3) / 2, the halvings of the three steps left out and taken
// together at the end: powers of two, so the bits are those of the steps as
// written (10 FP64 operations a pair with the product instead of 16).
__device__ __forceinline__ double becke_s(double mu) {
  const double n1 = mu * (3.0 - mu * mu);       // 2 p(mu)
  const double n2 = n1 * (12.0 - n1 * n1);      // 16 p(p(mu))
  const double n3 = n2 * (768.0 - n2 * n2);     // 8192 p(p(p(mu)))
  return 0.5 - n3 * (1.0 / 16384.0);
}

// Every cell's product over all pairs of centres, one point per thread: for few
// centres (launch_becke), where the search for the near ones costs more than it
// leaves out.  A lone centre takes the whole weight at any point.
__global__ __launch_bounds__(kThreads) void k_becke_all(int na, const double *__restrict__ axyz,
                                                        const double *__restrict__ inv_dist,
                                                        long npts, long stride,
                                                        const double *__restrict__ pts,
                                                        const int *__restrict__ owner,
                                                        const double *__restrict__ wat,
                                                        double *__restrict__ wout) {
  const long p = (long)blockIdx.x * kThreads + threadIdx.x;
  if (p >= npts) return;
  const double x = pts[p], y = pts[stride + p], z = pts[2 * stride + p];
  const int own = owner[p];
  auto dist = [&](int i) {
    const double dx = axyz[3 * i] - x, dy = axyz[3 * i + 1] - y, dz = axyz[3 * i + 2] - z;
    return sqrt(dx * dx + dy * dy + dz * dz);
  };
  double sum = 0.0, pown = 0.0;
  for (int i = 0; i < na; ++i) {
    const double ri = dist(i);
    double pi = 1.0;
    for (int k = 0; k < na; ++k) {
      if (k == i) continue;
      pi *= becke_s((ri - dist(k)) * inv_dist[(long)i * na + k]);
    }
    sum += pi;
    if (i == own) pown = pi;
  }
  wout[p] = wat[p] * (pown / sum);
}

// One point per thread.  Written out, P_i = prod_k s(mu_ik) over all pairs is
// FP64 arithmetic on n^2 pairs a point, and almost all of the P_i are too small
// to change a bit of their sum: a centre far from the point has a factor of
// 1e-2 to 1e-10 with each centre near the point.  So the kNear nearest centres
// are found first, P of the nearest one is formed in full (it is at most the
// sum), and a centre whose product over just the kNear nearest ones is at or
// below 2^-64 of that (2^-54 over their number for more than 1024 centres) is left
// out of the sum, unless it owns the point: all of them together are below half
// an ulp of it.  The rest are formed in full, over
// the centres in order, kForm at a time so that a centre's distance is found
// once for all of them; a wave forms the centres any of its points needs.
// Bound by FP64 arithmetic.  (H2O)32, 96 centres, 1 961 792 points: 33 centres
// a wave are formed in full (14 for a single point), 5.0 ms in one launch; every
// product over all centres took 21.9 ms.  pgxc_becke_weights launches it per part
// of 2^18 points, 1024 workgroups, half of what the device holds: 7.3 ms in all,
// beside the transfers they overlap.
constexpr int kNear = 8, kForm = 8;

__global__ __launch_bounds__(kThreads) void k_becke(int na, const double *__restrict__ axyz,
                                                    const double *__restrict__ inv_dist,
                                                    long npts, long stride,
                                                    const double *__restrict__ pts,
                                                    const int *__restrict__ owner,
                                                    const double *__restrict__ wat,
                                                    double *__restrict__ wout) {
  const long p = (long)blockIdx.x * kThreads + threadIdx.x;
  if (p >= npts) return;
  const double x = pts[p], y = pts[stride + p], z = pts[2 * stride + p];
  const int own = owner[p];
  auto dist = [&](int i) {
    const double dx = axyz[3 * i] - x, dy = axyz[3 * i + 1] - y, dz = axyz[3 * i + 2] - z;
    return sqrt(dx * dx + dy * dy + dz * dz);
  };
  // the nearest centres, nearest first (a point without finite distances
  // keeps centre 0 and gets NaN products below)
  double rn[kNear];
  int in[kNear];
#pragma unroll
  for (int t = 0; t < kNear; ++t) {
    rn[t] = __builtin_inf();
    in[t] = 0;
  }
  for (int i = 0; i < na; ++i) {
    double v = dist(i);
    int id = i;
    if (!__any(v < rn[kNear - 1])) continue;
#pragma unroll
    for (int t = 0; t < kNear; ++t)
      if (v < rn[t]) {
        const double tv = rn[t];
        const int ti = in[t];
        rn[t] = v;
        in[t] = id;
        v = tv;
        id = ti;
      }
  }
  // here and below a centre's factor with itself is s(0) = 1/2: starts at 2
  double floor_p = 2.0 * becke_negligible(na);
#pragma unroll 2
  for (int k = 0; k < na; ++k) {
    floor_p *= becke_s((rn[0] - dist(k)) * inv_dist[(long)in[0] * na + k]);
  }
  double sum = 0.0, pown = 0.0;
  int b[kForm] = {}, nb = 0;  // the next centres to form, the last nb entries
  auto form = [&]() {
    double ri[kForm], pi[kForm];
#pragma unroll
    for (int m = 0; m < kForm; ++m) {
      ri[m] = dist(b[m]);
      pi[m] = 2.0;
    }
#pragma unroll 2
    for (int k = 0; k < na; ++k) {
      const double rk = dist(k);
#pragma unroll
      for (int m = 0; m < kForm; ++m) {
        pi[m] *= becke_s((ri[m] - rk) * inv_dist[(long)b[m] * na + k]);
      }
    }
#pragma unroll
    for (int m = 0; m < kForm; ++m)
      if (m >= kForm - nb) {
        sum += pi[m];
        if (b[m] == own) pown = pi[m];
      }
    nb = 0;
  };
  for (int i = 0; i < na; ++i) {
    const double ri = dist(i);
    // (a centre at another's position has NaN on the table's diagonal, so it
    // is formed in full)
    double pi = 2.0 + inv_dist[(long)i * na + i];
    bool need = true;
#pragma unroll
    for (int t = 0; t < kNear; ++t)
      if (need && t < na) {
        pi *= becke_s((ri - rn[t]) * inv_dist[(long)i * na + in[t]]);
        if (t == kNear / 2 - 1) need = __any(!(pi <= floor_p) || i == own);
      }
    if (!need || !__any(!(pi <= floor_p) || i == own)) continue;
#pragma unroll
    for (int m = 0; m + 1 < kForm; ++m) b[m] = b[m + 1];
    b[kForm - 1] = i;
    if (++nb == kForm) form();
  }
  if (nb) form();
  wout[p] = wat[p] * (pown / sum);
}

// Inverse distances of every pair of centres, inv[i][k] = 1/|R_i - R_k|, one
// thread per pair; the table k_becke reads.  On the diagonal 0, or NaN where
// another centre has the same position (whose pair of infinities k_becke may
// otherwise leave out).
__global__ __launch_bounds__(kThreads) void k_inv_dist(int na, const double *__restrict__ axyz,
                                                       double *__restrict__ inv) {
  const long q = (long)blockIdx.x * kThreads + threadIdx.x;
  if (q >= (long)na * na) return;
  const int i = (int)(q / na), k = (int)(q % na);
  double v = 0.0;
  if (i != k) {
    const double dx = axyz[3 * i] - axyz[3 * k], dy = axyz[3 * i + 1] - axyz[3 * k + 1],
                 dz = axyz[3 * i + 2] - axyz[3 * k + 2];
    v = 1.0 / sqrt(dx * dx + dy * dy + dz * dz);
  } else {
    for (int j = 0; j < na; ++j)
      if (j != i && axyz[3 * j] == axyz[3 * i] && axyz[3 * j + 1] == axyz[3 * i + 1] &&
          axyz[3 * j + 2] == axyz[3 * i + 2])
        v = __builtin_nan("");
  }
  inv[q] = v;
}

void launch_inv_dist(hipStream_t s, int na, const double *axyz, double *inv) {
  const long n = (long)na * na;
  hipLaunchKernelGGL(k_inv_dist, dim3((unsigned)((n + kThreads - 1) / kThreads)), dim3(kThreads), 0,
                     s, na, axyz, inv);
}

void launch_becke(hipStream_t s, int na, const double *axyz, const double *inv_dist, long npts,
                  long stride, const double *pts, const int *owner, const double *wat, double *wout) {
  hipLaunchKernelGGL(na <= kAllPairs ? k_becke_all : k_becke,
                     dim3((unsigned)((npts + kThreads - 1) / kThreads)), dim3(kThreads), 0, s, na, axyz, inv_dist,
                     npts, stride, pts, owner, wat, wout);
}
}  // namespace pgxc
