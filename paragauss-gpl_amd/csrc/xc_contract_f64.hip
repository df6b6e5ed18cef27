// FP64 instances of the contraction kernels.
#include "xc_contract.h"

namespace pgxc {
template void launch_density<double>(hipStream_t, bool, int, const StageList &);
template void launch_potential<double>(hipStream_t, int, int, const StageList &);
void launch_xz(hipStream_t s, int var, const StageList &L, const double *P, double *XZ, int nplanes,
               int nspin, int spin) {
  launch_xz_impl(s, var, L, P, XZ, nplanes, nspin, spin);
}
}  // namespace pgxc
