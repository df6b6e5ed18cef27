// FP64 instances of the contraction kernels.
#include "xc_contract.h"

namespace pgxc {
template void launch_density<double>(hipStream_t, bool, int, int, const StageList &);
template void launch_potential<double>(hipStream_t, int, int, const StageList &);
}  // namespace pgxc
