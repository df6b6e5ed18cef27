// FP32 instances of the contraction kernels.
#include "xc_contract.h"

namespace pgxc {
template void launch_density<float>(hipStream_t, bool, int, const StageList &);
template void launch_potential<float>(hipStream_t, int, int, const StageList &);
}  // namespace pgxc
