// mqe_walker_f64.hip -- the general walker kernel, FP64, bonds above 64.
#include <hip/hip_runtime.h>

#include "mqe_general.h"

namespace mqe {

void launch_walker_f64(const WalkerLaunch &l, const Sys &S, const Pool &P, const double *trial, int flags) {
    hipLaunchKernelGGL((walker_kernel<double, false>), dim3(l.grid), dim3(MQE_NT), l.lds, l.stream, S, P, trial, flags);
}

hipError_t lds_attr_f64(size_t lds) {
    return hipFuncSetAttribute((const void *)walker_kernel<double, false>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds);
}

}  // namespace mqe
