// mqe_walker_tile.hip -- the FP32 tile kernel of nearest-neighbour chains.
#include <hip/hip_runtime.h>

#include "mqe_kernels.h"
#include "mqe_tile32.h"

namespace mqe {
namespace t32 {

void launch_walker32(const WalkerLaunch &l, const Sys &S, const Pool &P, const float *TN, const float *TT, int flags,
                     bool learn) {
    if (learn)
        hipLaunchKernelGGL(walker32_kernel<true>, dim3(l.grid), dim3(MQE_NT), lds_bytes(), l.stream, S, P, TN, TT,
                           flags);
    else
        hipLaunchKernelGGL(walker32_kernel<false>, dim3(l.grid), dim3(MQE_NT), lds_bytes(), l.stream, S, P, TN, TT,
                           flags);
}

hipError_t lds_attr32() {
    const hipError_t r = hipFuncSetAttribute((const void *)walker32_kernel<false>,
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds_bytes());
    if (r != hipSuccess) return r;
    return hipFuncSetAttribute((const void *)walker32_kernel<true>, hipFuncAttributeMaxDynamicSharedMemorySize,
                               (int)lds_bytes());
}

}  // namespace t32
}  // namespace mqe
