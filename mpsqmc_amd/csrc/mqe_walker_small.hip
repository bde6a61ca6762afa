// mqe_walker_small.hip -- the FP32 kernel of nearest-neighbour chains with bonds up to 16.
#include <hip/hip_runtime.h>

#include "mqe_kernels.h"
#include "mqe_tile16.h"

namespace mqe {
namespace t16 {

void launch_walker16(const WalkerLaunch &l, const Sys &S, const Pool &P, const float *TN, const float *TT, int flags) {
    hipLaunchKernelGGL(walker16_kernel, dim3(l.grid), dim3(64), 0, l.stream, S, P, TN, TT, flags);
}

}  // namespace t16
}  // namespace mqe
