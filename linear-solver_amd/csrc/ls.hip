// ls.hip -- the stand-alone m x m least-squares solves on the device (one
// wavefront each; see ls_body.h).
#include "ls_body.h"

namespace aar {

template <int M>
__global__ __launch_bounds__(64) void ls_kernel(Ctrl *c, int n, int flags)
{
    __shared__ LsLds<M> L;
    if (c->done) return;
    ls_from_ctrl<M>(L, c, n, flags);
}

hipError_t launch_ls(Ctrl *ctrl, int n, int flags, hipStream_t st)
{
    if (n < 1 || n > MAXM_LS) return hipErrorInvalidValue;
    if (n <= 8) hipLaunchKernelGGL((ls_kernel<8>), dim3(1), dim3(64), 0, st, ctrl, n, flags);
    else if (n <= 16) hipLaunchKernelGGL((ls_kernel<16>), dim3(1), dim3(64), 0, st, ctrl, n, flags);
    else hipLaunchKernelGGL((ls_kernel<32>), dim3(1), dim3(64), 0, st, ctrl, n, flags);
    return hipGetLastError();
}

}  // namespace aar
