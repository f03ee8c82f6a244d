// fp32 implicit GEMM on the 16-bit matrix cores: a convolution with at most 64 output channels and the 1x1 convolution after it in one
// launch (p.a_split and p.w2 in the split form).
#include "igemm_f3_kernel.hpp"

namespace onhip {

int f3_launch_pw(const IgemmProblem &p, dim3 grid, hipStream_t stream) {
    if (p.a_split_bytes >= (1LL << 31) || split_weights_bytes(p.m2, p.M) >= (1LL << 30) || !p.use_tapmask)
        return set_error(ONHIP_ERR_ARG, "conv + 1x1: not a problem of the kernel on the 16-bit matrix cores");
    if (p.res)
        hipLaunchKernelGGL((igemm_f3_kernel<BL_TAPC, 64, 64, 2, 2, true, true>), grid, dim3(THREADS), 0, stream, p);
    else
        hipLaunchKernelGGL((igemm_f3_kernel<BL_TAPC, 64, 64, 2, 2, false, true>), grid, dim3(THREADS), 0, stream, p);
    ONHIP_CHECK_HIP(hipGetLastError());
    return ONHIP_OK;
}

}  // namespace onhip
