// fp32 implicit GEMM on the 16-bit matrix cores: the kernels for convolutions with a filter (tap-major and original weights).
#include "igemm_f3_kernel.hpp"

namespace onhip {

int f3_launch_tapc(const IgemmLaunch &cfg, const IgemmProblem &p, hipStream_t stream) {
    return p.res ? f3_launch_tile<BL_TAPC, true>(cfg, p, stream) : f3_launch_tile<BL_TAPC, false>(cfg, p, stream);
}
int f3_launch_gather(const IgemmLaunch &cfg, const IgemmProblem &p, hipStream_t stream) {
    return p.res ? f3_launch_tile<BL_GATHER, true>(cfg, p, stream) : f3_launch_tile<BL_GATHER, false>(cfg, p, stream);
}

}  // namespace onhip
