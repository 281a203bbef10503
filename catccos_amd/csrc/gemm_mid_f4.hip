// Instantiates the mid-size GEMM template: MXFP4 kernels (plain and SwiGLU epilogues), B stored [K, N] and [N, K].
#include "gemm_mid_kernel.h"

namespace cch {
template int launch_mid_t<KIND_F4, EPI_PLAIN, CCH_FMT_E2M1, 0>(const GemmProblem &, int, int, hipStream_t);
template int launch_mid_t<KIND_F4, EPI_PLAIN, CCH_FMT_E2M1, 1>(const GemmProblem &, int, int, hipStream_t);
template int launch_mid_t<KIND_F4, EPI_SWIGLU, CCH_FMT_E2M1, 0>(const GemmProblem &, int, int, hipStream_t);
template int launch_mid_t<KIND_F4, EPI_SWIGLU, CCH_FMT_E2M1, 1>(const GemmProblem &, int, int, hipStream_t);
}  // namespace cch
