// Instantiates the mid-size GEMM template: MXFP8 kernels (SwiGLU epilogue), B stored [K, N] and [N, K].
#include "gemm_mid_kernel.h"

namespace cch {
template int launch_mid_t<KIND_F8, EPI_SWIGLU, CCH_FMT_E4M3, 0>(const GemmProblem &, int, int, hipStream_t);
template int launch_mid_t<KIND_F8, EPI_SWIGLU, CCH_FMT_E4M3, 1>(const GemmProblem &, int, int, hipStream_t);
template int launch_mid_t<KIND_F8, EPI_SWIGLU, CCH_FMT_E5M2, 0>(const GemmProblem &, int, int, hipStream_t);
template int launch_mid_t<KIND_F8, EPI_SWIGLU, CCH_FMT_E5M2, 1>(const GemmProblem &, int, int, hipStream_t);
}  // namespace cch
