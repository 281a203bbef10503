// Instantiates the weight-streaming GEMM template: int8 kernels (dequant and dequant + SwiGLU epilogues), B stored [K, N] and [N, K].
#include "gemm_stream_kernel.h"

namespace cch {
template int launch_stream_t<KIND_I8, EPI_DEQUANT, 0, 0>(const GemmProblem &, int, hipStream_t);
template int launch_stream_t<KIND_I8, EPI_DEQUANT, 0, 1>(const GemmProblem &, int, hipStream_t);
template int launch_stream_t<KIND_I8, EPI_DEQUANT_SWIGLU, 0, 0>(const GemmProblem &, int, hipStream_t);
template int launch_stream_t<KIND_I8, EPI_DEQUANT_SWIGLU, 0, 1>(const GemmProblem &, int, hipStream_t);
}  // namespace cch
