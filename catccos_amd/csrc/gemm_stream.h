// Shape of the weight-streaming GEMM kernels and what the host side needs to know of it.
#pragma once
#include <cstdint>

#include "gemm_common.h"

namespace cch {

constexpr int STREAM_TM = 32, STREAM_TN = 64;                  // rows of A and columns of B per tile
constexpr int STREAM_STAGE = (STREAM_TM + STREAM_TN) * 128;    // one chunk of A and B: each wave's piece of LDS
constexpr int STREAM_RUN = 4;                                  // consecutive tiles per XCD

// Workgroup b runs on XCD b % 8: tiles are dealt in runs of STREAM_RUN.
__host__ __device__ inline int stream_tile_of(int b) { return (b & ~(8 * STREAM_RUN - 1)) | ((b & 7) * STREAM_RUN) | ((b >> 3) & (STREAM_RUN - 1)); }
inline int64_t stream_grid(int64_t tiles) { return (tiles + 8 * STREAM_RUN - 1) / (8 * STREAM_RUN) * (8 * STREAM_RUN); }

}  // namespace cch
