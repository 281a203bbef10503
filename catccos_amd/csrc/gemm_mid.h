// Shape of the mid-size GEMM kernels and the order of their tiles.
#pragma once
#include <algorithm>
#include <cstdint>

#include "gemm_common.h"

namespace cch {

// A tile has 64 * mb rows and 32 * jb * wn columns of B (2 x wn waves of 32 * mb x 32 * jb outputs).
constexpr int mid_cols(int wn, int jb) { return 32 * jb * wn; }
constexpr int mid_stage_bytes(int mb, int wn, int jb) { return (64 * mb + mid_cols(wn, jb)) * 128; }   // A and B panel of one step
constexpr int mid_stages(int mb, int wn) { return mb == 2 && wn == 2 ? 2 : 3; }           // of the ring: what two workgroups per CU (the wide tiles: one) leave room for
constexpr int mid_round(int cols) { return cols > 128 ? 256 : 512; }                      // workgroups that run at a time
constexpr int mid_run(int cols) { return cols > 128 ? 4 : 8; }                            // column tiles per block of a group's tiles
// MX: K-steps whose scales one 16-byte fetch per row holds (rows that can start 2 bytes past a dword leave room for the shift),
// and buffers of them: a group is requested S steps ahead, when the steps of the group it replaces must all have been read
constexpr int mid_steps_per_scales(int kind, int ua) { return kind == KIND_I8 ? 1 : (ua ? 2 : 4) / (kind == KIND_F4 ? 2 : 1); }
constexpr int mid_scale_buffers(int stages, int spg) { return 1 + (stages - 1 + spg - 1) / spg; }

// Tile of workgroup b when there are `total` tiles, -1 for none.  Workgroup b runs on XCD b % 8: of each round of tiles (the last
// one may be smaller) every XCD takes an equal run of consecutive ones.
__host__ __device__ inline int mid_tile_of(int b, int total, int round_size)
{
    const int round = b & ~(round_size - 1), in = b & (round_size - 1);
    const int n = total - round < round_size ? total - round : round_size;
    if (n <= 0) return -1;
    const int run = (n + 7) >> 3, pos = in >> 3, t = (in & 7) * run + pos;
    return pos < run && t < n ? round + t : -1;
}
// Workgroups to launch for at most `tiles` tiles: where fewer exist the runs of the last round are shorter, never longer.
inline int64_t mid_grid(int64_t tiles) { return (tiles + 7) / 8 * 8; }

}  // namespace cch
