// Routing sort in one workgroup, as a piece of a kernel: the sort's own launch up to 1024 rows (routing.hip) and the FFN's first one up to
// 8192 (moe_ffn.hip, beside the quantiser's workgroups) run it.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace cch {

// Lanes of the wave that hold the same key as this lane (keys below 2^bits; lanes with
// routed == false match nobody): one ballot per key bit.
__device__ __forceinline__ uint64_t same_key_lanes(int key, bool routed, int bits)
{
    uint64_t m = __ballot(routed);
    for (int b = 0; b < bits; b++) {
        const uint64_t set = __ballot(routed && ((key >> b) & 1));
        m &= ((key >> b) & 1) ? set : ~set;
    }
    return routed ? m : 0;
}

// Few rows and experts (a decode step's routes): the whole sort in one workgroup and one launch.  Sixteen waves
// walk their sixteenths of the rows in order, 64 at a time, exactly like the waves of the placement pass above;
// the per-wave counts per expert meet in LDS, thread e scans expert e's counts over the waves, the experts'
// totals are scanned across the workgroup, and a second walk over the rows (keys and lane sets kept in registers)
// hands the positions out.  No workspace.
//
// One CU does all of it, so what counts are chains of latencies and the stores' addresses: all keys of a wave are
// requested before the first is looked at, the totals are scanned inside waves (three barriers in all, where a scan over
// LDS took sixteen), and dst_to_src is put together in LDS and leaves in order (a wave's 64 scattered stores are 64 lines).
// Measured (before -> now): 24 and 384 routes 3.2 -> 2.4 us, 1024 over 64 experts 3.9 -> 2.8, 3072 5.3 -> 4.5, 8192 over 16 experts
// 9.4 -> 7.6, over 256 12.8 -> 10.6.
constexpr int ONE_WAVES = 16, ONE_MAX_GROUPS = 8, ONE_MAX_EXPERTS = 256;
constexpr int ONE_MAX_ROWS = ONE_WAVES * ONE_MAX_GROUPS * 64;   // 8192
template <int GROUPS>   // of 64 rows per wave
__device__ __forceinline__ void route_one_workgroup(const int32_t *__restrict__ expert_idx, int rows, int experts, int bits,
                                                    int32_t *__restrict__ dst_to_src, int32_t *__restrict__ src_to_dst,
                                                    int32_t *__restrict__ expert_tokens, int cumsum)
{
    __shared__ int32_t cnt[ONE_WAVES][ONE_MAX_EXPERTS];
    __shared__ int32_t sorted[ONE_WAVES * GROUPS * 64];
    __shared__ int32_t wave_total[ONE_MAX_EXPERTS / 64];
    __shared__ int32_t first[ONE_MAX_EXPERTS];   // sorted position of an expert's first row
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int base = w * GROUPS * 64;
    const uint64_t below = (1ull << lane) - 1ull;
    int key[GROUPS];
    uint64_t same[GROUPS];
#pragma unroll
    for (int g = 0; g < GROUPS; g++) {
        const int r = base + g * 64 + lane;
        key[g] = r < rows ? expert_idx[r] : -1;
    }
    // a wave's own counters: it alone touches them until the first barrier
    for (int e = lane; e < ONE_MAX_EXPERTS; e += 64) cnt[w][e] = 0;
#pragma unroll
    for (int g = 0; g < GROUPS; g++) {
        const int e = key[g];
        const bool routed = e >= 0 && e < experts;
        if (!routed) key[g] = -1;
        same[g] = same_key_lanes(e, routed, bits);
        if (routed && (same[g] & below) == 0) cnt[w][e] += __popcll(same[g]);   // first lane of its key
    }
    __syncthreads();
    // thread e: expert e's counts over the waves -> exclusive running sums; the totals scanned inside each wave
    int total = 0, incl = 0;
    if (w < ONE_MAX_EXPERTS / 64) {
        const int e = threadIdx.x;
#pragma unroll
        for (int v = 0; v < ONE_WAVES; v++) {
            const int c = cnt[v][e];
            cnt[v][e] = total;
            total += c;
        }
        incl = total;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int up = __shfl_up(incl, off, 64);
            if (lane >= off) incl += up;
        }
        if (lane == 63) wave_total[w] = incl;
        first[e] = incl - total;   // (within its 64 experts)
    }
    __syncthreads();
    int upto[ONE_MAX_EXPERTS / 64 + 1] = {0};
#pragma unroll
    for (int v = 0; v < ONE_MAX_EXPERTS / 64; v++) upto[v + 1] = upto[v] + wave_total[v];
    auto before = [&](int block) { return block == 0 ? upto[0] : block == 1 ? upto[1] : block == 2 ? upto[2] : upto[3]; };
    if ((int)threadIdx.x < experts) expert_tokens[threadIdx.x] = cumsum ? before(w) + incl : total;
    const int routed_rows = upto[ONE_MAX_EXPERTS / 64];
#pragma unroll
    for (int g = 0; g < GROUPS; g++) {
        const int r = base + g * 64 + lane;
        const bool routed = key[g] >= 0;
        int pos = -1;
        if (routed) pos = before(key[g] >> 6) + first[key[g]] + cnt[w][key[g]] + __popcll(same[g] & below);
        if (routed && (same[g] & below) == 0) cnt[w][key[g]] += __popcll(same[g]);
        if (r < rows) src_to_dst[r] = pos;
        if (pos >= 0) sorted[pos] = r;
    }
    __syncthreads();
    // (sorted positions past the routed rows hold no row)
    for (int i = threadIdx.x; i < rows; i += 64 * ONE_WAVES) dst_to_src[i] = i < routed_rows ? sorted[i] : -1;
}

inline bool route_fits_one_workgroup(int64_t rows, int num_experts) { return rows > 0 && rows <= ONE_MAX_ROWS && num_experts <= ONE_MAX_EXPERTS; }
inline int route_key_bits(int num_experts)
{
    int bits = 0;
    while ((1 << bits) < num_experts) bits++;
    return bits;
}

}  // namespace cch
