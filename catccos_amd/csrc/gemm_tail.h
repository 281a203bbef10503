// The last rows of some groups as a launch of their own.
//
// Grouped problems end with a partly filled round of 256 x 256 tiles: 304 tiles on 256 CUs take as long as 512 (MXFP8, 3072 rows over 16
// experts, K 7168, N 4096: 174 us; the same rows in 256 tiles 118 us, with the second launch 157).  Such a round exists because of short row tiles - the last
// rows of groups - and those are what the 256 x 256 kernel is worst at: a step of one takes 0.75 of a whole tile's time, however
// few rows it has.  So where the row tiles that make up the last round can all be short ones, the launch leaves them out and a
// second one of 64 x 128 tiles (gemm_mid_kernel.h, the same sums in the same order) computes those rows.
// Both launches work out which rows these are, from the group sizes that only the device has: the smallest remainders (rows of a
// group modulo 256, ties by group) that empty the last round, each at most TAIL_ROWS and all of them together at most one tile of the
// second kernel to a CU.  With two to a CU its steps take longer than the round it replaces: of 132 measured problems (1 to 2
// rounds, 16 to 64 steps of K) whose second launch had 257 to 512 tiles 110 were slower with it, by 10 % on average and up to 36 %; of
// 155 with at most 256 tiles 36 were slower and 85 faster, by 3 % on average and up to 19 %.
#pragma once
#include "gemm_device.h"

namespace cch {

// Above 192 rows a remainder is four row tiles of the second kernel, which take longer than the one they replace.
constexpr int TAIL_ROWS = 192;

// Rows of each group: lane l holds groups l, 64 + l, 128 + l, 192 + l.  The running row after group g is
// min(T, sum of the non-negative sizes so far): once the rows are used up every later group is empty, before
// that nothing is clipped (the reference's golden zero-pads the remainder,
// examples/utils/gen_data_fp4_mx_alltoallv_gmm.py:788-790).
struct GroupRows {
    static constexpr int NB = MAX_GROUPS / 64;
    int lo[NB], hi[NB];   // (no group: lo == hi)
    int used;             // rows that belong to groups
};
__device__ __forceinline__ GroupRows group_rows(const GemmProblem &p)
{
    const int lane = threadIdx.x & 63;
    GroupRows r;
    uint32_t sz[GroupRows::NB];
#pragma unroll
    for (int b = 0; b < GroupRows::NB; b++) {
        const int g = b * 64 + lane;
        sz[b] = 0;
        if (b * 64 < p.num_groups && g < p.num_groups) sz[b] = p.group_sizes ? (uint32_t)min(max(p.group_sizes[g], 0), p.T) : (uint32_t)p.T;
    }
    uint32_t before = 0;   // saturating sum of the sizes of the groups before this batch
#pragma unroll
    for (int b = 0; b < GroupRows::NB; b++) {
        r.lo[b] = r.hi[b] = 0;
        if (b * 64 < p.num_groups) {
            const uint32_t incl = sat_add(before, wave_scan_sat(sz[b]));
            // (the exclusive sum is the neighbour's inclusive one: incl - sz would be wrong once the sum has saturated)
            const uint32_t prev = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x138, 0xF, 0xF, false);   // wave_shr:1
            r.hi[b] = (int)min(incl, (uint32_t)p.T);
            r.lo[b] = (int)min(lane == 0 ? before : prev, (uint32_t)p.T);
            before = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        }
    }
    r.used = (int)min(before, (uint32_t)p.T);
    return r;
}

// A remainder's rank among the remainders: its rows, then its group.  0xFFFFFFFF: none that the second launch could take.
__device__ __forceinline__ uint32_t remainder_key(const GroupRows &r, int b)
{
    const int rem = (r.hi[b] - r.lo[b]) & (BM - 1);
    return rem > 0 && rem <= TAIL_ROWS ? (uint32_t)(rem * MAX_GROUPS + b * 64 + (int)(threadIdx.x & 63)) : 0xFFFFFFFFu;
}
__device__ __forceinline__ bool in_tail(const GroupRows &r, int b, uint32_t key) { return remainder_key(r, b) <= key; }

// The largest key that belongs to the second launch, 0 if it has nothing to do.
template <bool SWIGLU>
__device__ __forceinline__ uint32_t tail_key(const GemmProblem &p, const GroupRows &r)
{
    constexpr int NB = GroupRows::NB;
    const int n_tiles = (p.n_out + (SWIGLU ? 128 : 256) - 1) / (SWIGLU ? 128 : 256);   // column tiles of this kernel and
    const int n_mid = (p.n_out + (SWIGLU ? 64 : 128) - 1) / (SWIGLU ? 64 : 128);       // of the other
    int row_tiles = 0;
    uint32_t key[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) {
        key[b] = 0xFFFFFFFFu;
        if (b * 64 < p.num_groups) {
            row_tiles += __builtin_amdgcn_readlane((int)wave_scan_sat((uint32_t)((r.hi[b] - r.lo[b] + BM - 1) / BM)), 63);
            key[b] = remainder_key(r, b);
        }
    }
    const int64_t total = (int64_t)row_tiles * n_tiles;
    if (total < p.tail_cus) return 0;
    const int over = (int)(total % p.tail_cus), want = (over + n_tiles - 1) / n_tiles;   // row tiles that make up the last round
    auto up_to = [&](uint32_t k) {
        int n = 0;
#pragma unroll
        for (int b = 0; b < NB; b++)
            if (b * 64 < p.num_groups) n += __builtin_popcountll(__ballot(key[b] <= k));
        return n;
    };
    constexpr uint32_t LAST = TAIL_ROWS * MAX_GROUPS + MAX_GROUPS - 1;
    if (want == 0 || up_to(LAST) < want) return 0;
    uint32_t lo = 0, hi = LAST;   // up_to(lo) < want <= up_to(hi); all keys differ, so up_to(hi) == want in the end
    while (hi - lo > 1) {
        const uint32_t mid = (lo + hi) >> 1;
        if (up_to(mid) < want) lo = mid; else hi = mid;
    }
    int mid_rows = 0;   // row tiles of the other kernel
#pragma unroll
    for (int b = 0; b < NB; b++)
        if (b * 64 < p.num_groups) {
            const int rem = (r.hi[b] - r.lo[b]) & (BM - 1);
            mid_rows += __builtin_amdgcn_readlane((int)wave_scan_sat(key[b] <= hi ? (uint32_t)((rem + 63) / 64) : 0u), 63);
        }
    return (int64_t)mid_rows * n_mid <= TAIL_TILES ? hi : 0u;
}

}  // namespace cch
