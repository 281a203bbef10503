// MoE routing: stable sort of the flat (token, route) list by expert.  Produces both directions of
// the permutation and the tokens per expert, which is what the gather + dynamic quantisation
// (dyn_quant.hip), the grouped matmul (group sizes) and the un-permute (unpermute.hip) consume.
//
// Follows the sort stage of moe_init_routing_quant_v2
// (examples/aux_ops/moe_init_routing_quant_v2/moe_init_routing_quant_v2.h:70-110: sort by expert,
// MoeV2SrcToDstOp inverts the permutation, MoeV2ExpertTokenOut counts) and its CPU stand-in
// (examples/utils/gen_data_moe.py:48-57: torch.argsort(stable=True) + bincount).  Keys are small
// integers, so the sort is a counting sort: per-chunk histograms, and a placement pass in which four waves
// walk their quarters of a chunk in order.  Between the two stands a scan over (expert, chunk), in a launch of its own where the
// chunks are very many; otherwise every workgroup of the placement pass adds up what it needs.  Up to 32768 rows and 256 experts the sort is one launch.
#include <algorithm>
#include <atomic>

#include "common.h"
#include "route_keys.h"

namespace cch {

constexpr int ROUTE_CHUNK = 1024;       // rows per workgroup
constexpr int ROUTE_MAX_EXPERTS = 1024;
// cch_set_option("routing_three_launches", 1): the general path also where one launch would do (for tests)
std::atomic<int> g_route_three_launches{0};

// hist[e * nchunks + c] (BY_CHUNK: hist[c * experts + e]) = rows of chunk c routed to expert e; dst_to_src of the chunk's positions
// is preset to -1 (positions past the routed rows keep it).
template <bool BY_CHUNK>
__global__ __launch_bounds__(256) void route_histogram_kernel(const int32_t *__restrict__ expert_idx, int rows, int experts,
                                                              int nchunks, int32_t *__restrict__ hist,
                                                              int32_t *__restrict__ dst_to_src)
{
    __shared__ int32_t h[ROUTE_MAX_EXPERTS];
    for (int e = threadIdx.x; e < experts; e += 256) h[e] = 0;
    __syncthreads();
    const int base = blockIdx.x * ROUTE_CHUNK;
    for (int i = threadIdx.x; i < ROUTE_CHUNK; i += 256) {
        const int r = base + i;
        if (r < rows) {
            const int e = expert_idx[r];
            if (e >= 0 && e < experts) atomicAdd(&h[e], 1);
            dst_to_src[r] = -1;
        }
    }
    __syncthreads();
    for (int e = threadIdx.x; e < experts; e += 256) hist[BY_CHUNK ? (size_t)blockIdx.x * experts + e : (size_t)e * nchunks + blockIdx.x] = h[e];
}

// In-place exclusive scan of hist in (expert, chunk) order: hist[e * nchunks + c] becomes the first
// sorted position of expert e's rows of chunk c.  One workgroup of 16 waves: a wave sums the
// (contiguous) row of an expert, the per-expert totals are scanned across the workgroup, and the
// wave then scans its rows 64 chunks at a time from the expert's start.  Also writes the
// per-expert token counts (or their running sum).
__global__ __launch_bounds__(1024) void route_scan_kernel(int32_t *__restrict__ hist, int experts, int nchunks,
                                                          int32_t *__restrict__ expert_tokens, int cumsum)
{
    __shared__ int32_t part[1024];   // per-expert totals, then their inclusive scan (experts <= 1024)
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    part[threadIdx.x] = 0;
    __syncthreads();
    for (int e = wave; e < experts; e += 16) {
        int sum = 0;
        for (int c = lane; c < nchunks; c += 64) sum += hist[(size_t)e * nchunks + c];
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) sum += __shfl_xor(sum, off, 64);
        if (lane == 0) part[e] = sum;
    }
    __syncthreads();
    const int own = part[threadIdx.x];
    // Hillis-Steele inclusive scan over the 1024 totals
    for (int off = 1; off < 1024; off <<= 1) {
        const int add = threadIdx.x >= off ? part[threadIdx.x - off] : 0;
        __syncthreads();
        part[threadIdx.x] += add;
        __syncthreads();
    }
    if ((int)threadIdx.x < experts) expert_tokens[threadIdx.x] = cumsum ? part[threadIdx.x] : own;
    for (int e = wave; e < experts; e += 16) {
        int run = e > 0 ? part[e - 1] : 0;   // first position of expert e
        for (int c0 = 0; c0 < nchunks; c0 += 64) {
            const int c = c0 + lane;
            const int v = c < nchunks ? hist[(size_t)e * nchunks + c] : 0;
            int incl = v;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const int up = __shfl_up(incl, off, 64);
                if (lane >= off) incl += up;
            }
            if (c < nchunks) hist[(size_t)e * nchunks + c] = run + incl - v;
            run += __shfl(incl, 63, 64);
        }
    }
}

// Four waves per chunk, 256 consecutive rows each, 64 at a time.  Inside a group of 64 the rank
// of a row among the rows of the same expert is a population count over the lanes that hold the
// same key; a wave first counts its rows per expert, the counts of the waves before it (and the
// chunk's scanned start) give its first position per expert, and a second walk over the same
// rows hands the positions out in order.  A wave's LDS accesses execute in program order, so
// "all lanes read the counter, then the first lane of each key moves it on" needs no barrier.
//
// SCANNED: hist holds first positions (route_scan_kernel).  Otherwise it holds the counts by chunk, and the workgroup sums each expert's
// counts over all chunks and over the chunks before its own; workgroup 0 writes the tokens per expert.
constexpr int ROUTE_WAVES = 4;
constexpr int ROUTE_GROUPS = ROUTE_CHUNK / 64 / ROUTE_WAVES;   // groups of 64 rows per wave
template <bool SCANNED>
__global__ __launch_bounds__(64 * ROUTE_WAVES) void route_place_kernel(const int32_t *__restrict__ expert_idx, int rows, int experts,
                                                                      int nchunks, int bits, const int32_t *__restrict__ hist,
                                                                      int32_t *__restrict__ dst_to_src,
                                                                      int32_t *__restrict__ src_to_dst,
                                                                      int32_t *__restrict__ expert_tokens, int cumsum)
{
    constexpr int THREADS = 64 * ROUTE_WAVES, MAX_E = ROUTE_MAX_EXPERTS;
    __shared__ int32_t cnt[ROUTE_WAVES][MAX_E];
    __shared__ int32_t total[SCANNED ? 1 : MAX_E], before[SCANNED ? 1 : MAX_E], wave_total[ROUTE_WAVES];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    for (int e = threadIdx.x; e < (SCANNED ? experts : MAX_E); e += THREADS) {
#pragma unroll
        for (int v = 0; v < ROUTE_WAVES; v++) cnt[v][e] = 0;
        if constexpr (!SCANNED) total[e] = before[e] = 0;
    }
    __syncthreads();
    if constexpr (!SCANNED) {
        // thread t: expert t % span (and those THREADS further on), every parts-th chunk
        const int span = min(1 << bits, THREADS), parts = THREADS / span, part = threadIdx.x / span;
        for (int e = threadIdx.x % span; e < experts; e += span) {
            int all = 0, mine = 0;
#pragma unroll 8
            for (int c = part; c < nchunks; c += parts) {
                const int v = hist[(size_t)c * experts + e];
                all += v;
                mine += c < (int)blockIdx.x ? v : 0;
            }
            atomicAdd(&total[e], all);
            atomicAdd(&before[e], mine);
        }
    }
    const int base = blockIdx.x * ROUTE_CHUNK + w * (ROUTE_GROUPS * 64);
    const uint64_t below = (1ull << lane) - 1ull;
    int key[ROUTE_GROUPS];
    uint64_t same[ROUTE_GROUPS];
#pragma unroll
    for (int g = 0; g < ROUTE_GROUPS; g++) {
        const int r = base + g * 64 + lane;
        const int e = r < rows ? expert_idx[r] : -1;
        const bool routed = e >= 0 && e < experts;
        key[g] = routed ? e : -1;
        same[g] = same_key_lanes(e, routed, bits);
        if (routed && (same[g] & below) == 0) cnt[w][e] += __popcll(same[g]);   // first lane of its key
    }
    __syncthreads();
    if constexpr (!SCANNED) {
        // thread t holds experts 4 t .. 4 t + 3: the totals before each of them, inside the wave and then over the waves
        constexpr int PER = MAX_E / THREADS;
        int sum = 0, own[PER];
#pragma unroll
        for (int i = 0; i < PER; i++) sum += own[i] = total[threadIdx.x * PER + i];
        int incl = sum;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int up = __shfl_up(incl, off, 64);
            if (lane >= off) incl += up;
        }
        if (lane == 63) wave_total[w] = incl;
        __syncthreads();
        int run = incl - sum;
        for (int v = 0; v < w; v++) run += wave_total[v];
#pragma unroll
        for (int i = 0; i < PER; i++) {
            const int e = threadIdx.x * PER + i;
            before[e] += run;
            run += own[i];
            if (blockIdx.x == 0 && e < experts) expert_tokens[e] = cumsum ? run : own[i];
        }
        __syncthreads();
    }
    // counts -> first positions: the chunk's start per expert, then the waves in order
    for (int e = threadIdx.x; e < experts; e += 64 * ROUTE_WAVES) {
        int run = SCANNED ? hist[(size_t)e * nchunks + blockIdx.x] : before[e];
#pragma unroll
        for (int v = 0; v < ROUTE_WAVES; v++) {
            const int c = cnt[v][e];
            cnt[v][e] = run;
            run += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int g = 0; g < ROUTE_GROUPS; g++) {
        const int r = base + g * 64 + lane;
        const bool routed = key[g] >= 0;
        int pos = -1;
        if (routed) pos = cnt[w][key[g]] + __popcll(same[g] & below);
        if (routed && (same[g] & below) == 0) cnt[w][key[g]] += __popcll(same[g]);
        if (r < rows) {
            src_to_dst[r] = pos;
            if (pos >= 0) dst_to_src[pos] = r;
        }
    }
}

// Up to 1024 rows (a decode step's routes): the whole sort in one workgroup.  Sixteen waves hold a row per lane, exactly like
// the waves of the placement pass above; the per-wave counts per expert meet in LDS, thread e scans expert e's counts over the waves,
// the experts' totals are scanned across the workgroup, and every lane finds its position.  No workspace.
//
// What counts here are chains of latencies and the stores' addresses: all keys are requested before anything is looked at, the totals are
// scanned inside waves (three barriers in all, where a scan over LDS took sixteen), and dst_to_src is put together in LDS and leaves in
// order (a wave's 64 scattered stores are 64 lines).  Measured (before -> now): 24 and 384 routes 3.2 -> 2.4 us, 1024 over 64 experts 3.9 -> 2.8.
constexpr int ONE_WAVES = 16, ONE_MAX_EXPERTS = 256;
__global__ __launch_bounds__(64 * ONE_WAVES) void route_one_workgroup_kernel(const int32_t *__restrict__ expert_idx, int rows, int experts,
                                                                            int bits, int32_t *__restrict__ dst_to_src,
                                                                            int32_t *__restrict__ src_to_dst,
                                                                            int32_t *__restrict__ expert_tokens, int cumsum)
{
    __shared__ int32_t cnt[ONE_WAVES][ONE_MAX_EXPERTS];
    __shared__ int32_t sorted[ONE_WAVES * 64];
    __shared__ int32_t wave_total[ONE_MAX_EXPERTS / 64];
    __shared__ int32_t first[ONE_MAX_EXPERTS];   // sorted position of an expert's first row
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, r = threadIdx.x;
    const uint64_t below = (1ull << lane) - 1ull;
    int key = r < rows ? expert_idx[r] : -1;
    // a wave's own counters: it alone touches them until the first barrier
    for (int e = lane; e < ONE_MAX_EXPERTS; e += 64) cnt[w][e] = 0;
    if (key >= experts) key = -1;
    const uint64_t same = same_key_lanes(key, key >= 0, bits);
    if (key >= 0 && (same & below) == 0) cnt[w][key] = __popcll(same);   // first lane of its key
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
    const int pos = key >= 0 ? before(key >> 6) + first[key] + cnt[w][key] + __popcll(same & below) : -1;
    if (r < rows) src_to_dst[r] = pos;
    if (pos >= 0) sorted[pos] = r;
    __syncthreads();
    // (sorted positions past the routed rows hold no row)
    if (r < rows) dst_to_src[r] = r < routed_rows ? sorted[r] : -1;
}

// 1025 to 32768 rows, of which every workgroup places 1024, still in one launch and without memory of its own: each counts all rows (their keys come
// from the L2), for its expert totals and for the rows in front of its own, so no workgroup waits for another.  In one workgroup the sort is
// bound by the ballots that find a row's rank, 40 cycles per key bit and 64 rows; here a workgroup ranks its own rows only and counts the rest with
// LDS atomics.  Measured against one workgroup (graph replays, us, 16 / 256 experts): 2048 rows 3.8 / 4.5 -> 3.6 / 4.1, 4096 5.1 / 6.5 -> 3.8 / 4.4, 8192
// 8.0 / 10.9 -> 4.2 / 5.0; against the two launches below: 8200 7.5 / 9.1 -> 4.8 / 5.5, 16384 7.5 / 9.2 -> 5.1 / 5.8, 32768 7.9 / 10.1 -> 6.7 / 7.5.  (All rows
// counted by ballots: 8192 rows 6.5 / 9.1.)
constexpr int GROUPS_MAX_ROWS = 32 * 64 * ONE_WAVES;   // 32768: the counts of two halves share a register
template <int GROUPS>   // of 1024 rows, one to a workgroup
__global__ __launch_bounds__(64 * ONE_WAVES) void route_groups_kernel(const int32_t *__restrict__ expert_idx, int rows, int experts, int bits,
                                                                     int32_t *__restrict__ dst_to_src, int32_t *__restrict__ src_to_dst,
                                                                     int32_t *__restrict__ expert_tokens, int cumsum)
{
    __shared__ int32_t own[ONE_WAVES][ONE_MAX_EXPERTS];   // rows of this workgroup by wave, then their first positions
    // all rows of every sixteenth lane by expert; in the upper half those in front of this workgroup (31744 at most).  Lanes of one wave that hold
    // one expert meet at four to an address, and a seventeenth counter keeps experts on different banks.
    constexpr int COPIES = 16, PITCH = COPIES + 1;
    __shared__ int32_t all[ONE_MAX_EXPERTS * PITCH];
    __shared__ int32_t wave_total[ONE_MAX_EXPERTS / 64];
    __shared__ int32_t first[ONE_MAX_EXPERTS];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, group = blockIdx.x;
    const uint64_t below = (1ull << lane) - 1ull;
    int key[GROUPS], my_key = -1;
#pragma unroll
    for (int g = 0; g < GROUPS; g++) {
        const int r = g * 64 * ONE_WAVES + (int)threadIdx.x;
        key[g] = r < rows ? expert_idx[r] : -1;
    }
    for (int e = lane; e < ONE_MAX_EXPERTS; e += 64) own[w][e] = 0;   // (the wave's own until the second barrier)
    for (int i = threadIdx.x; i < experts * PITCH; i += 64 * ONE_WAVES) all[i] = 0;
    __syncthreads();
#pragma unroll
    for (int g = 0; g < GROUPS; g++) {
        const bool routed = key[g] >= 0 && key[g] < experts;
        if (routed) atomicAdd(&all[key[g] * PITCH + lane % COPIES], g < group ? 0x10001 : 1);
        if (g == group) my_key = routed ? key[g] : -1;
    }
    const uint64_t my_same = same_key_lanes(my_key, my_key >= 0, bits);
    if (my_key >= 0 && (my_same & below) == 0) own[w][my_key] = __popcll(my_same);   // first lane of its key
    __syncthreads();
    // thread e: expert e's totals, scanned inside each wave, and the first positions of this workgroup's waves
    int total = 0, incl = 0;
    if (w < ONE_MAX_EXPERTS / 64) {
        const int e = threadIdx.x;
        int sum = 0;
#pragma unroll
        for (int v = 0; v < COPIES; v++) sum += e < experts ? all[e * PITCH + v] : 0;
        total = sum & 0xFFFF;
        int run = sum >> 16;
#pragma unroll
        for (int v = 0; v < ONE_WAVES; v++) {
            const int c = own[v][e];
            own[v][e] = run;
            run += c;
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
    if (group == 0 && (int)threadIdx.x < experts) expert_tokens[threadIdx.x] = cumsum ? before(w) + incl : total;
    const int r = group * 64 * ONE_WAVES + (int)threadIdx.x;
    if (r >= rows) return;
    const int pos = my_key >= 0 ? before(my_key >> 6) + first[my_key] + own[w][my_key] + __popcll(my_same & below) : -1;
    src_to_dst[r] = pos;
    if (pos >= 0) dst_to_src[pos] = r;
    if (r >= upto[ONE_MAX_EXPERTS / 64]) dst_to_src[r] = -1;   // (sorted positions past the routed rows hold no row)
}

// Checks shared by the two entry points; fills nchunks.
static int route_check(const char *who, const int32_t *expert_idx, int64_t rows, int num_experts, const int32_t *dst_to_src,
                       const int32_t *src_to_dst, const int32_t *expert_tokens, int64_t *nchunks)
{
    CCH_REQUIRE(rows >= 0 && rows < ((int64_t)1 << 30), "%s: rows=%lld", who, (long long)rows);
    CCH_REQUIRE(num_experts >= 1 && num_experts <= ROUTE_MAX_EXPERTS, "%s: num_experts=%d outside 1..%d", who, num_experts,
                ROUTE_MAX_EXPERTS);
    CCH_REQUIRE(expert_tokens != nullptr, "%s: null expert_tokens", who);
    *nchunks = std::max<int64_t>((rows + ROUTE_CHUNK - 1) / ROUTE_CHUNK, 1);
    CCH_REQUIRE(*nchunks * num_experts < ((int64_t)1 << 31), "%s: rows x experts too large", who);
    CCH_REQUIRE(rows == 0 || (expert_idx && dst_to_src && src_to_dst), "%s: null pointer", who);
    return CCH_OK;
}

// hist holds nchunks * num_experts entries, every one of which the histogram pass writes before it is read (nothing has to start at zero).
// Two launches or three: the placement's sums grow with chunks x chunks x experts, the scan's with chunks x experts on one CU.  Three -> two
// (graph replays, us): 32768 routes over 256 experts 26.7 -> 10.0, 131072 over 256 37.5 -> 15.1, 50000 over 1024 75 -> 20, 1048576 (1024 chunks)
// over 16 24.7 -> 15.5, over 256 194 -> 83; but 4096 chunks over 16 67 -> 78.
constexpr int64_t ROUTE_SUM_CHUNKS = 1024;
static int route_launch(const int32_t *expert_idx, int64_t rows, int num_experts, int64_t nchunks, int32_t *dst_to_src,
                        int32_t *src_to_dst, int32_t *expert_tokens, int cumsum, int32_t *hist, hipStream_t s)
{
    if (rows > 0 && rows <= GROUPS_MAX_ROWS && num_experts <= ONE_MAX_EXPERTS && !g_route_three_launches.load(std::memory_order_relaxed)) {
        const int bits = route_key_bits(num_experts), groups = (int)((rows + 64 * ONE_WAVES - 1) / (64 * ONE_WAVES));
        auto kern = groups <= 1 ? route_one_workgroup_kernel : groups <= 2 ? route_groups_kernel<2> : groups <= 4 ? route_groups_kernel<4>
                          : groups <= 8 ? route_groups_kernel<8> : groups <= 16 ? route_groups_kernel<16> : route_groups_kernel<32>;
        hipLaunchKernelGGL(kern, dim3((unsigned)groups), dim3(64 * ONE_WAVES), 0, s, expert_idx, (int)rows, num_experts, bits, dst_to_src, src_to_dst,
                           expert_tokens, cumsum);
        return launch_status("route kernel");
    }
    const int bits = route_key_bits(num_experts);
    const bool sums = rows > 0 && nchunks <= ROUTE_SUM_CHUNKS && !g_route_three_launches.load(std::memory_order_relaxed);
    hipLaunchKernelGGL(sums ? route_histogram_kernel<true> : route_histogram_kernel<false>, dim3((unsigned)nchunks), dim3(256), 0, s, expert_idx,
                       (int)rows, num_experts, (int)nchunks, hist, dst_to_src);
    if (!sums)
        hipLaunchKernelGGL(route_scan_kernel, dim3(1), dim3(1024), 0, s, hist, num_experts, (int)nchunks, expert_tokens, cumsum);
    if (rows > 0)
        hipLaunchKernelGGL(sums ? route_place_kernel<false> : route_place_kernel<true>, dim3((unsigned)nchunks), dim3(64 * ROUTE_WAVES), 0, s,
                           expert_idx, (int)rows, num_experts, (int)nchunks, bits, hist, dst_to_src, src_to_dst, expert_tokens, cumsum);
    return launch_status("route kernels");
}

// Histogram area of cch_moe_init_routing_noalloc: part of the library's device image, so every GPU
// the library runs on holds its own copy (1 MiB) from load to process end.  The name is only a
// host-side handle; the device address is looked up once per device and kept in g_scratch_ptr.
constexpr int64_t ROUTE_STATIC_ENTRIES = CCH_ROUTING_NOALLOC_MAX_ENTRIES;
static __device__ __align__(256) int32_t scratch[ROUTE_STATIC_ENTRIES];
constexpr int ROUTE_MAX_DEVICES = 64;
static std::atomic<int32_t *> g_scratch_ptr[ROUTE_MAX_DEVICES];

// Device address of `scratch` on the current device (looked up on first use, or by cch_init).
int routing_scratch_setup(int32_t **out)
{
    int dev = 0;
    CCH_HIP(hipGetDevice(&dev));
    CCH_REQUIRE(dev >= 0 && dev < ROUTE_MAX_DEVICES, "routing scratch: device %d outside 0..%d", dev, ROUTE_MAX_DEVICES - 1);
    int32_t *ptr = g_scratch_ptr[dev].load(std::memory_order_acquire);
    if (ptr == nullptr) {
        void *sym = nullptr;
        CCH_HIP(hipGetSymbolAddress(&sym, HIP_SYMBOL(scratch)));
        if (sym == nullptr) return fail(CCH_EHIP, "routing scratch: hipGetSymbolAddress gave a null address on device %d", dev);
        ptr = static_cast<int32_t *>(sym);
        g_scratch_ptr[dev].store(ptr, std::memory_order_release);   // two threads racing here store the same address
    }
    if (out) *out = ptr;
    return CCH_OK;
}

}  // namespace cch

extern "C" int64_t cch_moe_init_routing_workspace_bytes(int64_t rows, int num_experts)
{
    if (rows < 0 || num_experts < 1) return 0;
    const int64_t nchunks = (rows + cch::ROUTE_CHUNK - 1) / cch::ROUTE_CHUNK;
    return std::max<int64_t>(nchunks, 1) * num_experts * (int64_t)sizeof(int32_t);
}

extern "C" int cch_moe_init_routing(const int32_t *expert_idx, int64_t rows, int num_experts, int32_t *dst_to_src,
                                    int32_t *src_to_dst, int32_t *expert_tokens, int cumsum, void *workspace,
                                    int64_t workspace_bytes, void *stream)
{
    using namespace cch;
    int64_t nchunks = 0;
    int rc = route_check("cch_moe_init_routing", expert_idx, rows, num_experts, dst_to_src, src_to_dst, expert_tokens, &nchunks);
    if (rc) return rc;
    CCH_REQUIRE(workspace != nullptr && workspace_bytes >= cch_moe_init_routing_workspace_bytes(rows, num_experts),
                "cch_moe_init_routing: workspace of %lld bytes, need %lld", (long long)workspace_bytes,
                (long long)cch_moe_init_routing_workspace_bytes(rows, num_experts));
    return route_launch(expert_idx, rows, num_experts, nchunks, dst_to_src, src_to_dst, expert_tokens, cumsum,
                        static_cast<int32_t *>(workspace), static_cast<hipStream_t>(stream));
}

extern "C" int cch_moe_init_routing_noalloc(const int32_t *expert_idx, int64_t rows, int num_experts, int32_t *dst_to_src,
                                            int32_t *src_to_dst, int32_t *expert_tokens, int cumsum, void *stream)
{
    using namespace cch;
    int64_t nchunks = 0;
    int rc = route_check("cch_moe_init_routing_noalloc", expert_idx, rows, num_experts, dst_to_src, src_to_dst, expert_tokens,
                         &nchunks);
    if (rc) return rc;
    CCH_REQUIRE(nchunks * num_experts <= ROUTE_STATIC_ENTRIES,
                "cch_moe_init_routing_noalloc: ceil(rows/%d) * num_experts = %lld exceeds the built-in area of %lld entries; "
                "use cch_moe_init_routing with a workspace", ROUTE_CHUNK, (long long)(nchunks * num_experts),
                (long long)ROUTE_STATIC_ENTRIES);
    int32_t *hist = nullptr;
    rc = routing_scratch_setup(&hist);
    if (rc) return rc;
    return route_launch(expert_idx, rows, num_experts, nchunks, dst_to_src, src_to_dst, expert_tokens, cumsum, hist,
                        static_cast<hipStream_t>(stream));
}
