// The MXFP8 MoE FFN of one rank that holds every expert, routing to combine, as one call: routing sort and MXFP8
// quantise-and-scatter, GMM1 + SwiGLU + MXFP8 quantise, GMM2, weighted un-permute (the reference's Ascend950DispatchFFNCombine,
// examples/ascend950_dispatch_ffn_combine/ascend950_dispatch_ffn_combine_device.h:124-176).  What lies between the launches is one
// workspace of the caller's.
//
// Packed rows [payload | scales] between the first two stages start on 128-byte lines: a row of K bytes and 2*ceil(K/64) scales is no
// multiple of 4 bytes where K is an odd multiple of 64, and then went to the one-thread-per-element GEMM (45 tokens to 6 of 16 experts, K 4160, N 512:
// 6.2 ms for the call, now 0.037; 300 to 8 of 8, K 1984, N 1024: 12.2 ms, now 0.043).
//
// Where the routes are few enough the sort and the quantiser are one launch.  The quantiser needs where its tokens' routes go, which the sort
// says at its end; but those places are two counts per expert, all routes and the routes of earlier tokens, which a workgroup takes
// for itself while its tokens are on their way from memory.  Together the workgroups have what the later stages ask of the sort: each
// writes its routes' places, the first one the tokens per expert.  (With a workgroup of its own that sorted once more beside the others, as one CU can,
// the launch waited for it, and its registers and LDS cost the others half of their places on a CU from 4097 routes on: 4096 tokens to 2 of 16, K 2048
// 61.4 -> 54.4 us for the call without it, 8192 to 1 of 256, K 512 48.0 -> 41.4.)
// The routes are counted with LDS atomics; by ballots over the keys' bits the whole call took, from some thousand routes on, 1 to 4 % longer.
//
// The rule: up to FFN_MAX_COUNTED routes looked at by all workgroups together.  Each looks at all routes, and there are the more of them the longer
// tokens are.  Whole calls, two launches -> one (us, n 256 or 512): 256 to 1 of 64, K 512 18.4 -> 17.2, 1500 to 2 of 64, K 2048 37.9 -> 36.2, 512 to 8 of 64,
// K 7168 94.3 -> 92.5 (1.0 M looked at), 1024 to 8 of 64, K 8192 171 -> 167 (4.2 M), 2048 to 4 of 64, K 8192 178.7 -> 171.7, 2048 to 4 of 8, K 8192 173 -> 159 and
// 4096 to 1 of 16, K 7168 103 -> 101 (8.4 M each); but 8192 to 1 of 16, K 4096 102 -> 106 (16.8 M), 8192 to 1 of 64, K 7168 192 -> 204 and 8192 to 1 of 64,
// K 8192 211 -> 220 (33 M).
//
// Packed rows are stored with the non-temporal hint where the weights are more than the caches hold (FFN_CACHED_WEIGHTS), as the quantiser's own launch
// stores them: 3000 to 1 of 256, K 7168, n 256 302 us without, 288 with it, 512 to 6 of 16, K 7168, n 4096 225 and 215.  Where the weights stay in the caches
// the rows had better do so too: 512 to 6 of 16, K 7168, n 512 70.5 without, 75 with it, 2048 to 1 of 64, K 7168, n 256 86.7 and 90.3.
#include <algorithm>
#include <atomic>

#include "common.h"
#include "mx_formats.h"
#include "mx_quant_block.h"
#include "route_keys.h"

namespace cch {

extern std::atomic<int> g_route_three_launches;   // routing.hip
int quant_scatter(const void *x, const int32_t *expanded_row_idx, void *packed_out, int64_t out_rows, int64_t row_pitch, int64_t tokens, int64_t k, int top_k,
                  int fmt, int rounding, void *stream);
int mx_gmm_swiglu_mx_rows(const void *packed_a, int64_t row_pitch, const void *b, const void *sb, const int32_t *group_sizes, void *payload, void *scales,
                          int64_t num_experts, int64_t t, int64_t n, int64_t k, int fmt, int trans_b, int out_fmt, void *stream);

constexpr int FFN_WAVES = 16;
constexpr int FFN_MAX_TOPK = 8;
constexpr int FFN_TOKENS_ROUTES = FFN_WAVES * FFN_MAX_TOPK;   // of one workgroup's tokens
constexpr int FFN_MAX_GROUPS = 8, FFN_MAX_ROUTES = FFN_MAX_GROUPS * 64 * FFN_WAVES;   // of a call in one launch
constexpr int FFN_MAX_EXPERTS = 256;   // as many groups as the projections take
constexpr int64_t FFN_MAX_COUNTED = (int64_t)1 << 23;
constexpr double FFN_CACHED_WEIGHTS = 256e6;

// Every workgroup: `tpw` tokens, of `ppr` pieces of up to 1024 elements each (`rest` in a token's last), a wave to a piece.  For the places
// of their routes the waves share the list of all routes, GROUPS x 64 entries each; the first workgroup also writes the tokens per expert.
template <int GROUPS, bool HINT>
__global__ __launch_bounds__(64 * FFN_WAVES) void moe_dispatch_kernel(const uint16_t *__restrict__ x, const int32_t *__restrict__ expert_idx, int tokens, int topk,
                                                                     int experts, int bits, int32_t *__restrict__ src_to_dst, int32_t *__restrict__ expert_tokens,
                                                                     uint8_t *__restrict__ packed, int K, int pitch, int ppr, int rest, int tpw)
{
    const int rows = tokens * topk;
    // routes per expert, those of every sixteenth lane; in the upper half those before this workgroup's (8191 at most)
    constexpr int COPIES = 16, PITCH = COPIES + 1;   // (17: experts on different banks)
    __shared__ int32_t count[FFN_MAX_EXPERTS * PITCH];
    __shared__ int32_t total[FFN_MAX_EXPERTS], place_of[FFN_MAX_EXPERTS], place[FFN_TOKENS_ROUTES];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int t0 = (int)blockIdx.x * tpw, mine = min(tpw, tokens - t0), routes = mine * topk, items = mine * ppr;
    auto item_of = [&](int i, int &t, int &have) {
        t = i / ppr;
        const int c = i - t * ppr;
        have = c == ppr - 1 ? rest : 1024;
        return c;
    };
    u32x4 v[2] = {};
    int t = 0, have = 0, c = 0;
    if (wave < items) {
        c = item_of(wave, t, have);
        load_piece(x + (size_t)(t0 + t) * K + (size_t)c * 1024, have, v);
    }
    int key[GROUPS];
#pragma unroll
    for (int u = 0; u < GROUPS; u++) {
        const int i = (u * FFN_WAVES + wave) * 64 + lane;
        key[u] = i < rows ? expert_idx[i] : -1;
    }
    // this workgroup's routes, two per lane
    const int first = t0 * topk;
    int own[2];
#pragma unroll
    for (int h = 0; h < 2; h++) own[h] = h * 64 + lane < routes ? expert_idx[first + h * 64 + lane] : -1;
    for (int i = threadIdx.x; i < experts * PITCH; i += 64 * FFN_WAVES) count[i] = 0;
    __syncthreads();
    const uint64_t below = (1ull << lane) - 1ull;
#pragma unroll
    for (int u = 0; u < GROUPS; u++)
        if (key[u] >= 0 && key[u] < experts) atomicAdd(&count[key[u] * PITCH + lane % COPIES], (u * FFN_WAVES + wave) * 64 + lane < first ? 0x10001 : 1);
    __syncthreads();
    for (int e = threadIdx.x; e < FFN_MAX_EXPERTS; e += 64 * FFN_WAVES) {
        int sum = 0;
#pragma unroll
        for (int i = 0; i < COPIES; i++) sum += e < experts ? count[e * PITCH + i] : 0;
        total[e] = sum & 0xFFFF;
        place_of[e] = sum >> 16;
        if (blockIdx.x == 0 && e < experts) expert_tokens[e] = sum & 0xFFFF;
    }
    __syncthreads();
    // the place of an expert's first route here: the routes of the experts before it, and its own of earlier workgroups
    if (wave == 0) {
        int sum = 0, part[FFN_MAX_EXPERTS / 64];
#pragma unroll
        for (int v = 0; v < FFN_MAX_EXPERTS / 64; v++) {
            part[v] = sum;
            sum += total[lane * (FFN_MAX_EXPERTS / 64) + v];
        }
        int incl = sum;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int up = __shfl_up(incl, off, 64);
            if (lane >= off) incl += up;
        }
#pragma unroll
        for (int v = 0; v < FFN_MAX_EXPERTS / 64; v++) place_of[lane * (FFN_MAX_EXPERTS / 64) + v] += incl - sum + part[v];
        // (one wave's LDS accesses execute in program order)
#pragma unroll
        for (int h = 0; h < 2; h++) {
            if (h * 64 >= routes) break;
            const bool routed = own[h] >= 0 && own[h] < experts;
            const uint64_t same = same_key_lanes(own[h], routed, bits);
            int at = -1;
            if (routed) at = place_of[own[h]] + __builtin_popcountll(same & below);
            if (routed && (same & below) == 0) place_of[own[h]] += __builtin_popcountll(same);
            place[h * 64 + lane] = at;
            if (h * 64 + lane < routes) src_to_dst[first + h * 64 + lane] = at;
        }
    }
    __syncthreads();
    for (int i = wave; i < items; i += FFN_WAVES) {
        if (i != wave) {
            c = item_of(i, t, have);
            load_piece(x + (size_t)(t0 + t) * K + (size_t)c * 1024, have, v);
        }
        uint32_t q[2][2], sdw[2];
        quant_piece<CCH_FMT_E4M3, false>(v, q, sdw);
        const PieceOut o = piece_out<CCH_FMT_E4M3>(q, sdw);
        for (int j = 0; j < topk; j++) {
            const int at = __builtin_amdgcn_readfirstlane(place[t * topk + j]);
            if (at < 0) continue;
            uint8_t *row = packed + (size_t)at * pitch;
            store_piece<CCH_FMT_E4M3, HINT>(o, have, row + c * 1024, row + K + c * 32);
        }
    }
}

// Bytes between packed rows: whole lines, unless that alone would put the buffer out of the GEMM's 32-bit reach.
static int64_t ffn_pitch(int64_t rows, int64_t k)
{
    const int64_t row = k + 2 * ((k + 63) / 64), lines = (row + 127) & ~(int64_t)127;
    return rows * lines < ((int64_t)1 << 31) ? lines : row;
}

static int ffn_dispatch(const void *x, const int32_t *expert_idx, int64_t m, int64_t k, int top_k, int experts, int32_t *dst_to_src, int32_t *src_to_dst,
                        int32_t *expert_tokens, void *packed, int64_t pitch, int64_t n, void *route_ws, int64_t route_bytes, void *stream)
{
    const int64_t rows = m * top_k, ppr = (k + 1023) / 1024, tpw = std::max<int64_t>(1, FFN_WAVES / ppr), workgroups = (m + tpw - 1) / tpw;
    const bool one_launch = rows <= FFN_MAX_ROUTES && workgroups * rows <= FFN_MAX_COUNTED && k % 64 == 0 && pitch % 16 == 0 && aligned(x, 16) &&
                            aligned(packed, 16) && !g_route_three_launches.load(std::memory_order_relaxed);
    if (!one_launch) {
        const int rc = cch_moe_init_routing(expert_idx, rows, experts, dst_to_src, src_to_dst, expert_tokens, 0, route_ws, route_bytes, stream);
        return rc ? rc : quant_scatter(x, src_to_dst, packed, rows, pitch, m, k, top_k, CCH_FMT_E4M3, CCH_ROUND_RNE, stream);
    }
    const int groups = (int)((rows + 64 * FFN_WAVES - 1) / (64 * FFN_WAVES));
    const bool hint = 1.5 * (double)k * (double)n * experts > FFN_CACHED_WEIGHTS;   // (the down projection has half as many as the up projection)
    auto kern = groups <= 1   ? (hint ? moe_dispatch_kernel<1, true> : moe_dispatch_kernel<1, false>)
                : groups <= 2 ? (hint ? moe_dispatch_kernel<2, true> : moe_dispatch_kernel<2, false>)
                : groups <= 4 ? (hint ? moe_dispatch_kernel<4, true> : moe_dispatch_kernel<4, false>)
                              : (hint ? moe_dispatch_kernel<8, true> : moe_dispatch_kernel<8, false>);
    hipLaunchKernelGGL(kern, dim3((unsigned)workgroups), dim3(64 * FFN_WAVES), 0, static_cast<hipStream_t>(stream),
                       static_cast<const uint16_t *>(x), expert_idx, (int)m, top_k, experts, route_key_bits(experts), src_to_dst, expert_tokens,
                       static_cast<uint8_t *>(packed), (int)k, (int)pitch, (int)ppr, (int)(k - (ppr - 1) * 1024), (int)tpw);
    return launch_status("moe_dispatch_kernel");
}

// Pieces of the workspace, each on a boundary that every kernel is content with.
struct FfnWorkspace {
    int64_t d2s, s2d, cnt, route, route_bytes, packed, act, scales, y, end;
};
static FfnWorkspace ffn_workspace(int64_t m, int64_t k, int64_t top_k, int64_t e, int64_t n)
{
    const int64_t rows = m * top_k, h = n / 2;
    FfnWorkspace w{};
    auto piece = [&](int64_t bytes) {
        const int64_t at = w.end;
        w.end += (bytes + 511) & ~(int64_t)511;
        return at;
    };
    w.route_bytes = std::max<int64_t>(cch_moe_init_routing_workspace_bytes(rows, (int)e), 4);
    w.d2s = piece(rows * 4);
    w.s2d = piece(rows * 4);
    w.cnt = piece(e * 4);
    w.route = piece(w.route_bytes);
    w.packed = piece(rows * ffn_pitch(rows, k));
    w.act = piece(rows * h);
    w.scales = piece(rows * 2 * ((h + 63) / 64));
    w.y = piece(rows * k * 2);
    return w;
}

}  // namespace cch

extern "C" int64_t cch_moe_ffn_mxfp8_workspace_bytes(int64_t m, int64_t k, int top_k, int64_t num_experts, int64_t n)
{
    if (m < 0 || k < 0 || top_k < 1 || num_experts < 1 || n < 0 || m >> 31 || k >> 31 || n >> 31 || num_experts >> 31) return 0;
    return std::max<int64_t>(cch::ffn_workspace(m, k, top_k, num_experts, n).end, 1);
}

extern "C" int cch_moe_ffn_mxfp8(const void *x, const int32_t *expert_idx, const float *probs, const void *w1, const void *sw1, const void *w2, const void *sw2,
                                 void *out, int64_t m, int64_t k, int top_k, int64_t num_experts, int64_t n, int trans_b, void *workspace, int64_t workspace_bytes,
                                 void *stream)
{
    using namespace cch;
    clear_error();
    CCH_REQUIRE(m >= 0 && k >= 0 && n >= 0 && !(m >> 31) && !(k >> 30) && !(n >> 31), "cch_moe_ffn_mxfp8: bad shape m=%lld k=%lld n=%lld", (long long)m, (long long)k, (long long)n);
    CCH_REQUIRE(top_k >= 1 && top_k <= FFN_MAX_TOPK, "cch_moe_ffn_mxfp8: top_k=%d outside 1..%d", top_k, FFN_MAX_TOPK);
    CCH_REQUIRE(num_experts >= 1 && num_experts <= FFN_MAX_EXPERTS, "cch_moe_ffn_mxfp8: num_experts=%lld outside 1..%d", (long long)num_experts, FFN_MAX_EXPERTS);
    CCH_REQUIRE(n % 2 == 0, "cch_moe_ffn_mxfp8: n=%lld must be even (gate | up halves)", (long long)n);
    CCH_REQUIRE(trans_b == 0 || trans_b == 1, "cch_moe_ffn_mxfp8: trans_b %d", trans_b);
    const int64_t rows = m * top_k, h = n / 2;
    CCH_REQUIRE(!(rows >> 31), "cch_moe_ffn_mxfp8: %lld routes", (long long)rows);
    if (m == 0 || k == 0) return CCH_OK;
    const FfnWorkspace w = ffn_workspace(m, k, top_k, num_experts, n);
    CCH_REQUIRE(x && expert_idx && probs && out && (n == 0 || (w1 && sw1 && w2 && sw2)), "cch_moe_ffn_mxfp8: null pointer");
    CCH_REQUIRE(workspace && aligned(workspace, 512) && workspace_bytes >= w.end, "cch_moe_ffn_mxfp8: workspace of %lld bytes, need %lld on a 512-byte boundary",
                (long long)workspace_bytes, (long long)w.end);
    uint8_t *p = static_cast<uint8_t *>(workspace);
    int32_t *s2d = reinterpret_cast<int32_t *>(p + w.s2d), *cnt = reinterpret_cast<int32_t *>(p + w.cnt);
    const int64_t pitch = ffn_pitch(rows, k);
    int rc = ffn_dispatch(x, expert_idx, m, k, top_k, (int)num_experts, reinterpret_cast<int32_t *>(p + w.d2s), s2d, cnt, p + w.packed, pitch, n, p + w.route,
                          w.route_bytes, stream);
    char note[512] = "";   // that the up projection ran on the generic kernels, if it did: the down projection's call empties the message
    if (rc == CCH_OK) {
        rc = mx_gmm_swiglu_mx_rows(p + w.packed, pitch, w1, sw1, cnt, p + w.act, p + w.scales, num_experts, rows, n, k, CCH_FMT_E4M3, trans_b, CCH_FMT_E4M3, stream);
        snprintf(note, sizeof(note), "%s", cch_last_error());
    }
    if (rc == CCH_OK) rc = cch_mx_gmm(p + w.act, p + w.scales, w2, sw2, cnt, p + w.y, num_experts, rows, k, h, CCH_FMT_E4M3, trans_b, stream);
    if (rc == CCH_OK && note[0] && !cch_last_error()[0]) fail(CCH_OK, "%s", note);
    if (rc == CCH_OK) rc = cch_moe_token_unpermute(p + w.y, s2d, probs, out, rows, m, k, top_k, stream);
    return rc;
}
