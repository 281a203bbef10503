// MX block quantiser: bf16 -> FP8 (E4M3/E5M2) or FP4 (E2M1/E1M2) payload + one E8M0 scale per
// 32 elements.  Streaming, HBM-bound kernel: every lane owns 8 consecutive elements (one
// 16-byte load), four neighbouring lanes own one MX block and reduce its maximum with two
// DPP quad permutes; payload leaves as one 8-byte (FP8) or 4-byte (FP4) store per lane.
//
// Follows CommBlockMxQuant::ComputeMxQuant (include/catccos/comm/block/comm_block_mx_quant.hpp:414-663)
// in intent and the generator examples/utils/gen_mx_quant_allgather_data.py:255-313, :385-449
// bit for bit.
#include <atomic>
#include <cstring>

#include "common.h"
#include "mx_formats.h"
#include "mx_quant_block.h"

namespace cch {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32_any __attribute__((aligned(1)));                          // global memory takes them at any address
typedef uint32_t u32x2_any __attribute__((ext_vector_type(2), aligned(1)));

constexpr int QUANT_THREADS = 512;        // large workgroups: the dispatcher places 512 blocks of 256 threads noticeably slower
constexpr int QUANT_UNROLL = 2;           // wave-steps (64 lanes x 8 elements) per batch
constexpr int QUANT_BLOCKS_PER_CU = 8;    // resident workgroups per CU the grid is sized for

// x [rows,K] bf16.  One wave-step = 64 lanes x 8 elements of one row; a row has `wpr` wave-steps.
// The grid is sized to the machine, not to the problem: every wave walks the list of wave-steps
// with a grid stride, QUANT_UNROLL at a time, and requests the next batch before it converts the
// current one, so that each wave always has loads in flight.
// VEC: K % 8 == 0 and all pointers suitably aligned (SCATTER: x alone), so whole-vector accesses are legal.
// PAIR (needs VEC, K % 16 == 0 and 16-byte aligned payload rows): neighbouring lanes swap halves
// of two wave-steps so that each lane stores one 16-byte (FP8) or 8-byte (FP4) piece instead of
// two of half that size; the store path's cost is per instruction, not per byte.
// SCATTER (without PAIR): row r of x is written to rows dst_idx[r*topk + 0 .. topk-1] of the output
// instead of row r; negative entries are skipped.  The row's destinations are read with the row
// itself, one batch ahead of their use.  `sstride` is the distance between scale rows (equal to
// `sld` unless payload and scales share one packed row).
constexpr int QUANT_MAX_TOPK = 8;
template <int FMT, int RND, bool HWCVT, bool VEC, bool PAIR, bool SCATTER = false>
__global__ __launch_bounds__(QUANT_THREADS) void mx_quant_rows_kernel(
    const uint16_t *__restrict__ x, uint8_t *__restrict__ payload, uint8_t *__restrict__ scales, int rows, int K,
    int nblk, int sld, int pld, int wpr, int total_ws, const int32_t *__restrict__ dst_idx = nullptr, int topk = 1,
    int sstride = 0, int out_rows = 0x7FFFFFFF)
{
    static_assert(!(SCATTER && PAIR), "the scatter variant stores one wave-step at a time");
    if (!SCATTER) sstride = sld;
    constexpr bool FP4 = is_fp4_v<FMT>;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (QUANT_THREADS / 64) + (threadIdx.x >> 6)));
    const int stride = (int)gridDim.x * (QUANT_THREADS / 64) * QUANT_UNROLL;

    struct Batch {
        uint32_t w[QUANT_UNROLL][4];
        int row[QUANT_UNROLL], k0[QUANT_UNROLL];
        int dst[QUANT_UNROLL][SCATTER ? QUANT_MAX_TOPK : 1];
    };
    auto fetch = [&](int ws0, Batch &bt) {
#pragma unroll
        for (int u = 0; u < QUANT_UNROLL; u++) {
            const int ws = ws0 + u;
            const int r = ws / wpr;
            bt.row[u] = ws < total_ws ? r : -1;
            bt.k0[u] = ((ws - r * wpr) * 64 + lane) * 8;
            bt.w[u][0] = bt.w[u][1] = bt.w[u][2] = bt.w[u][3] = 0;
            if constexpr (SCATTER) {
#pragma unroll
                for (int t = 0; t < QUANT_MAX_TOPK; t++) {
                    bt.dst[u][t] = (bt.row[u] >= 0 && t < topk) ? dst_idx[(size_t)bt.row[u] * topk + t] : -1;
                    if (bt.dst[u][t] >= out_rows) bt.dst[u][t] = -1;   // a row past the output is skipped like a negative one
                }
            }
            if (bt.row[u] >= 0 && bt.k0[u] < K) {
                const uint16_t *src = x + (size_t)bt.row[u] * K + bt.k0[u];
                if (VEC) {
                    const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4 *>(src));
                    bt.w[u][0] = v[0]; bt.w[u][1] = v[1]; bt.w[u][2] = v[2]; bt.w[u][3] = v[3];
                } else {
#pragma unroll
                    for (int i = 0; i < 8; i++)
                        if (bt.k0[u] + i < K) bt.w[u][i >> 1] |= (uint32_t)src[i] << ((i & 1) * 16);
                }
            }
        }
    };
    auto convert = [&](const Batch &bt) {
        uint32_t held[2] = {0, 0};  // PAIR: payload of the even wave-step, waiting for its partner
#pragma unroll
        for (int u = 0; u < QUANT_UNROLL; u++) {
            if (bt.row[u] < 0) continue;  // wave-uniform
            const uint32_t amax_bits = block_amax_bits(bt.w[u]);
            int e;
            bool is_nan;
            const uint32_t sbyte = shared_exp_byte<FMT>(amax_bits, e, is_nan);
            uint32_t q[2];
            quant8<FMT, RND, HWCVT>(bt.w[u], e, is_nan, q);
            const int k0 = bt.k0[u], blk = k0 >> 5;
            if (PAIR) {
                // Wave-steps come in pairs (u even, u odd); a pair is complete unless the list
                // ends on the even one.  Even lanes end up with the even step's 16 (8) bytes of
                // lanes l and l+1, odd lanes with the odd step's bytes of lanes l-1 and l.
                const bool odd_lane = lane & 1;
                const bool partner = (u & 1) || (u + 1 < QUANT_UNROLL && bt.row[u + 1] >= 0);  // wave-uniform
                if (!(u & 1) && partner) {
                    held[0] = q[0];
                    held[1] = q[1];
                } else if (u & 1) {
                    const int ke = bt.k0[u - 1], ko = k0;  // same lane offset in both steps unless the row changed
                    uint32_t send0 = odd_lane ? held[0] : q[0], send1 = odd_lane ? held[1] : q[1];
                    const uint32_t recv0 = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)send0, 0xB1, 0xF, 0xF, true);
                    const uint32_t recv1 = FP4 ? 0u : (uint32_t)__builtin_amdgcn_update_dpp(0, (int)send1, 0xB1, 0xF, 0xF, true);
                    const int rw = odd_lane ? bt.row[u] : bt.row[u - 1];
                    const int kk = odd_lane ? ko - 8 : ke;
                    if (kk < K) {
                        uint8_t *dst = payload + (size_t)rw * pld + (FP4 ? (kk >> 1) : kk);
                        if (FP4) {
                            u32x2 o = odd_lane ? (u32x2){recv0, q[0]} : (u32x2){held[0], recv0};
                            __builtin_nontemporal_store(o, reinterpret_cast<u32x2 *>(dst));
                        } else {
                            u32x4 o = odd_lane ? (u32x4){recv0, recv1, q[0], q[1]} : (u32x4){held[0], held[1], recv0, recv1};
                            __builtin_nontemporal_store(o, reinterpret_cast<u32x4 *>(dst));
                        }
                    }
                } else if (k0 < K) {  // unpaired last step
                    uint8_t *dst = payload + (size_t)bt.row[u] * pld + (FP4 ? (k0 >> 1) : k0);
                    if (FP4) {
                        __builtin_nontemporal_store(q[0], reinterpret_cast<uint32_t *>(dst));
                    } else {
                        u32x2 o = {q[0], q[1]};
                        __builtin_nontemporal_store(o, reinterpret_cast<u32x2 *>(dst));
                    }
                }
            } else if (SCATTER) {
#pragma unroll
                for (int t = 0; t < QUANT_MAX_TOPK; t++) {
                    const int drow = bt.dst[u][t];
                    if (drow < 0) continue;  // wave-uniform
                    if (k0 < K) {
                        uint8_t *dst = payload + (size_t)drow * pld + (FP4 ? (k0 >> 1) : k0);
                        if (VEC) {
                            // (packed rows of 66 bytes per 64 elements start on even addresses: vector stores of any alignment)
                            if (FP4) *reinterpret_cast<u32_any *>(dst) = q[0];
                            else *reinterpret_cast<u32x2_any *>(dst) = (u32x2_any){q[0], q[1]};
                        } else if (FP4) {
                            for (int i = 0; i < 4; i++)
                                if (k0 + 2 * i < K) dst[i] = (uint8_t)(q[0] >> (8 * i)) & (k0 + 2 * i + 1 < K ? 0xFF : 0x0F);
                        } else {
                            for (int i = 0; i < 8; i++)
                                if (k0 + i < K) dst[i] = (uint8_t)(q[i >> 2] >> (8 * (i & 3)));
                        }
                    }
                    if (blk < nblk) {
                        uint8_t *srow = scales + (size_t)drow * sstride;
                        if ((lane & 3) == 0) srow[blk] = (uint8_t)sbyte;
                        if ((lane & 3) == 1 && blk == nblk - 1 && sld != nblk) srow[nblk] = 127;  // even padding, 1.0
                    }
                }
                continue;
            } else if (k0 < K) {
                uint8_t *dst = payload + (size_t)bt.row[u] * pld + (FP4 ? (k0 >> 1) : k0);
                if (VEC) {
                    if (FP4) {
                        __builtin_nontemporal_store(q[0], reinterpret_cast<uint32_t *>(dst));
                    } else {
                        u32x2 o = {q[0], q[1]};
                        __builtin_nontemporal_store(o, reinterpret_cast<u32x2 *>(dst));
                    }
                } else if (FP4) {
                    for (int i = 0; i < 4; i++)
                        if (k0 + 2 * i < K) dst[i] = (uint8_t)(q[0] >> (8 * i)) & (k0 + 2 * i + 1 < K ? 0xFF : 0x0F);
                } else {
                    for (int i = 0; i < 8; i++)
                        if (k0 + i < K) dst[i] = (uint8_t)(q[i >> 2] >> (8 * (i & 3)));
                }
            }
            if (blk < nblk) {
                uint8_t *srow = scales + (size_t)bt.row[u] * sld;
                if ((lane & 3) == 0) srow[blk] = (uint8_t)sbyte;
                if ((lane & 3) == 1 && blk == nblk - 1 && sld != nblk) srow[nblk] = 127;  // even padding, 1.0
            }
        }
    };

    // Two batches in ping-pong: while one is converted and stored, the other's loads are in flight.
    Batch b0, b1;
    int ws0 = wave * QUANT_UNROLL;
    if (ws0 >= total_ws) return;
    fetch(ws0, b0);
    for (;;) {
        const int ws1 = ws0 + stride, ws2 = ws1 + stride;  // all wave-uniform
        if (ws1 < total_ws) fetch(ws1, b1);
        convert(b0);
        if (ws1 >= total_ws) break;
        if (ws2 < total_ws) fetch(ws2, b0);
        convert(b1);
        if (ws2 >= total_ws) break;
        ws0 = ws2;
    }
}

// Fast path of the row quantiser: round to nearest even with the hardware conversions, K a multiple of 64 and 16-byte
// aligned buffers.  Rows of whole pairs of MX blocks lie back to back, payload and scales alike, so the tensor is one run of
// elements: a wave owns pieces of 1024 consecutive ones (wherever rows begin), keeps its next piece in flight while it converts the current one,
// stores 16 (FP8) or 8 (FP4) payload bytes per lane and writes the 32 scale bytes as dwords gathered with row shifts.
// Only the last piece of the run can be partial; nothing else is checked per lane.  WHOLE: it is not (m * K, with SCATTER K, a multiple of 1024), and the
// loop carries no second form of its loads and stores: E4M3 4096 x 7168 15.9 us with both forms in the loop, 15.8 without, FP4 4096 x 7168 14.0 and 13.6,
// FP4 scattered to two rows 4096 x 5120 14.1 and 13.7, E4M3 scattered to one 4096 x 4096 11.3 and 10.9.
// Bound by HBM where large (4096 x 7168: 5.9 TB/s), by a launch and one load's latency where small.  Against the general kernel, which K no
// multiple of 1024 took before: 4096 x 6784 17.7 -> 14.9 us, 8192 x 1984 10.9 -> 9.3, 16384 x 1984 to FP4 18.0 -> 14.7, 8192 x 7104 from half
// 36.9 -> 30.9, 2048 x 3008 5.1 -> 4.0, 64 x 1984 3.0 -> 2.4.
// SCATTER: row r goes to rows dst_idx[r*topk + 0 .. topk-1], `pitch` bytes apart (a multiple of 16); a row is then `ppr` pieces of its
// own.  `rest` is what the last piece of the run (SCATTER: of each row) holds, a multiple of 64.  Rows of whole pieces are stored with the
// non-temporal hint, others without.  What the hint is worth depends on what the caches still hold, from one size to the next (E4M3, us, hinted and plain:
// whole 4096 x 7168 to two rows 24.4, 22.4, 8192 x 7168 to two 50.2, 53.2, to eight 141, 160; partial 4096 x 2560 to eight 28.3, 23.0, 16384 x 2560 to two
// 38.4, 33.3, to four 61.6, 67.2): over 52 sizes of whole pieces the two are equal in the mean, over 28 of
// partial ones the hint costs 3 %, and at three of them the general kernel, which stores without it, was ahead (4096 x 2560 to eight 27.0).
// HALF: the input is IEEE half instead of bf16 (same layout, same stores; the shared exponent comes
// from the block maximum widened to fp32 and the codes from the packed-half conversions).
template <int FMT, bool WHOLE, bool SCATTER = false, bool HALF = false>
__global__ __launch_bounds__(QUANT_THREADS) void mx_quant_rows_fast_kernel(
    const uint16_t *__restrict__ x, uint8_t *__restrict__ payload, uint8_t *__restrict__ scales, int npairs, int rest, int K, int pitch,
    int ppr, const int32_t *__restrict__ dst_idx, int topk, int out_rows)
{
    constexpr bool FP4 = is_fp4_v<FMT>;
    const int wave = __builtin_amdgcn_readfirstlane((int)(blockIdx.x * (QUANT_THREADS / 64) + (threadIdx.x >> 6)));
    const int stride = (int)gridDim.x * (QUANT_THREADS / 64);

    struct Dest {
        int row[SCATTER ? QUANT_MAX_TOPK : 1];
    };
    // (all wave-uniform)
    auto have = [&](int p) { return !WHOLE && (SCATTER ? p % ppr == ppr - 1 : p == npairs - 1) ? rest : 1024; };
    auto fetch = [&](int p, u32x4 (&v)[2], Dest &d) {
        const int r = SCATTER ? p / ppr : 0, c = SCATTER ? p - r * ppr : p;  // row, piece of it
        load_piece(x + (size_t)r * K + (size_t)c * 1024, have(p), v);
        if constexpr (SCATTER) {
#pragma unroll
            for (int t = 0; t < QUANT_MAX_TOPK; t++) {
                d.row[t] = t < topk ? dst_idx[(size_t)r * topk + t] : -1;
                if (d.row[t] >= out_rows) d.row[t] = -1;   // a row past the output is skipped like a negative one
            }
        }
    };
    auto convert = [&](int p, const u32x4 (&v)[2], const Dest &d) {
        uint32_t q[2][2], sdw[2];
        quant_piece<FMT, HALF>(v, q, sdw);
        const PieceOut o = piece_out<FMT>(q, sdw);
        const int n = have(p);
        if constexpr (SCATTER) {
            const int c = p % ppr;
#pragma unroll
            for (int t = 0; t < QUANT_MAX_TOPK; t++)
                if (d.row[t] >= 0) store_piece<FMT, WHOLE>(o, n, payload + (size_t)d.row[t] * pitch + c * (FP4 ? 512 : 1024), scales + (size_t)d.row[t] * pitch + c * 32);
        } else {
            store_piece<FMT, true>(o, n, payload + (size_t)p * (FP4 ? 512 : 1024), scales + (size_t)p * 32);
        }
    };

    u32x4 v0[2], v1[2];
    Dest d0, d1;
    int p0 = wave;
    if (p0 >= npairs) return;
    fetch(p0, v0, d0);
    for (;;) {
        const int p1 = p0 + stride, p2 = p1 + stride;  // wave-uniform
        if (p1 < npairs) fetch(p1, v1, d1);
        convert(p0, v0, d0);
        if (p1 >= npairs) break;
        if (p2 < npairs) fetch(p2, v0, d0);
        convert(p1, v1, d1);
        if (p2 >= npairs) break;
        p0 = p2;
    }
}

// The fast kernel's launch: returns 1 when the shape or the alignment is not its own, so that the caller takes its general kernel.
template <int FMT, bool HALF>
static int launch_rows_fast(const void *x, void *payload, void *scales, int64_t m, int64_t k, hipStream_t stream)
{
    const int64_t npairs = (m * k + 1023) / 1024;
    if (!(k % 64 == 0 && aligned(x, 16) && aligned(payload, 16) && aligned(scales, 4) && npairs < ((int64_t)1 << 30))) return 1;
    int dev = 0, cus = 0;
    CCH_HIP(hipGetDevice(&dev));
    CCH_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const unsigned grid = (unsigned)std::min<int64_t>((npairs + QUANT_THREADS / 64 - 1) / (QUANT_THREADS / 64), (int64_t)cus * QUANT_BLOCKS_PER_CU);
    const int rest = (int)(m * k - (npairs - 1) * 1024);
    auto kern = rest == 1024 ? mx_quant_rows_fast_kernel<FMT, true, false, HALF> : mx_quant_rows_fast_kernel<FMT, false, false, HALF>;
    hipLaunchKernelGGL(kern, dim3(grid), dim3(QUANT_THREADS), 0, stream, static_cast<const uint16_t *>(x), static_cast<uint8_t *>(payload),
                       static_cast<uint8_t *>(scales), (int)npairs, rest, 0, 0, 1, nullptr, 1, 0);
    return launch_status("mx_quant_rows_fast_kernel");
}

int mx_quant_rows_fast_half(const void *x, void *payload, void *scales, int64_t m, int64_t k, int fmt, hipStream_t stream)
{
    if (fmt == CCH_FMT_E4M3) return launch_rows_fast<CCH_FMT_E4M3, true>(x, payload, scales, m, k, stream);
    if (fmt == CCH_FMT_E5M2) return launch_rows_fast<CCH_FMT_E5M2, true>(x, payload, scales, m, k, stream);
    if (fmt == CCH_FMT_E2M1) return launch_rows_fast<CCH_FMT_E2M1, true>(x, payload, scales, m, k, stream);
    return 1;
}

template <int FMT, int RND, bool HWCVT>
static int launch_rows(const void *x, void *payload, void *scales, int64_t m, int64_t k, hipStream_t stream)
{
    const bool fp4 = is_fp4_v<FMT>;
    const int64_t nblk = (k + 31) / 32, sld = 2 * ((nblk + 1) / 2), pld = fp4 ? (k + 1) / 2 : k;
    const int64_t wpr = (nblk * 4 + 63) / 64;
    const bool vec = (k % 8 == 0) && aligned(x, 16) && aligned(payload, 8);
    const bool pair = vec && (k % 16 == 0) && aligned(payload, 16) && QUANT_UNROLL % 2 == 0;
    if constexpr (HWCVT) {
        const int rc = launch_rows_fast<FMT, false>(x, payload, scales, m, k, stream);
        if (rc != 1) return rc;
    }
    int dev = 0, cus = 0;
    CCH_HIP(hipGetDevice(&dev));
    CCH_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int64_t max_blocks = (int64_t)cus * QUANT_BLOCKS_PER_CU;
    const int64_t rows_per_launch = std::max<int64_t>(1, (int64_t)(1 << 30) / wpr);
    for (int64_t r0 = 0; r0 < m; r0 += rows_per_launch) {
        const int64_t rows = std::min(rows_per_launch, m - r0);
        const int64_t total_ws = rows * wpr;
        const int64_t waves = (total_ws + QUANT_UNROLL - 1) / QUANT_UNROLL;
        const unsigned grid = (unsigned)std::min<int64_t>((waves + QUANT_THREADS / 64 - 1) / (QUANT_THREADS / 64), max_blocks);
        const uint16_t *xs = static_cast<const uint16_t *>(x) + r0 * k;
        uint8_t *ps = static_cast<uint8_t *>(payload) + r0 * pld;
        uint8_t *ss = static_cast<uint8_t *>(scales) + r0 * sld;
        if (vec && pair)
            hipLaunchKernelGGL((mx_quant_rows_kernel<FMT, RND, HWCVT, true, true>), dim3(grid), dim3(QUANT_THREADS), 0, stream,
                               xs, ps, ss, (int)rows, (int)k, (int)nblk, (int)sld, (int)pld, (int)wpr, (int)total_ws);
        else if (vec)
            hipLaunchKernelGGL((mx_quant_rows_kernel<FMT, RND, HWCVT, true, false>), dim3(grid), dim3(QUANT_THREADS), 0, stream,
                               xs, ps, ss, (int)rows, (int)k, (int)nblk, (int)sld, (int)pld, (int)wpr, (int)total_ws);
        else
            hipLaunchKernelGGL((mx_quant_rows_kernel<FMT, RND, HWCVT, false, false>), dim3(grid), dim3(QUANT_THREADS), 0,
                               stream, xs, ps, ss, (int)rows, (int)k, (int)nblk, (int)sld, (int)pld, (int)wpr,
                               (int)total_ws);
        int rc = launch_status("mx_quant_rows_kernel");
        if (rc) return rc;
    }
    return CCH_OK;
}


// Quantiser for a right-hand operand b [K,N] with MX blocks running down K.  One thread owns
// two adjacent columns of one 32-row block: 32 coalesced 4-byte loads, results written in
// either boundary layout.  Input preparation, not a hot path.
template <int FMT, int RND>
__global__ __launch_bounds__(256) void mx_quant_b_kernel(const uint32_t *__restrict__ b, uint8_t *__restrict__ payload,
                                                         uint8_t *__restrict__ scales, int K, int N, int trans_b)
{
    using T = FmtTraits<FMT>;
    constexpr bool FP4 = is_fp4_v<FMT>;
    const int np = blockIdx.x * 256 + threadIdx.x;  // column pair
    const int kb = blockIdx.y;
    if (np * 2 >= N) return;
    const int sld = K / 32;
    uint32_t w[32];
    uint32_t m0 = 0, m1 = 0;
#pragma unroll
    for (int i = 0; i < 32; i++) {
        w[i] = b[((size_t)(kb * 32 + i) * N) / 2 + np];
        m0 = max(m0, w[i] & 0x7FFFu);
        m1 = max(m1, (w[i] >> 16) & 0x7FFFu);
    }
    int e0, e1;
    bool n0, n1;
    const uint32_t s0 = shared_exp_byte<FMT>(m0, e0, n0), s1 = shared_exp_byte<FMT>(m1, e1, n1);
    // 2^-e in two exact factors (2^-127 is no normal float)
    const float i0 = pow2i(-min(e0, 126)), i1 = pow2i(-min(e1, 126));
    const float j0 = e0 > 126 ? 0.5f : 1.0f, j1 = e1 > 126 ? 0.5f : 1.0f;
    uint32_t q0[32], q1[32];
#pragma unroll
    for (int i = 0; i < 32; i++) {
        q0[i] = n0 ? T::NANCODE : encode_small<FMT, RND>(__uint_as_float(w[i] << 16) * i0 * j0);
        q1[i] = n1 ? T::NANCODE : encode_small<FMT, RND>(__uint_as_float(w[i] & 0xFFFF0000u) * i1 * j1);
    }
    const int n = np * 2;
    if (!trans_b) {
#pragma unroll
        for (int i = 0; i < 32; i++) {
            const size_t k = (size_t)kb * 32 + i;
            if (FP4) payload[k * (N / 2) + np] = (uint8_t)(q0[i] | (q1[i] << 4));
            else *reinterpret_cast<uint16_t *>(payload + k * N + n) = (uint16_t)(q0[i] | (q1[i] << 8));
        }
        uint8_t *sp = scales + ((size_t)(kb >> 1) * N + n) * 2 + (kb & 1);
        sp[0] = (uint8_t)s0;
        sp[2] = (uint8_t)s1;
    } else {
        if (FP4) {
            uint8_t *d0 = payload + (size_t)n * (K / 2) + kb * 16, *d1 = d0 + K / 2;
#pragma unroll
            for (int i = 0; i < 16; i++) {
                d0[i] = (uint8_t)(q0[2 * i] | (q0[2 * i + 1] << 4));
                d1[i] = (uint8_t)(q1[2 * i] | (q1[2 * i + 1] << 4));
            }
        } else {
            uint8_t *d0 = payload + (size_t)n * K + kb * 32, *d1 = d0 + K;
#pragma unroll
            for (int i = 0; i < 32; i++) {
                d0[i] = (uint8_t)q0[i];
                d1[i] = (uint8_t)q1[i];
            }
        }
        scales[(size_t)n * sld + kb] = (uint8_t)s0;
        scales[(size_t)(n + 1) * sld + kb] = (uint8_t)s1;
    }
}

template <int FMT, int RND>
static int launch_b(const void *b, void *payload, void *scales, int64_t k, int64_t n, int trans_b, hipStream_t stream)
{
    dim3 grid((unsigned)((n / 2 + 255) / 256), (unsigned)(k / 32));
    hipLaunchKernelGGL((mx_quant_b_kernel<FMT, RND>), grid, dim3(256), 0, stream, static_cast<const uint32_t *>(b),
                       static_cast<uint8_t *>(payload), static_cast<uint8_t *>(scales), (int)k, (int)n, trans_b);
    return launch_status("mx_quant_b_kernel");
}

// Quantise-once, scatter-to-top-K launch: packed output rows of payload bytes + padded scale bytes, `row_bytes` apart.
template <int FMT, int RND, bool HWCVT>
static int launch_scatter(const void *x, const int32_t *dst_idx, void *packed, int64_t row_bytes, int64_t tokens, int64_t k, int topk,
                          int out_rows, hipStream_t stream)
{
    const bool fp4 = is_fp4_v<FMT>;
    const int64_t nblk = (k + 31) / 32, sld = 2 * ((nblk + 1) / 2), pbytes = fp4 ? (k + 1) / 2 : k;
    if (row_bytes == 0) row_bytes = pbytes + sld;
    const int64_t wpr = (nblk * 4 + 63) / 64;
    // Only the loads ask for alignment.  Packed rows are a multiple of 8 bytes for every fourth multiple of 64 columns only, and
    // with byte stores for the others 4096 x 6784 to two rows each took 58.7 us (now 24.7), 512 x 1984 to four 9.1 (5.5), 2 x 7040
    // to two 5.6 (3.5).  (The general kernel's stores are without the non-temporal hint, also where rows are aligned: 4096 x 6912 to two 27.9 us,
    // with it 29.8, 16384 x 2816 to four 77.3 against 84.9, 512 x 6912 to six 9.5 against 10.1, FP4 likewise, none slower.)
    const bool vec = (k % 8 == 0) && aligned(x, 16);
    int dev = 0, cus = 0;
    CCH_HIP(hipGetDevice(&dev));
    CCH_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int64_t max_blocks = (int64_t)cus * QUANT_BLOCKS_PER_CU;
    uint8_t *out = static_cast<uint8_t *>(packed);
    // (rows of at most half a piece would leave half of every wave idle: 16384 x 512 to two, four and eight rows 13.4, 17.5 and 24.2 us, 12.3, 16.7
    // and 23.7 in the general kernel)
    if constexpr (HWCVT)
    if (k > 512 && k % 64 == 0 && aligned(x, 16) && aligned(packed, 16) && row_bytes % 16 == 0 && tokens * ((k + 1023) / 1024) < ((int64_t)1 << 30)) {
        const int64_t ppr = (k + 1023) / 1024, npairs = tokens * ppr;
        const unsigned grid = (unsigned)std::min<int64_t>((npairs + QUANT_THREADS / 64 - 1) / (QUANT_THREADS / 64), max_blocks);
        auto kern = k % 1024 == 0 ? mx_quant_rows_fast_kernel<FMT, true, true> : mx_quant_rows_fast_kernel<FMT, false, true>;
        hipLaunchKernelGGL(kern, dim3(grid), dim3(QUANT_THREADS), 0, stream,
                           static_cast<const uint16_t *>(x), out, out + pbytes, (int)npairs, (int)(k - (ppr - 1) * 1024), (int)k, (int)row_bytes,
                           (int)ppr, dst_idx, topk, out_rows);
        return launch_status("mx_quant_rows_fast_kernel (scatter)");
    }
    const int64_t rows_per_launch = std::max<int64_t>(1, (int64_t)(1 << 30) / wpr);
    for (int64_t r0 = 0; r0 < tokens; r0 += rows_per_launch) {
        const int64_t rows = std::min(rows_per_launch, tokens - r0);
        const int64_t total_ws = rows * wpr;
        const int64_t waves = (total_ws + QUANT_UNROLL - 1) / QUANT_UNROLL;
        const unsigned grid = (unsigned)std::min<int64_t>((waves + QUANT_THREADS / 64 - 1) / (QUANT_THREADS / 64), max_blocks);
        const uint16_t *xs = static_cast<const uint16_t *>(x) + r0 * k;
        const int32_t *ds = dst_idx + r0 * topk;
        if (vec)
            hipLaunchKernelGGL((mx_quant_rows_kernel<FMT, RND, HWCVT, true, false, true>), dim3(grid), dim3(QUANT_THREADS), 0,
                               stream, xs, out, out + pbytes, (int)rows, (int)k, (int)nblk, (int)sld, (int)row_bytes, (int)wpr,
                               (int)total_ws, ds, topk, (int)row_bytes, out_rows);
        else
            hipLaunchKernelGGL((mx_quant_rows_kernel<FMT, RND, HWCVT, false, false, true>), dim3(grid), dim3(QUANT_THREADS), 0,
                               stream, xs, out, out + pbytes, (int)rows, (int)k, (int)nblk, (int)sld, (int)row_bytes, (int)wpr,
                               (int)total_ws, ds, topk, (int)row_bytes, out_rows);
        int rc = launch_status("mx_quant_rows_kernel (scatter)");
        if (rc) return rc;
    }
    return CCH_OK;
}

// Library switch "quant_integer_encoder": the E4M3 round-to-nearest-even quantiser runs through the
// integer encoder instead of the hardware conversion, so that the two can be compared bit for bit
// on the device.
static std::atomic<int> g_quant_integer_encoder{0};
bool quant_set_option(const char *name, int value)
{
    if (strcmp(name, "quant_integer_encoder") != 0) return false;
    g_quant_integer_encoder.store(value);
    return true;
}

int quant_scatter(const void *x, const int32_t *expanded_row_idx, void *packed_out, int64_t out_rows, int64_t row_pitch, int64_t tokens, int64_t k, int top_k,
                  int fmt, int rounding, void *stream);

}  // namespace cch

extern "C" int cch_mx_quant_scatter_packed(const void *x, const int32_t *expanded_row_idx, void *packed_out, int64_t tokens,
                                           int64_t k, int top_k, int fmt, int rounding, void *stream)
{
    return cch_mx_quant_scatter_packed_rows(x, expanded_row_idx, packed_out, 0x7FFFFFFF, tokens, k, top_k, fmt, rounding, stream);
}

extern "C" int cch_mx_quant_scatter_packed_rows(const void *x, const int32_t *expanded_row_idx, void *packed_out, int64_t out_rows,
                                                int64_t tokens, int64_t k, int top_k, int fmt, int rounding, void *stream)
{
    return cch::quant_scatter(x, expanded_row_idx, packed_out, out_rows, 0, tokens, k, top_k, fmt, rounding, stream);
}

// The same with rows `row_pitch` bytes apart (0: back to back; otherwise no less than a row).
int cch::quant_scatter(const void *x, const int32_t *expanded_row_idx, void *packed_out, int64_t out_rows, int64_t row_pitch, int64_t tokens, int64_t k,
                       int top_k, int fmt, int rounding, void *stream)
{
    CCH_REQUIRE(out_rows >= 0, "cch_mx_quant_scatter_packed: out_rows=%lld", (long long)out_rows);
    const int orows = (int)std::min<int64_t>(out_rows, 0x7FFFFFFF);
    CCH_REQUIRE(tokens >= 0 && k >= 0, "cch_mx_quant_scatter_packed: negative shape tokens=%lld k=%lld", (long long)tokens,
                (long long)k);
    CCH_REQUIRE(k < (int64_t)1 << 30, "cch_mx_quant_scatter_packed: k=%lld too large", (long long)k);
    CCH_REQUIRE(top_k >= 0 && top_k <= QUANT_MAX_TOPK, "cch_mx_quant_scatter_packed: top_k=%d outside 0..%d", top_k,
                QUANT_MAX_TOPK);
    CCH_REQUIRE(rounding == CCH_ROUND_RNE || rounding == CCH_ROUND_LUT, "cch_mx_quant_scatter_packed: rounding %d", rounding);
    if (tokens == 0 || k == 0 || top_k == 0) return CCH_OK;  // as the reference: nothing to do
    CCH_REQUIRE(x && expanded_row_idx && packed_out, "cch_mx_quant_scatter_packed: null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool lut = rounding == CCH_ROUND_LUT;
    switch (fmt) {
        case CCH_FMT_E4M3:
            return lut ? launch_scatter<CCH_FMT_E4M3, CCH_ROUND_LUT, false>(x, expanded_row_idx, packed_out, row_pitch, tokens, k, top_k, orows, s)
                       : launch_scatter<CCH_FMT_E4M3, CCH_ROUND_RNE, true>(x, expanded_row_idx, packed_out, row_pitch, tokens, k, top_k, orows, s);
        case CCH_FMT_E5M2:
            return lut ? launch_scatter<CCH_FMT_E5M2, CCH_ROUND_LUT, false>(x, expanded_row_idx, packed_out, row_pitch, tokens, k, top_k, orows, s)
                       : launch_scatter<CCH_FMT_E5M2, CCH_ROUND_RNE, true>(x, expanded_row_idx, packed_out, row_pitch, tokens, k, top_k, orows, s);
        case CCH_FMT_E2M1:
            return lut ? launch_scatter<CCH_FMT_E2M1, CCH_ROUND_LUT, false>(x, expanded_row_idx, packed_out, row_pitch, tokens, k, top_k, orows, s)
                       : launch_scatter<CCH_FMT_E2M1, CCH_ROUND_RNE, true>(x, expanded_row_idx, packed_out, row_pitch, tokens, k, top_k, orows, s);
        case CCH_FMT_E1M2:  // no hardware conversion for this format: integer encoder for both rules
            return lut ? launch_scatter<CCH_FMT_E1M2, CCH_ROUND_LUT, false>(x, expanded_row_idx, packed_out, row_pitch, tokens, k, top_k, orows, s)
                       : launch_scatter<CCH_FMT_E1M2, CCH_ROUND_RNE, false>(x, expanded_row_idx, packed_out, row_pitch, tokens, k, top_k, orows, s);
        default:
            return fail(CCH_EINVAL, "cch_mx_quant_scatter_packed: unknown format %d", fmt);
    }
}

extern "C" int cch_mx_quant_rows(const void *x, void *payload, void *scales, int64_t m, int64_t k, int fmt,
                                 int rounding, void *stream)
{
    using namespace cch;
    CCH_REQUIRE(m >= 0 && k >= 0, "cch_mx_quant_rows: negative shape m=%lld k=%lld", (long long)m, (long long)k);
    CCH_REQUIRE(k < (int64_t)1 << 30, "cch_mx_quant_rows: k=%lld too large", (long long)k);
    CCH_REQUIRE(rounding == CCH_ROUND_RNE || rounding == CCH_ROUND_LUT, "cch_mx_quant_rows: rounding %d", rounding);
    if (m == 0 || k == 0) return CCH_OK;
    CCH_REQUIRE(x && payload && scales, "cch_mx_quant_rows: null pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool lut = rounding == CCH_ROUND_LUT;
    switch (fmt) {
        case CCH_FMT_E4M3:
            if (!lut && g_quant_integer_encoder.load())   // cross-check of the hardware conversion on the device
                return launch_rows<CCH_FMT_E4M3, CCH_ROUND_RNE, false>(x, payload, scales, m, k, s);
            return lut ? launch_rows<CCH_FMT_E4M3, CCH_ROUND_LUT, false>(x, payload, scales, m, k, s)
                       : launch_rows<CCH_FMT_E4M3, CCH_ROUND_RNE, true>(x, payload, scales, m, k, s);
        case CCH_FMT_E5M2:
            return lut ? launch_rows<CCH_FMT_E5M2, CCH_ROUND_LUT, false>(x, payload, scales, m, k, s)
                       : launch_rows<CCH_FMT_E5M2, CCH_ROUND_RNE, true>(x, payload, scales, m, k, s);
        case CCH_FMT_E2M1:
            return lut ? launch_rows<CCH_FMT_E2M1, CCH_ROUND_LUT, false>(x, payload, scales, m, k, s)
                       : launch_rows<CCH_FMT_E2M1, CCH_ROUND_RNE, true>(x, payload, scales, m, k, s);
        case CCH_FMT_E1M2:  // no hardware conversion for this format: integer encoder for both rules
            return lut ? launch_rows<CCH_FMT_E1M2, CCH_ROUND_LUT, false>(x, payload, scales, m, k, s)
                       : launch_rows<CCH_FMT_E1M2, CCH_ROUND_RNE, false>(x, payload, scales, m, k, s);
        default:
            return fail(CCH_EINVAL, "cch_mx_quant_rows: unknown format %d", fmt);
    }
}

extern "C" int cch_mx_quant_b(const void *b, void *payload, void *scales, int64_t k, int64_t n, int fmt, int rounding,
                              int trans_b, void *stream)
{
    using namespace cch;
    CCH_REQUIRE(k >= 0 && n >= 0, "cch_mx_quant_b: negative shape");
    CCH_REQUIRE(k % 64 == 0 && n % 2 == 0, "cch_mx_quant_b: needs k %% 64 == 0 and n %% 2 == 0 (k=%lld n=%lld)",
                (long long)k, (long long)n);
    CCH_REQUIRE(k / 32 <= 65535 && k * n < ((int64_t)1 << 40), "cch_mx_quant_b: shape too large");
    CCH_REQUIRE(rounding == CCH_ROUND_RNE || rounding == CCH_ROUND_LUT, "cch_mx_quant_b: rounding %d", rounding);
    CCH_REQUIRE(trans_b == 0 || trans_b == 1, "cch_mx_quant_b: trans_b %d", trans_b);
    if (k == 0 || n == 0) return CCH_OK;
    CCH_REQUIRE(b && payload && scales, "cch_mx_quant_b: null pointer");
    CCH_REQUIRE(aligned(b, 4) && aligned(payload, 2), "cch_mx_quant_b: misaligned pointer");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool lut = rounding == CCH_ROUND_LUT;
    switch (fmt) {
        case CCH_FMT_E4M3:
            return lut ? launch_b<CCH_FMT_E4M3, CCH_ROUND_LUT>(b, payload, scales, k, n, trans_b, s)
                       : launch_b<CCH_FMT_E4M3, CCH_ROUND_RNE>(b, payload, scales, k, n, trans_b, s);
        case CCH_FMT_E5M2:
            return lut ? launch_b<CCH_FMT_E5M2, CCH_ROUND_LUT>(b, payload, scales, k, n, trans_b, s)
                       : launch_b<CCH_FMT_E5M2, CCH_ROUND_RNE>(b, payload, scales, k, n, trans_b, s);
        case CCH_FMT_E2M1:
            return lut ? launch_b<CCH_FMT_E2M1, CCH_ROUND_LUT>(b, payload, scales, k, n, trans_b, s)
                       : launch_b<CCH_FMT_E2M1, CCH_ROUND_RNE>(b, payload, scales, k, n, trans_b, s);
        case CCH_FMT_E1M2:
            return lut ? launch_b<CCH_FMT_E1M2, CCH_ROUND_LUT>(b, payload, scales, k, n, trans_b, s)
                       : launch_b<CCH_FMT_E1M2, CCH_ROUND_RNE>(b, payload, scales, k, n, trans_b, s);
        default:
            return fail(CCH_EINVAL, "cch_mx_quant_b: unknown format %d", fmt);
    }
}
