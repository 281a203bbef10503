// Weight-streaming MFMA GEMM for few rows per group (decode steps, small dense layers): the same operand kinds,
// layouts and epilogues as the tiled kernel, for problems that its 256 x 256 tiles leave most of the chip idle on.
//
// Such a problem is bound by the weights' way from HBM, and where it is small by latencies.  So the work is cut along
// N and K instead of M: a workgroup computes a tile of 32 rows x 64 columns, and its W waves split K into contiguous
// ranges.  Each wave is a pipeline of its own - it fetches a chunk (128 bytes of K: 4 KiB of A, 8 KiB of B) straight into
// its private piece of LDS, waits for it alone, takes the fragments into registers, requests the next chunk into the same
// place and only then issues the matrix instructions - so the K loop has no barrier, and 8 to 12 waves per CU keep 64 to
// 96 KiB of weights in flight (HBM's latency times its bandwidth is about 24 KiB per CU).  At the end the waves' partial
// sums meet in LDS and all threads finish the tile.  Workgroups are not persistent: the dispatcher deals them to whichever
// CU is free, and the up to three that share a CU hide each other's group lookup, first requests and epilogue.
// Measured (MXFP8, weights in the Infinity Cache): 16 x 2048 x 7168 8.8 us (18.2 on one 256 x 256 tile per CU), 64 x 7168 x 4096
// 18 us (44); int8 64 x 4096 x 8192 9 us (25).
//
// Tiles of one group are numbered row tile first, and runs of four consecutive tiles go to one XCD: they share weight
// lines (row tiles: the same panel; [K, N] columns: the other parts of a 128-byte line) through its L2.
#pragma once
#include <algorithm>
#include <atomic>

#include "gemm_finish.h"
#include "gemm_stream.h"

namespace cch {

template <int KIND, int EPI, int FMT, int TB, int W>
__global__ __launch_bounds__(W * 64, W == 4 ? 3 : 2) void gemm_stream_kernel(GemmProblem p)
{
    using KT = KindTraits<KIND>;
    using Acc = typename KT::Acc;
    constexpr bool MX = KIND != KIND_I8;
    constexpr bool SWIGLU = EPI == EPI_DEQUANT_SWIGLU || EPI == EPI_SWIGLU;
    constexpr bool DEQ = EPI == EPI_DEQUANT || EPI == EPI_DEQUANT_SWIGLU;
    constexpr int EPB = KT::ELEMS_PER_BYTE;
    constexpr int TM = STREAM_TM;
    constexpr int TN_OUT = SWIGLU ? STREAM_TN / 2 : STREAM_TN;   // SwiGLU: 32 gate columns, then the 32 up columns beside them
    constexpr int STAGE = STREAM_STAGE;                          // A: 32 rows x 128 B, then B: 8 KiB
    constexpr int B_OFF = 4096;
    constexpr int NSP = MX ? EPB : 0;                            // scale registers per 32 rows or columns and chunk, two K64 blocks each
    constexpr int CBSZ = FMT == CCH_FMT_E2M1 ? 4 : (FMT == CCH_FMT_E5M2 ? 1 : 0);

    touch_arguments(p);
    const int lane = threadIdx.x & 63;
    const int wave = uniform(threadIdx.x >> 6);
    const int r = lane & 31, g = lane >> 5;
    const int n_tiles = (p.n_out + TN_OUT - 1) / TN_OUT;
    const int tile = stream_tile_of((int)blockIdx.x);

    // ---- which tile is this: group e, rows m0 .. m0 + rows - 1, column tile ct
    int e = 0, m0 = 0, rows = 0, ct = 0;
    if (p.group_sizes == nullptr) {
        const int rt = (p.T + TM - 1) / TM;
        if (tile >= rt * n_tiles) return;
        ct = tile / rt;
        m0 = (tile - ct * rt) * TM;
        rows = min(TM, p.T - m0);
    } else {
        const GroupPlace at = find_place(p, tile, TM, n_tiles);
        zero_rest<EPI>(p, at.used);
        if (!at.found) return;
        e = at.e;
        ct = at.rel / at.rt;
        m0 = at.lo + (at.rel - ct * at.rt) * TM;
        rows = min(TM, at.hi - m0);
    }
    const int j0 = ct * TN_OUT;

    // ---- what the epilogue will need, requested before the K loop: item = 8 neighbouring output columns of one row
    constexpr int IPR = TN_OUT / 8;                                          // items per row
    constexpr int NITEM = (TM * IPR + W * 64 - 1) / (W * 64);                // items per thread
    const int icol = j0 + (int)(threadIdx.x % IPR) * 8;                      // (the same column for all of a thread's items)
    float ch[SWIGLU ? 16 : 8] = {}, tok[NITEM] = {};
    int mapped[NITEM];
    if constexpr (DEQ) {
        const float *pc = p.per_ch + (size_t)e * p.N + min(icol, p.n_out - 8);
#pragma unroll
        for (int x = 0; x < 8; x++) {
            ch[x] = pc[x];
            if constexpr (SWIGLU) ch[8 + x] = pc[p.n_out + x];
        }
    }
#pragma unroll
    for (int it = 0; it < NITEM; it++) {
        const int row = min((int)(threadIdx.x + it * W * 64) / IPR, rows - 1);
        if constexpr (DEQ) tok[it] = p.per_tok[m0 + row];
        mapped[it] = row;
        if constexpr (EPI == EPI_PLAIN) {
            if (p.out_row_map) mapped[it] = p.out_row_map[m0 + row];
        }
    }

    // ---- operands
    const int lda = p.K / EPB;
    const int pa = p.a_pitch ? (int)p.a_pitch : lda;
    const int psa = p.sa_pitch ? (int)p.sa_pitch : p.sld;
    const int ldb = TB ? lda : p.N / EPB;
    const Rsrc rs_a = make_rsrc(p.a + (size_t)m0 * pa, (uint32_t)(rows - 1) * (uint32_t)pa + (uint32_t)lda);
    const Rsrc rs_b = make_rsrc(p.b + (size_t)e * p.b_stride, (uint32_t)p.N * (uint32_t)lda);
    const uint32_t lds_base = (uint32_t)uniform((int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem);
    const uint32_t stage = lds_base + (uint32_t)(wave * STAGE);

    // Panels of K-contiguous rows: 8 rows of 128 B per request; lane l lands at row l/8, chunk position l%8 and fetches
    // chunk (l%8) ^ swizzle(row), which for an odd request is the even request's chunk ^ 4.
    const uint32_t kc0 = (uint32_t)(((lane & 7) ^ (lane >> 4)) << 4), kc1 = kc0 ^ 64u;
    const uint32_t a_lane = (uint32_t)(lane >> 3) * (uint32_t)pa;
    // B, [K, N]: a chunk is 128*EPB K-rows of 64/EPB bytes; one request fills 16*EPB of them.  Lane l lands at K-row
    // l / (4/EPB), chunk position l % (4/EPB); the 16-byte chunks of a row are swizzled by a row bit so that the
    // transposing reads below touch all banks once.
    uint32_t b_lane;
    if constexpr (TB) {
        b_lane = (uint32_t)(lane >> 3) * (uint32_t)lda + (uint32_t)j0 * (uint32_t)lda;
    } else if constexpr (EPB == 1) {
        const int chunk = (lane & 3) ^ (2 * ((lane >> 4) & 1));
        b_lane = (uint32_t)(lane >> 2) * (uint32_t)ldb + (uint32_t)(j0 + (SWIGLU ? (chunk >> 1) * p.n_out + (chunk & 1) * 16 : chunk * 16));
    } else {
        const int chunk = (lane & 1) ^ ((lane >> 4) & 1);
        b_lane = (uint32_t)(lane >> 1) * (uint32_t)ldb + (uint32_t)(j0 + chunk * (SWIGLU ? p.n_out : 32)) / 2u;
    }
    const uint32_t b_up = SWIGLU ? (uint32_t)(p.n_out - 32) * (uint32_t)lda : 0u;   // [N, K]: from row 32 on the up columns

    auto request = [&](int c) {
        const uint32_t koff = (uint32_t)c * BKB;
        const bool ok0 = (int)(koff + kc0) < lda, ok1 = (int)(koff + kc1) < lda;   // the row's last piece: lanes past its end fetch nothing
        const uint32_t va0 = ok0 ? a_lane + kc0 + koff : NO_FETCH, va1 = ok1 ? a_lane + kc1 + koff : NO_FETCH;
        static_for<4>([&](auto q_c) {
            constexpr int q = decltype(q_c)::value;
            const uint32_t v = (q & 1) ? va1 : va0, d = (uint32_t)(q * 8) * (uint32_t)pa;
            load16_to_lds_at<q * 1024>(rs_a, ((q & 1) ? ok1 : ok0) ? v + d : NO_FETCH, 0u, stage);
        });
        if constexpr (TB) {
            const uint32_t vb0 = b_lane + kc0 + koff, vb1 = b_lane + kc1 + koff;
            static_for<8>([&](auto q_c) {
                constexpr int q = decltype(q_c)::value;
                const uint32_t d = (uint32_t)(q * 8) * (uint32_t)lda + (q >= 4 ? b_up : 0u);
                load16_to_lds_at<B_OFF + q * 1024>(rs_b, ((q & 1) ? ok1 : ok0) ? ((q & 1) ? vb1 : vb0) + d : NO_FETCH, 0u, stage);
            });
        } else {
            const uint32_t vb = b_lane + (uint32_t)c * (uint32_t)(BKB * EPB) * (uint32_t)ldb;   // K-rows past the last lie past the descriptor
            static_for<8>([&](auto q_c) {
                constexpr int q = decltype(q_c)::value;
                load16_to_lds_at<B_OFF + q * 1024>(rs_b, vb + (uint32_t)(q * 16 * EPB) * (uint32_t)ldb, 0u, stage);
            });
        }
    };

    // ---- scales: straight to registers, one E8M0 pair (a K64 block) per 16 bits
    __amdgpu_buffer_rsrc_t rs_sa, rs_sb;
    uint32_t sa_off = 0, sb_off[2] = {};
    bool sa4 = false, sb4 = false;   // all scale rows start on 4-byte boundaries: two K64 blocks per load
    const int nblk = (p.K + 31) >> 5;
    if constexpr (MX) {
        // (the array's size is rounded up to the dword that its last scale lies in: the bounds check drops a 16-bit load from
        // a dword that the size cuts)
        rs_sa = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(p.sa), 0, (int)(((uint32_t)(p.T - 1) * (uint32_t)psa + (uint32_t)p.sld + 3u) & ~3u), 0x00020000);
        rs_sb = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(p.sb) + (size_t)e * p.sb_stride, 0, (int)((uint32_t)p.N * (uint32_t)p.sld), 0x00020000);
        sa4 = (psa & 3) == 0;
        sb4 = TB && (p.sld & 3) == 0 && (p.sb_stride & 3) == 0;
        sa_off = (uint32_t)(m0 + r) * (uint32_t)psa;
#pragma unroll
        for (int j = 0; j < 2; j++) {
            const uint32_t col = (uint32_t)(j0 + r + (SWIGLU ? j * p.n_out : j * 32));
            sb_off[j] = TB ? col * (uint32_t)p.sld : col * 2u;
        }
    }
    // (raw_hi holds the second K64 block where a load brought one of them; nothing is combined before the wait for the chunk)
    uint32_t raw[NSP > 0 ? NSP : 1][3] = {}, raw_hi[NSP > 0 ? NSP : 1][3] = {};   // rows of A, columns 0..31 and 32..63 of B
    auto load_scales = [&](int c) {
        if constexpr (MX) {
#pragma unroll
            for (int d = 0; d < NSP; d++) {
                const uint32_t k64 = (uint32_t)(c * 2 * EPB + 2 * d);
                if (sa4) {
                    raw[d][0] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_sa, (int)(sa_off + k64 * 2u), 0, 0);
                } else {
                    raw[d][0] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs_sa, (int)(sa_off + k64 * 2u), 0, 0);
                    raw_hi[d][0] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs_sa, (int)(sa_off + k64 * 2u + 2u), 0, 0);
                }
                if (TB && sb4) {
#pragma unroll
                    for (int j = 0; j < 2; j++) raw[d][1 + j] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rs_sb, (int)(sb_off[j] + k64 * 2u), 0, 0);
                } else {
                    const uint32_t at = TB ? k64 * 2u : k64 * (uint32_t)p.N * 2u, next = TB ? 2u : (uint32_t)p.N * 2u;
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        raw[d][1 + j] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs_sb, (int)(sb_off[j] + at), 0, 0);
                        raw_hi[d][1 + j] = (uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rs_sb, (int)(sb_off[j] + at + next), 0, 0);
                    }
                }
            }
        }
    };

    // ---- fragment addresses (as in the tiled kernel): lane (r, g) feeds 16-byte chunks ks*4 + g and ks*4 + 2 + g
    uint32_t fr[4], fbt[2];
#pragma unroll
    for (int x = 0; x < 4; x++) fr[x] = stage + (uint32_t)r * BKB + ((((uint32_t)((x >> 1) * 4 + (x & 1) * 2 + g)) ^ swizzle_of_row(r)) << 4);
    {
        const int q = lane >> 4, i = lane & 15;
        const uint32_t at = EPB == 2 ? (uint32_t)(32 * (q >> 1) + i) * 32u + (uint32_t)(i >> 3) * 16u + (uint32_t)(q & 1) * 8u
                                     : (uint32_t)(16 * (q >> 1) + (i >> 1)) * 64u + (uint32_t)((q & 1) ^ (2 * (i >> 3))) * 16u + (uint32_t)(i & 1) * 8u;
#pragma unroll
        for (int j = 0; j < 2; j++) fbt[j] = stage + (uint32_t)B_OFF + (at ^ ((uint32_t)j << (EPB == 2 ? 4 : 5)));
    }

    Acc acc[2] = {(Acc)(0), (Acc)(0)};

    // ---- K loop of this wave: chunks c0 .. c1 - 1
    const int chunks = (lda + BKB - 1) / BKB;
    const int c0 = wave * chunks / W, c1 = (wave + 1) * chunks / W;
    if (c0 < c1) {
        request(c0);
        load_scales(c0);
    }
    for (int c = c0; c < c1; c++) {
        CCH_WAIT_VM(0);
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        uint32_t sc[NSP > 0 ? NSP : 1][3];
        if constexpr (MX) {
            // this lane's bytes (block g of either K64 block) in bytes 0 and 2; those of blocks past K cleared: their
            // payload is zero, and a zero byte keeps the product zero where a stray 0xFF (NaN) would not
#pragma unroll
            for (int d = 0; d < NSP; d++) {
                const int b0 = (c * 2 * EPB + 2 * d) * 2 + g;
                const uint32_t keep = (b0 < nblk ? 0xFFu : 0u) | (b0 + 2 < nblk ? 0xFF0000u : 0u);
#pragma unroll
                for (int s = 0; s < 3; s++) {
                    const bool whole = s == 0 ? sa4 : TB && sb4;
                    sc[d][s] = ((whole ? raw[d][s] : raw[d][s] | raw_hi[d][s] << 16) >> (8 * g)) & keep;
                }
            }
        }
        v8i fa[2], fb[2][2];
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            {
                const v4i lo = lds_read16_abs(fr[2 * ks]), hi = lds_read16_abs(fr[2 * ks + 1]);
                fa[ks] = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
            }
#pragma unroll
            for (int j = 0; j < 2; j++) {
                if constexpr (TB) {
                    const v4i lo = lds_read16_abs(fr[2 * ks] + (uint32_t)(B_OFF + j * 4096)), hi = lds_read16_abs(fr[2 * ks + 1] + (uint32_t)(B_OFF + j * 4096));
                    fb[j][ks] = (v8i){lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
                } else {
                    typedef __attribute__((address_space(3))) v2i *LdsV2;
                    const uint32_t at = fbt[j] + (uint32_t)(ks * 4096);
                    v2i t0, t1, t2, t3;
                    if constexpr (EPB == 2) {
                        t0 = __builtin_amdgcn_ds_read_tr4_b64_v2i32((LdsV2)(uintptr_t)(at));
                        t1 = __builtin_amdgcn_ds_read_tr4_b64_v2i32((LdsV2)(uintptr_t)(at + 512u));
                        t2 = __builtin_amdgcn_ds_read_tr4_b64_v2i32((LdsV2)(uintptr_t)(at + 2048u));
                        t3 = __builtin_amdgcn_ds_read_tr4_b64_v2i32((LdsV2)(uintptr_t)(at + 2560u));
                    } else {
                        t0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2)(uintptr_t)(at));
                        t1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2)(uintptr_t)(at + 512u));
                        t2 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2)(uintptr_t)(at + 2048u));
                        t3 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2)(uintptr_t)(at + 2560u));
                    }
                    fb[j][ks] = (v8i){t0[0], t0[1], t1[0], t1[1], t2[0], t2[1], t3[0], t3[1]};
                }
            }
        }
        // the chunk is in registers: its place in LDS is free for the next one
        __builtin_amdgcn_sched_barrier(0);
        CCH_WAIT_LGKM0();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
        if (c + 1 < c1) {
            request(c + 1);
            load_scales(c + 1);
        }
#pragma unroll
        for (int ks = 0; ks < 2; ks++) {
            if constexpr (KIND == KIND_F8) {
#pragma unroll
                for (int j = 0; j < 2; j++) {
                    if (ks == 0) acc[j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[0], fb[j][0], acc[j], CBSZ, CBSZ, 0, (int)sc[0][0], 0, (int)sc[0][1 + j]);
                    else acc[j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[1], fb[j][1], acc[j], CBSZ, CBSZ, 2, (int)sc[0][0], 2, (int)sc[0][1 + j]);
                }
            } else {
#pragma unroll
                for (int half = 0; half < 2; half++)
#pragma unroll
                    for (int j = 0; j < 2; j++) {
                        const v8i &a = fa[ks], &b = fb[j][ks];
                        if constexpr (KIND == KIND_F4) {
                            const int d = ks % NSP;
                            const v8i ah = (v8i){a[4 * half], a[4 * half + 1], a[4 * half + 2], a[4 * half + 3], 0, 0, 0, 0};
                            const v8i bh = (v8i){b[4 * half], b[4 * half + 1], b[4 * half + 2], b[4 * half + 3], 0, 0, 0, 0};
                            if (half == 0) acc[j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(ah, bh, acc[j], 4, 4, 0, (int)sc[d][0], 0, (int)sc[d][1 + j]);
                            else acc[j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(ah, bh, acc[j], 4, 4, 2, (int)sc[d][0], 2, (int)sc[d][1 + j]);
                        } else {
                            const v4i ah = (v4i){a[4 * half], a[4 * half + 1], a[4 * half + 2], a[4 * half + 3]};
                            const v4i bh = (v4i){b[4 * half], b[4 * half + 1], b[4 * half + 2], b[4 * half + 3]};
                            acc[j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ah, bh, acc[j], 0, 0, 0);
                        }
                    }
            }
        }
    }

    // ---- the waves' partial sums: [row][64 columns] of 32 bits in each wave's own stage (nothing of it is in use any more)
    {
        const uint32_t at = (uint32_t)(wave * STAGE) + (uint32_t)(g * 4) * 256u + (uint32_t)r * 4u;
        typedef typename std::remove_reference<decltype(acc[0][0])>::type Elem;
#pragma unroll
        for (int j = 0; j < 2; j++)
#pragma unroll
            for (int x = 0; x < 16; x++) *reinterpret_cast<Elem *>(smem + at + (uint32_t)((x >> 2) * 8 + (x & 3)) * 256u + (uint32_t)j * 128u) = acc[j][x];
    }
    __syncthreads();

    typedef typename std::conditional<KIND == KIND_I8, v4i, __attribute__((ext_vector_type(4))) float>::type Sum4;
    auto sum8 = [&](int row, int col, float (&v)[8]) {
        Sum4 s0 = *reinterpret_cast<const Sum4 *>(smem + (uint32_t)row * 256u + (uint32_t)col * 4u);
        Sum4 s1 = *reinterpret_cast<const Sum4 *>(smem + (uint32_t)row * 256u + (uint32_t)col * 4u + 16u);
#pragma unroll
        for (int w = 1; w < W; w++) {
            s0 += *reinterpret_cast<const Sum4 *>(smem + (uint32_t)(w * STAGE) + (uint32_t)row * 256u + (uint32_t)col * 4u);
            s1 += *reinterpret_cast<const Sum4 *>(smem + (uint32_t)(w * STAGE) + (uint32_t)row * 256u + (uint32_t)col * 4u + 16u);
        }
#pragma unroll
        for (int x = 0; x < 4; x++) {
            v[x] = (float)s0[x];
            v[4 + x] = (float)s1[x];
        }
    };
    with_output_kind<EPI>(p, [&](auto step_c, auto half_c) {
#pragma unroll
        for (int it = 0; it < NITEM; it++) {
            const int item = (int)threadIdx.x + it * W * 64;
            const int row = item / IPR, lcol = (item % IPR) * 8;
            if (TM * IPR % (W * 64) != 0 && row >= TM) break;
            float v[8], up[8] = {};
            sum8(row, lcol, v);
            if constexpr (SWIGLU) sum8(row, 32 + lcol, up);
            finish8<EPI, decltype(step_c)::value != 0>(v, up, ch, tok[it]);
            store8<EPI, decltype(half_c)::value != 0>(p, v, row < rows && icol + 8 <= p.n_out, m0 + row, mapped[it], icol);
        }
    });
}

template <int KIND, int EPI, int FMT, int TB, int W>
static int launch_stream_w(const GemmProblem &p, hipStream_t stream)
{
    constexpr int lds = W * STREAM_STAGE;
    auto kern = gemm_stream_kernel<KIND, EPI, FMT, TB, W>;
    if constexpr (lds > 65536) {
        // set once per device and kernel; setting it twice from two threads is harmless
        static std::atomic<uint64_t> attr_set{0};
        int dev = 0;
        CCH_HIP(hipGetDevice(&dev));
        const uint64_t dev_bit = (uint64_t)1 << (dev & 63);
        if (dev >= 64 || !(attr_set.load(std::memory_order_acquire) & dev_bit)) {
            CCH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
            attr_set.fetch_or(dev_bit, std::memory_order_release);
        }
    }
    constexpr int tn_out = (EPI == EPI_DEQUANT_SWIGLU || EPI == EPI_SWIGLU) ? STREAM_TN / 2 : STREAM_TN;
    const int64_t tiles = row_tiles_bound(p, STREAM_TM) * ((p.n_out + tn_out - 1) / tn_out);
    hipLaunchKernelGGL(kern, dim3((unsigned)stream_grid(tiles)), dim3(W * 64), lds, stream, p);
    return launch_status("gemm_stream_kernel");
}

template <int KIND, int EPI, int FMT, int TB>
int launch_stream_t(const GemmProblem &p, int waves, hipStream_t stream)
{
    return waves == 8 ? launch_stream_w<KIND, EPI, FMT, TB, 8>(p, stream) : launch_stream_w<KIND, EPI, FMT, TB, 4>(p, stream);
}

}  // namespace cch
