// Mid-size MFMA GEMM: tiles of 64*MB rows x 32*JB*WN columns (64 x 128, 128 x 128, 128 x 256, 192 x 192) for problems that have too few
// 256 x 256 tiles to fill the chip, or groups of a few rows each, and too many rows to stream the weights once.
//
// 2 x WN waves, each 32*MB x 32*JB outputs, keep a ring of stages of 128 bytes of K in LDS.  With three stages a step is
//   wait for this step's stage (the younger one stays in flight) | barrier | all fragments of the step into registers, and
//   between the matrix instructions the requests of the step after the next, into the stage of the step before
// With two (128 x 128 tiles, of which the LDS of a CU then holds two) the stage just read is requested anew behind a second
// barrier.  Two workgroups of the narrow tiles share a CU and hide each other's waits, group lookup and epilogue.
// Every element is summed in the order of the 256 x 256 kernel (K ascending, one accumulator): the results are the same bits.
//
// What bounds it, measured (MXFP8 128 x 128, 512 tiles on the chip): a step of two workgroups takes 1.15 us, of which their matrix
// instructions are 0.43 us at the boost clock, the 64 KiB of requests 0.65 us alone (L2 gives 25 TB/s to such panels) and the LDS reads
// with the matrix instructions 0.72 us without requests; per product that is twice the traffic of 256 x 256 tiles, which stay ahead
// where they fill the chip.  512 x 7168 x 4096 takes 29 us (67 on 32 256 x 256 tiles), 1024 x 7168 x 4096 41 (67), int8 256 x 4096 x 1024 15
// (38); 16 groups of 24 tokens, K 7168, N 4096: 90 us (102), of 192 skewed ones: 148 us (177).
// 192 x 192 (JB 3) is four waves, one per SIMD, with a step of their own (deep_step): 3000 x 1984 x 3000 28.0 us (32.9 on 256 x 256 tiles, 35.6 on
// 128 x 128).  Its step takes 1.1 us, of which the matrix instructions are 0.48 and 0.74 with the LDS reads among them; the requests alone take 0.9:
// their latency (1.2 to 1.5 us from the Infinity Cache) over the two stages that three leave under way.  Reads and requests
// in front of the matrix instructions instead of between them cost 8 % more.
// The epilogue's choices (output type, the int8 step through half) are branches around the passes, not inside them, and the launch's arguments
// are fetched at once: a launch of one tile 5.2 -> 4.6 us on 128 x 128, 6.0 -> 5.4 on 128 x 256; int8 5932 x 512 x 5120 42.0 -> 37.3 on 128 x 128.
// Not kept: deeper rings for one workgroup per CU (five stages of 64 x 128, four of 128 x 128: -4 to +8 %), the two halves of the
// 128 x 256 workgroup alternating between memory and matrix slots as in the 256 x 256 kernel (5 % slower).
//
// Workgroups are not persistent.  The dispatcher deals workgroup b to XCD b % 8; an XCD takes runs of consecutive tiles, a
// group's tiles are numbered in blocks of eight (wide tiles four) columns, rows inside: the tiles that run on an XCD at a time
// share their panels in its L2.
#pragma once
#include <atomic>

#include "gemm_finish.h"
#include "gemm_mid.h"

namespace cch {

template <int KIND, int EPI, int FMT, int TB, int UA, int MB, int WN, int JB>
__global__ __launch_bounds__(128 * WN, JB == 3 ? 1 : 2) void gemm_mid_kernel(GemmProblem p)
{
    using KT = KindTraits<KIND>;
    using Acc = typename KT::Acc;
    constexpr bool MX = KIND != KIND_I8;
    constexpr bool SWIGLU = EPI == EPI_DEQUANT_SWIGLU || EPI == EPI_SWIGLU;
    constexpr bool DEQ = EPI == EPI_DEQUANT || EPI == EPI_DEQUANT_SWIGLU;
    constexpr int EPB = KT::ELEMS_PER_BYTE;
    constexpr int NW = 2 * WN, TM = 64 * MB, TN = mid_cols(WN, JB);
    static_assert(JB == 2 || (TB && EPI == EPI_PLAIN), "96 columns per wave: whole gate and up blocks, K-rows of whole requests and one column per lane need 64");
    constexpr bool DEEP = JB == 3;                 // one wave per SIMD: see the step
    constexpr int TN_OUT = SWIGLU ? TN / 2 : TN;   // SwiGLU: the tile's gate columns, then their up columns
    // A wave's 32-column blocks of the panel start WC * wn columns in and lie JC apart (SwiGLU: one gate, one up).
    constexpr int WC = SWIGLU ? 32 : 32 * JB, JC = SWIGLU ? TN / 2 : 32;
    constexpr int S = mid_stages(MB, WN);                  // stages of the ring
    constexpr int A_BYTES = TM * BKB, STAGE = mid_stage_bytes(MB, WN, JB);
    constexpr int SC_OFF = S * STAGE, SC_BUF = (TM + TN) * 16;   // MX scales: buffers of 16 bytes per row and column
    constexpr int NSP = MX ? EPB : 0;                      // scale dwords per row and step
    // steps per 16-byte scale fetch; rows that can start 2 bytes past a dword leave room for the shift
    constexpr int SPG = mid_steps_per_scales(KIND, UA);
    constexpr int NSB = mid_scale_buffers(S, SPG);
    constexpr int CBSZ = FMT == CCH_FMT_E2M1 ? 4 : (FMT == CCH_FMT_E5M2 ? 1 : 0);
    constexpr int NA = TM / 8 / NW, NBQ = TN / 8 / NW;     // 1 KiB requests per wave and step: A, B
    constexpr int NREQ = NA + NBQ;
    constexpr int SINK_OFF = SC_OFF + NSB * SC_BUF;        // (MX) 1 KiB where scale requests that are not due land
    constexpr uint32_t FAR = 0x80000000u;                  // a lane offset past every descriptor that row offsets can be added to

    constexpr int RUN = mid_run(TN);
    constexpr int NSR = MX ? (TM / 64 + TN / 64 + NW - 1) / NW : 0;   // scale requests per wave and step

    touch_arguments(p);
    const int lane = threadIdx.x & 63;
    const int wave = uniform(threadIdx.x >> 6);
    const int wm = wave / WN, wn = wave % WN;
    const int r = lane & 31, g = lane >> 5;
    const int n_tiles = (p.n_out + TN_OUT - 1) / TN_OUT;

    // ---- which tile is this: group e, rows m0 .. m0 + rows - 1, first output column j0
    int e = 0, lo = 0, hi = p.T, rel, rt;
    if (p.group_sizes == nullptr) {
        rt = (p.T + TM - 1) / TM;
        rel = mid_tile_of((int)blockIdx.x, rt * n_tiles, mid_round(TN));
        if (rel < 0) return;
    } else if (MB == 1 && p.tail_cus) {
        const GroupPlace at = find_tail<SWIGLU>(p, (int)blockIdx.x, TM, n_tiles, mid_round(TN));
        if (!at.found) return;
        e = at.e;
        lo = at.lo;
        hi = at.hi;
        rel = at.rel;
        rt = at.rt;
    } else {
        const GroupPlace all = find_place(p, -1, TM, n_tiles);
        zero_rest<EPI>(p, all.used);
        const int tile = mid_tile_of((int)blockIdx.x, all.total, mid_round(TN));
        if (tile < 0) return;
        const GroupPlace at = find_place(p, tile, TM, n_tiles);
        e = at.e;
        lo = at.lo;
        hi = at.hi;
        rel = at.rel;
        rt = at.rt;
    }
    const int cb = rel / (rt * RUN), in = rel - cb * rt * RUN, cw = min(RUN, n_tiles - cb * RUN);
    const int row_tile = in / cw;
    const int m0 = lo + row_tile * TM, rows = min(TM, hi - m0);
    const int j0 = (cb * RUN + in - row_tile * cw) * TN_OUT;

    // ---- operands and this lane's source offsets
    constexpr int CPR = TN / EPB / 16, RPR = 64 / CPR;     // [K, N] panel: 16-byte chunks per K-row, K-rows per request
    auto b_swizzle = [](int row) { return EPB == 1 ? (CPR == 8 ? 2 * ((row >> 1) & 3) : 2 * (row & 7)) : (CPR == 4 ? (row >> 2) & 3 : (row >> 1) & 7); };
    const int lda = p.K / EPB;
    const int pa = p.a_pitch ? (int)p.a_pitch : lda;
    const int psa = p.sa_pitch ? (int)p.sa_pitch : p.sld;
    const int ldb = TB ? lda : p.N / EPB;
    const Rsrc rs_a = make_rsrc(p.a + (size_t)m0 * pa, (uint32_t)(rows - 1) * (uint32_t)pa + (uint32_t)lda);
    const Rsrc rs_b = make_rsrc(p.b + (size_t)e * p.b_stride, (uint32_t)p.N * (uint32_t)lda);
    const uint32_t lds_base = (uint32_t)uniform((int)(uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t *)smem);

    // K-contiguous panels: request q of 8 rows; lane l lands at row l/8, chunk position l%8 and fetches chunk (l%8) ^ swizzle,
    // which for an odd request is the even request's chunk ^ 4.
    const uint32_t kc0 = (uint32_t)(((lane & 7) ^ (lane >> 4)) << 4), kc1 = kc0 ^ 64u;   // (a wave's first row is a multiple of 16)
    const uint32_t a_lane = (uint32_t)(wave * NA * 8 + (lane >> 3)) * (uint32_t)pa;
    // tile column c -> column of B.  SwiGLU: as long a piece of a row of [K, N] weights as there is on either side (64 or 128 bytes;
    // with gate and up blocks of 32 alternating, MXFP8 3072 x 7168 x 4096 over 16 groups took 163 us on 128 x 256 tiles and 215 on
    // 128 x 128, so 158 and 208; 384 rows on 64 x 128 tiles 129, so 125)
    auto col_of = [&](int c) { return j0 + (SWIGLU ? c / JC * p.n_out + c % JC : c); };
    uint32_t b_lane, b_odd = 0;   // [K, N]: of the even and the odd requests
    if constexpr (TB) {
        b_lane = (uint32_t)(col_of(wave * NBQ * 8) + (lane >> 3)) * (uint32_t)lda;
    } else {
        // K-rows of TN / EPB bytes, CPR chunks of 16: a chunk's position is swizzled by row bits, so that the K-rows x chunks of one
        // pass of the transposing read (8 rows x 2 neighbouring chunks, FP4 16 rows x 1 chunk) touch all banks once
        // (a wave's rows start at a multiple of 16, and two requests span a period of the swizzle)
        const int kr = lane / CPR, c0 = (lane % CPR) ^ b_swizzle(kr), c1 = (lane % CPR) ^ b_swizzle(kr + RPR);
        const uint32_t row0 = (uint32_t)(wave * NBQ * RPR + kr) * (uint32_t)ldb;
        b_lane = row0 + (uint32_t)col_of(c0 * 16 * EPB) / EPB;
        b_odd = row0 + (uint32_t)col_of(c1 * 16 * EPB) / EPB;
    }
    const uint32_t lds_a = lds_base + (uint32_t)(wave * NA * 1024), lds_b = lds_base + (uint32_t)(A_BYTES + wave * NBQ * 1024);

    // Scales: requests 0 .. MB-1 of the workgroup fetch those of 64 rows of A each, the ones behind them those of 64 columns of B each
    // ([N, K]) or 1 KiB each of the group's eight K64 rows ([K/64][N][2]); wave w has requests w, w + NW, ...
    Rsrc rs_sc[NSR > 0 ? NSR : 1];
    uint32_t off_sc[NSR > 0 ? NSR : 1], step_sc[NSR > 0 ? NSR : 1], lds_sc[NSR > 0 ? NSR : 1];
    bool has_sc[NSR > 0 ? NSR : 1];
#pragma unroll
    for (int i = 0; i < NSR; i++) {
        const int at = wave + i * NW, bw = at - MB;
        rs_sc[i] = make_rsrc(nullptr, 0);
        off_sc[i] = FAR;
        step_sc[i] = 0;
        has_sc[i] = bw < TN / 64;
        lds_sc[i] = lds_base + (uint32_t)(SC_OFF + (at < MB ? at * 1024 : TM * 16 + bw * 1024));
        if (at < MB) {
            // (the array's size is rounded up to the dword that its last scale lies in, see gemm_stream_kernel.h)
            rs_sc[i] = make_rsrc(p.sa, ((uint32_t)(p.T - 1) * (uint32_t)psa + (uint32_t)p.sld + 3u) & ~3u);
            off_sc[i] = ((uint32_t)(m0 + at * 64 + lane) * (uint32_t)psa) & ~3u;
            step_sc[i] = (uint32_t)(SPG * NSP * 4);
        } else if (has_sc[i]) {
            rs_sc[i] = make_rsrc(p.sb + (size_t)e * p.sb_stride, (uint32_t)p.N * (uint32_t)p.sld);
            if constexpr (TB) {
                off_sc[i] = ((uint32_t)col_of(bw * 64 + lane) * (uint32_t)p.sld) & ~3u;
                step_sc[i] = (uint32_t)(SPG * NSP * 4);
            } else {
                constexpr int LPR = TN / 8;   // lanes per K64 row: 8 columns of 2 bytes each
                const int kr = (bw * 64 + lane) / LPR;
                if (kr < SPG * NSP * 2) off_sc[i] = ((uint32_t)kr * (uint32_t)p.N + (uint32_t)col_of((lane % LPR) * 8)) * 2u;
                step_sc[i] = (uint32_t)(SPG * NSP * 2) * (uint32_t)p.N * 2u;
            }
        }
    }
    const int steps = (lda + BKB - 1) / BKB;

    // The requests of step k into stage STG, one piece at a time (piece 0: the scale groups that are due, pieces 1 .. NREQ: 1 KiB of
    // A or B).  Requests are never skipped, so that a step is one basic block and the number in flight a constant: past the last
    // step they go against empty descriptors, and scales that are not due into a place that nobody reads.
    struct Ahead {
        Rsrc a, b, sc[NSR > 0 ? NSR : 1];
        uint32_t va0, va1, vb0, vb1, vsc[NSR > 0 ? NSR : 1], dst[NSR > 0 ? NSR : 1], la, lb;
    };
    auto ahead_of = [&](int k) {
        Ahead q;
        const bool more = k < steps;
        q.a = rs_a;
        q.b = rs_b;
        q.a[2] = more ? rs_a[2] : 0;
        q.b[2] = more ? rs_b[2] : 0;
        q.la = lds_a + (uint32_t)(k % S * STAGE);
        q.lb = lds_b + (uint32_t)(k % S * STAGE);
        const uint32_t koff = (uint32_t)k * BKB;
        const bool ok0 = (int)(koff + kc0) < lda, ok1 = (int)(koff + kc1) < lda;   // the row's last piece: lanes past its end fetch nothing
        q.va0 = ok0 ? a_lane + kc0 + koff : FAR;
        q.va1 = ok1 ? a_lane + kc1 + koff : FAR;
        if constexpr (TB) {
            q.vb0 = ok0 ? b_lane + kc0 + koff : FAR;
            q.vb1 = ok1 ? b_lane + kc1 + koff : FAR;
        } else {
            const uint32_t at = (uint32_t)k * (uint32_t)(BKB * EPB) * (uint32_t)ldb;   // (K-rows past the last lie past the descriptor)
            q.vb0 = b_lane + at;
            q.vb1 = b_odd + at;
        }
        if constexpr (MX) {
            const int grp = k / SPG;
#pragma unroll
            for (int i = 0; i < NSR; i++) {
                const bool due = k - grp * SPG == 0 && more && has_sc[i];
                q.sc[i] = rs_sc[i];
                q.sc[i][2] = due ? rs_sc[i][2] : 0;
                q.vsc[i] = off_sc[i] + (uint32_t)grp * step_sc[i];
                q.dst[i] = due ? lds_sc[i] + (uint32_t)((grp % NSB) * SC_BUF) : lds_base + (uint32_t)SINK_OFF;
            }
        }
        return q;
    };
    auto request = [&](const Ahead &n, auto piece_c) {
        constexpr int PIECE = decltype(piece_c)::value;
        if constexpr (PIECE == 0) {
            static_for<NSR>([&](auto i_c) { load16_to_lds(n.sc[decltype(i_c)::value], n.vsc[decltype(i_c)::value], 0u, n.dst[decltype(i_c)::value]); });
        } else if constexpr (PIECE <= NA) {
            constexpr int q = PIECE - 1;
            load16_to_lds_at<q * 1024>(n.a, ((q & 1) ? n.va1 : n.va0) + (uint32_t)(q * 8) * (uint32_t)pa, 0u, n.la);
        } else {
            constexpr int q = PIECE - 1 - NA;
            load16_to_lds_at<q * 1024>(n.b, ((q & 1) ? n.vb1 : n.vb0) + (uint32_t)(q * (TB ? 8 : RPR)) * (uint32_t)ldb, 0u, n.lb);
        }
    };

    // ---- fragment and scale addresses
    constexpr uint32_t ROW8 = CPR * 16 * 2 * EPB;          // [K, N] panel: bytes of 2 (FP4: 4) K-rows
    uint32_t fr_a[4], fr_b[4], fbt[2];
#pragma unroll
    for (int x = 0; x < 4; x++) {
        const uint32_t at = (uint32_t)r * BKB + ((((uint32_t)((x >> 1) * 4 + (x & 1) * 2 + g)) ^ swizzle_of_row(r)) << 4);
        fr_a[x] = lds_base + (uint32_t)(wm * 32 * MB) * BKB + at;
        fr_b[x] = lds_base + (uint32_t)A_BYTES + (uint32_t)(wn * WC) * BKB + at;
    }
    {
        const int q = lane >> 4, i = lane & 15;
        // (column blocks start at multiples of 32 columns) fp8 / int8: lane addresses K-row 16*(q/2) + i/2, chunk q & 1 of the block, half
        // i & 1; FP4: K-row 32*(q/2) + i, half q & 1 (the rows of the further reads are multiples of 8 or 16 away: the same row bits)
        const int row = EPB == 2 ? 32 * (q >> 1) + i : 16 * (q >> 1) + (i >> 1), chunk = wn * WC / (16 * EPB) + (EPB == 2 ? 0 : q & 1);
        const uint32_t at = (uint32_t)row * (CPR * 16u) + (uint32_t)(chunk ^ b_swizzle(row)) * 16u + (uint32_t)(EPB == 2 ? q & 1 : i & 1) * 8u;
#pragma unroll
        for (int j = 0; j < 2; j++) fbt[j] = lds_base + (uint32_t)A_BYTES + (at ^ (uint32_t)(j * (JC / EPB)));   // (that bit of the chunk is free)
    }
    const uint32_t rd_sa = (uint32_t)(SC_OFF + (wm * 32 * MB + r) * 16), rd_sb = (uint32_t)(SC_OFF + TM * 16) + (uint32_t)(wn * WC + r) * (TB ? 16u : 2u);
    const uint32_t ph_a = UA ? ((uint32_t)(m0 + r) * (uint32_t)psa) & 3u : 0u;
    const uint32_t ph_b = UA ? ((uint32_t)(j0 + r) * (uint32_t)p.sld) & 3u : 0u;   // (the other terms are multiples of four rows)
    const int nblk = (p.K + 31) >> 5;

    Acc acc[MB][JB];
#pragma unroll
    for (int i = 0; i < MB; i++)
#pragma unroll
        for (int j = 0; j < JB; j++) acc[i][j] = (Acc)(0);

    // ---- the pieces of a step
    uint32_t scales[DEEP ? 2 : 1][NSP > 0 ? NSP : 1][MB + JB];   // (DEEP: of odd and of even steps)
    v8i fa[MB][2], fb[JB][2];
    auto read_scales = [&](int k, uint32_t (&sc)[NSP > 0 ? NSP : 1][MB + JB]) {
        if constexpr (MX) {
            const int grp = k / SPG, ws = k - grp * SPG;
            const uint32_t buf = (uint32_t)((grp % NSB) * SC_BUF);
#pragma unroll
            for (int d = 0; d < NSP; d++) {
                const uint32_t sa_at = rd_sa + buf + (uint32_t)((ws * NSP + d) * 4);
#pragma unroll
                for (int i = 0; i < MB; i++) {
                    if constexpr (UA) sc[d][i] = (uint32_t)smem[sa_at + i * 512u + ph_a + g] | (uint32_t)smem[sa_at + i * 512u + ph_a + g + 2] << 16;
                    else sc[d][i] = *reinterpret_cast<const uint32_t *>(smem + sa_at + i * 512u);
                }
#pragma unroll
                for (int j = 0; j < JB; j++) {
                    if constexpr (!TB) {
                        const uint32_t at = rd_sb + buf + (uint32_t)((ws * NSP + d) * 4 * TN) + (uint32_t)(j * JC * 2 + g);
                        sc[d][MB + j] = (uint32_t)smem[at] | (uint32_t)smem[at + 2u * TN] << 16;
                    } else {
                        const uint32_t at = rd_sb + buf + (uint32_t)((ws * NSP + d) * 4 + j * JC * 16);
                        if constexpr (UA) sc[d][MB + j] = (uint32_t)smem[at + ph_b + g] | (uint32_t)smem[at + ph_b + g + 2] << 16;
                        else sc[d][MB + j] = *reinterpret_cast<const uint32_t *>(smem + at);
                    }
                }
            }
        }
    };
    auto read_half = [&](auto stg_c, auto ks_c) {
        constexpr int STG = decltype(stg_c)::value, ks = decltype(ks_c)::value;
#pragma unroll
        for (int i = 0; i < MB; i++) {
            const v4i l = lds_read16_abs(fr_a[2 * ks] + (uint32_t)(STG * STAGE + i * 4096)), h = lds_read16_abs(fr_a[2 * ks + 1] + (uint32_t)(STG * STAGE + i * 4096));
            fa[i][ks] = (v8i){l[0], l[1], l[2], l[3], h[0], h[1], h[2], h[3]};
        }
#pragma unroll
        for (int j = 0; j < JB; j++) {
            if constexpr (TB) {
                const v4i l = lds_read16_abs(fr_b[2 * ks] + (uint32_t)(STG * STAGE + j * JC * BKB)), h = lds_read16_abs(fr_b[2 * ks + 1] + (uint32_t)(STG * STAGE + j * JC * BKB));
                fb[j][ks] = (v8i){l[0], l[1], l[2], l[3], h[0], h[1], h[2], h[3]};
            } else {
                typedef __attribute__((address_space(3))) v2i *LdsV2;
                const uint32_t at = fbt[j] + (uint32_t)(STG * STAGE + ks * 32 * ROW8);
                v2i t0, t1, t2, t3;
                if constexpr (EPB == 2) {
                    t0 = __builtin_amdgcn_ds_read_tr4_b64_v2i32((LdsV2)(uintptr_t)(at));
                    t1 = __builtin_amdgcn_ds_read_tr4_b64_v2i32((LdsV2)(uintptr_t)(at + 4u * ROW8));
                    t2 = __builtin_amdgcn_ds_read_tr4_b64_v2i32((LdsV2)(uintptr_t)(at + 16u * ROW8));
                    t3 = __builtin_amdgcn_ds_read_tr4_b64_v2i32((LdsV2)(uintptr_t)(at + 20u * ROW8));
                } else {
                    t0 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2)(uintptr_t)(at));
                    t1 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2)(uintptr_t)(at + 4u * ROW8));
                    t2 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2)(uintptr_t)(at + 16u * ROW8));
                    t3 = __builtin_amdgcn_ds_read_tr8_b64_v2i32((LdsV2)(uintptr_t)(at + 20u * ROW8));
                }
                fb[j][ks] = (v8i){t0[0], t0[1], t1[0], t1[1], t2[0], t2[1], t3[0], t3[1]};
            }
        }
    };
    // (K-contiguous panels) read number x of a half: 16 bytes of a fragment of A, then of B
    auto read_piece = [&](auto stg_c, auto ks_c, auto x_c) {
        constexpr int STG = decltype(stg_c)::value, ks = decltype(ks_c)::value, x = decltype(x_c)::value, i = x / 2, h = x % 2;
        static_assert(TB || !DEEP, "a transposing read brings 8 bytes");
        if constexpr (i < MB) {
            const v4i v = lds_read16_abs(fr_a[2 * ks + h] + (uint32_t)(STG * STAGE + i * 4096));
#pragma unroll
            for (int w = 0; w < 4; w++) fa[i][ks][4 * h + w] = v[w];
        } else {
            const v4i v = lds_read16_abs(fr_b[2 * ks + h] + (uint32_t)(STG * STAGE + (i - MB) * JC * BKB));
#pragma unroll
            for (int w = 0; w < 4; w++) fb[i - MB][ks][4 * h + w] = v[w];
        }
    };
    // This lane's scale bytes (block g of either K64 block) to bytes 0 and 2; those of blocks past K cleared (their payload is zero,
    // and a zero byte keeps the product zero where a stray 0xFF, NaN, would not).
    auto finish_scales = [&](int k, uint32_t (&sc)[NSP > 0 ? NSP : 1][MB + JB]) {
        if constexpr (MX) {
#pragma unroll
            for (int d = 0; d < NSP; d++) {
                const int b0 = (k * NSP + d) * 4 + g;
                const uint32_t keep = (b0 < nblk ? 0xFFu : 0u) | (b0 + 2 < nblk ? 0xFF0000u : 0u);
#pragma unroll
                for (int s = 0; s < MB + JB; s++) sc[d][s] = (UA && s < MB) || (UA && TB) || (!TB && s >= MB) ? sc[d][s] & keep : (sc[d][s] >> (8 * g)) & keep;
            }
        }
    };
    // one matrix instruction of 64-byte half ks, number m of NM
    auto mfma = [&](auto ks_c, auto m_c, const uint32_t (&sc)[NSP > 0 ? NSP : 1][MB + JB]) {
        constexpr int ks = decltype(ks_c)::value, m = decltype(m_c)::value;
        constexpr int half = m / (JB * MB), i = (m / JB) % MB, j = m % JB, d = NSP > 1 ? ks : 0;
        if constexpr (KIND == KIND_F8) {
            acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fa[i][ks], fb[j][ks], acc[i][j], CBSZ, CBSZ, 2 * ks, (int)sc[0][i], 2 * ks, (int)sc[0][MB + j]);
        } else {
            const v8i &a = fa[i][ks], &b = fb[j][ks];
            if constexpr (KIND == KIND_F4) {
                const v8i ah = (v8i){a[4 * half], a[4 * half + 1], a[4 * half + 2], a[4 * half + 3], 0, 0, 0, 0};
                const v8i bh = (v8i){b[4 * half], b[4 * half + 1], b[4 * half + 2], b[4 * half + 3], 0, 0, 0, 0};
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(ah, bh, acc[i][j], 4, 4, 2 * half, (int)sc[d][i], 2 * half, (int)sc[d][MB + j]);
            } else {
                const v4i ah = (v4i){a[4 * half], a[4 * half + 1], a[4 * half + 2], a[4 * half + 3]};
                const v4i bh = (v4i){b[4 * half], b[4 * half + 1], b[4 * half + 2], b[4 * half + 3]};
                acc[i][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(ah, bh, acc[i][j], 0, 0, 0);
            }
        }
    };
    constexpr int NM = (KIND == KIND_F8 ? 1 : 2) * JB * MB;   // matrix instructions per half
    constexpr int STEP_REQ = NREQ + NSR;

    // Two stages: a step's stage is requested anew within the step, behind a second barrier.  Three: the stage of the step
    // before, which everybody has left when the step's own barrier opens.
    constexpr bool ONE_BARRIER = S >= 3;
    constexpr int AHEAD = ONE_BARRIER && !DEEP ? S - 1 : S;   // steps from a request to its use
    auto step = [&](int k, auto stg_c) {
        auto &sc = scales[0];
        // this step's stage has landed (the younger ones may still be on their way)
        CCH_WAIT_VM((AHEAD - 1) * STEP_REQ);
        CCH_BARRIER();
        read_scales(k, sc);
        read_half(stg_c, IC<0>{});
        __builtin_amdgcn_sched_barrier(0);
        read_half(stg_c, IC<1>{});
        __builtin_amdgcn_sched_barrier(0);
        Ahead nx;
        if constexpr (ONE_BARRIER) {
            nx = ahead_of(k + AHEAD);
            request(nx, IC<0>{});
            request(nx, IC<1>{});
        }
        // (LDS reads return in order: all but the second half's are there)
        CCH_WAIT_LGKM((TB ? 4 : 8) + 2 * MB);
        __builtin_amdgcn_sched_barrier(0);
        finish_scales(k, sc);
        // The first half's products run while the second half's fragments arrive.  The address unit takes a request in about
        // the time of a quarter of a matrix instruction, so the requests sit between those instead of in front of them.
        constexpr int DONE = ONE_BARRIER ? 2 : 1, REST = NREQ + 1 - DONE;   // (two barriers: all but the scales between the second half's)
        static_for<NM>([&](auto m_c) {
            constexpr int m = decltype(m_c)::value;
            mfma(IC<0>{}, m_c, sc);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (ONE_BARRIER) {
                constexpr int from = DONE + REST * m / (2 * NM), to = DONE + REST * (m + 1) / (2 * NM);
                static_for<to - from>([&](auto x_c) { request(nx, IC<from + decltype(x_c)::value>{}); });
                __builtin_amdgcn_sched_barrier(0);
            }
        });
        if constexpr (!ONE_BARRIER) {
            __builtin_amdgcn_sched_barrier(0);
            CCH_WAIT_LGKM0();
            CCH_BARRIER();
            nx = ahead_of(k + AHEAD);
            request(nx, IC<0>{});
            __builtin_amdgcn_sched_barrier(0);
        }
        static_for<NM>([&](auto m_c) {
            constexpr int m = decltype(m_c)::value;
            mfma(IC<1>{}, m_c, sc);
            __builtin_amdgcn_sched_barrier(0);
            constexpr int from = ONE_BARRIER ? DONE + REST * (NM + m) / (2 * NM) : DONE + REST * m / NM;
            constexpr int to = ONE_BARRIER ? DONE + REST * (NM + m + 1) / (2 * NM) : DONE + REST * (m + 1) / NM;
            static_for<to - from>([&](auto x_c) { request(nx, IC<from + decltype(x_c)::value>{}); });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // One wave per SIMD (DEEP): nobody else covers a wait, and a wave issues in order, so everything a matrix instruction needs is read
    // half a step before it, and whatever else there is to issue sits a few instructions at a time between matrix instructions, in
    // the cycles that the wave waits for the pipe.  The second half's fragments arrive while the first half is multiplied; towards its end the next
    // step's stage has landed and everybody has read this step's (one barrier says both); then the next step's first half arrives
    // and this stage is requested anew, three steps ahead.
    auto deep_step = [&](int k, auto stg_c, auto nstg_c, auto par_c) {
        constexpr int par = decltype(par_c)::value;
        constexpr int RD = 2 * (MB + JB), R0 = NM * 2 / 3, R1 = NM * 7 / 9;   // fragment reads per half; gaps that hold them
        auto &sc = scales[par], &sn = scales[par ^ 1];
        Ahead nx;
        static_for<NM>([&](auto m_c) {
            constexpr int m = decltype(m_c)::value;
            mfma(IC<0>{}, m_c, sc);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (m < R0) {
                constexpr int from = RD * m / R0, to = RD * (m + 1) / R0;
                static_for<to - from>([&](auto x_c) { read_piece(stg_c, IC<1>{}, IC<from + decltype(x_c)::value>{}); });
            } else if constexpr (m == R0) {
                CCH_WAIT_VM_LGKM0((AHEAD - 2) * STEP_REQ);
                CCH_BARRIER();
            } else if constexpr (m == R0 + 1) {
                nx = ahead_of(k + AHEAD);
            } else if constexpr (m == NM - 1) {
                read_scales(k + 1, sn);
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        static_for<NM>([&](auto m_c) {
            constexpr int m = decltype(m_c)::value;
            mfma(IC<1>{}, m_c, sc);
            __builtin_amdgcn_sched_barrier(0);
            if constexpr (m < R1) {
                constexpr int from = RD * m / R1, to = RD * (m + 1) / R1;
                static_for<to - from>([&](auto x_c) { read_piece(nstg_c, IC<0>{}, IC<from + decltype(x_c)::value>{}); });
            }
            constexpr int from = (NREQ + 1) * m / NM, to = (NREQ + 1) * (m + 1) / NM;
            static_for<to - from>([&](auto x_c) { request(nx, IC<from + decltype(x_c)::value>{}); });
            if constexpr (m == NM - 1) finish_scales(k + 1, sn);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    for (int k = 0; k < AHEAD; k++) {
        const Ahead n = ahead_of(k);
        static_for<NREQ + 1>([&](auto x_c) { request(n, x_c); });
    }
    if constexpr (DEEP) {
        CCH_WAIT_VM((AHEAD - 1) * STEP_REQ);
        CCH_BARRIER();
        read_scales(0, scales[0]);
        read_half(IC<0>{}, IC<0>{});
        finish_scales(0, scales[0]);
        for (int k = 0; k < steps; k += 2 * S)
            static_for<2 * S>([&](auto s_c) {
                constexpr int s = decltype(s_c)::value;
                if (k + s < steps) deep_step(k + s, IC<s % S>{}, IC<(s + 1) % S>{}, IC<s % 2>{});
            });
    } else {
        for (int k = 0; k < steps; k += S)
            static_for<S>([&](auto s_c) {
                if (k + decltype(s_c)::value < steps) step(k + decltype(s_c)::value, s_c);
            });
    }

    // ---- epilogue, each wave on its own: its outputs as [row][64 columns] of 32 bits through a part of the ring (every wave has
    // read its last fragments), then 8 neighbouring output columns of a row per lane and pass
    constexpr int IPR = SWIGLU ? 4 : 4 * JB;               // items per row
    constexpr int NPASS = 32 * MB * IPR / 64;
    constexpr uint32_t ROW = 128 * JB;                     // bytes of a staged row
    // a lane's columns: the same in every pass where a pass is whole rows
    auto item_col = [&](int it) { return (it * 64 + lane) % IPR * 8; };
    const int icol = j0 + wn * (SWIGLU ? 32 : 32 * JB) + (lane % IPR) * 8;
    float ch[SWIGLU ? 16 : 8] = {}, tok[NPASS] = {};
    int mapped[NPASS] = {};
    if constexpr (DEQ) {
        const float *pc = p.per_ch + (size_t)e * p.N + min(icol, p.n_out - 8);
#pragma unroll
        for (int x = 0; x < 8; x++) {
            ch[x] = pc[x];
            if constexpr (SWIGLU) ch[8 + x] = pc[p.n_out + x];
        }
    }
#pragma unroll
    for (int it = 0; it < NPASS; it++) {
        const int row = min(wm * 32 * MB + (it * 64 + lane) / IPR, rows - 1);
        if constexpr (DEQ) tok[it] = p.per_tok[m0 + row];
        if constexpr (EPI == EPI_PLAIN) {
            if (p.out_row_map) mapped[it] = p.out_row_map[m0 + row];
        }
    }
    CCH_WAIT_VM(0);   // (requests against empty descriptors write zeros)
    CCH_BARRIER();
    const uint32_t mine = (uint32_t)(wave * MB * 32) * ROW;
    {
        typedef typename std::remove_reference<decltype(acc[0][0][0])>::type Elem;
        const uint32_t at = mine + (uint32_t)(g * 4) * ROW + (uint32_t)r * 4u;
#pragma unroll
        for (int i = 0; i < MB; i++)
#pragma unroll
            for (int j = 0; j < JB; j++)
#pragma unroll
                for (int x = 0; x < 16; x++) *reinterpret_cast<Elem *>(smem + at + (uint32_t)(i * 32 + (x >> 2) * 8 + (x & 3)) * ROW + (uint32_t)j * 128u) = acc[i][j][x];
    }
    asm volatile("" ::: "memory");   // (one wave's LDS operations execute in order)
    typedef typename std::conditional<KIND == KIND_I8, v4i, __attribute__((ext_vector_type(4))) float>::type Raw4;
    auto read8 = [&](int row, int col, float (&v)[8]) {
        const Raw4 s0 = *reinterpret_cast<const Raw4 *>(smem + mine + (uint32_t)row * ROW + (uint32_t)col * 4u);
        const Raw4 s1 = *reinterpret_cast<const Raw4 *>(smem + mine + (uint32_t)row * ROW + (uint32_t)col * 4u + 16u);
#pragma unroll
        for (int x = 0; x < 4; x++) {
            v[x] = (float)s0[x];
            v[4 + x] = (float)s1[x];
        }
    };
    with_output_kind<EPI>(p, [&](auto step_c, auto half_c) {
#pragma unroll
        for (int it = 0; it < NPASS; it++) {
            const int lrow = (it * 64 + lane) / IPR, lcol = item_col(it), row = wm * 32 * MB + lrow;
            const int col = JB == 2 ? icol : j0 + wn * 32 * JB + lcol;
            float v[8], up[8] = {};
            read8(lrow, lcol, v);
            if constexpr (SWIGLU) read8(lrow, 32 + lcol, up);
            finish8<EPI, decltype(step_c)::value != 0>(v, up, ch, tok[it]);
            store8<EPI, decltype(half_c)::value != 0>(p, v, row < rows && col + 8 <= p.n_out, m0 + row, mapped[it], col);
        }
    });
}

template <int KIND, int EPI, int FMT, int TB, int UA, int MB, int WN, int JB = 2>
static int launch_mid_mb(const GemmProblem &p, hipStream_t stream)
{
    constexpr int S = mid_stages(MB, WN), TN = mid_cols(WN, JB);
    constexpr int lds = S * mid_stage_bytes(MB, WN, JB) + (KIND == KIND_I8 ? 0 : mid_scale_buffers(S, mid_steps_per_scales(KIND, UA)) * (64 * MB + TN) * 16 + 1024);
    static_assert(lds <= 160 * 1024, "the ring and the scales of a CU");
    auto kern = gemm_mid_kernel<KIND, EPI, FMT, TB, UA, MB, WN, JB>;
    // set once per device and kernel; setting it twice from two threads is harmless
    static std::atomic<uint64_t> attr_set{0};
    int dev = 0;
    CCH_HIP(hipGetDevice(&dev));
    const uint64_t dev_bit = (uint64_t)1 << (dev & 63);
    if (dev >= 64 || !(attr_set.load(std::memory_order_acquire) & dev_bit)) {
        CCH_HIP(hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, lds));
        attr_set.fetch_or(dev_bit, std::memory_order_release);
    }
    constexpr int tn_out = (EPI == EPI_DEQUANT_SWIGLU || EPI == EPI_SWIGLU) ? TN / 2 : TN;
    const int64_t col_tiles = (p.n_out + tn_out - 1) / tn_out;
    const int64_t tiles = p.tail_cus ? std::min<int64_t>(TAIL_TILES, p.num_groups * (TAIL_ROWS / 64) * col_tiles) : row_tiles_bound(p, 64 * MB) * col_tiles;
    hipLaunchKernelGGL(kern, dim3((unsigned)mid_grid(tiles)), dim3(128 * WN), lds, stream, p);
    return launch_status("gemm_mid_kernel");
}

template <int KIND, int EPI, int FMT, int TB, int UA>
static int launch_mid_ua(const GemmProblem &p, int rows, int cols, hipStream_t stream)
{
    // (MXFP4 rows that can start 2 bytes past a dword need a scale buffer per stage, which the wide tile's ring leaves no room for)
    if constexpr (KIND != KIND_F4 || !UA) {
        if (cols == 256) return launch_mid_mb<KIND, EPI, FMT, TB, UA, 2, 4>(p, stream);
        if constexpr (TB && EPI == EPI_PLAIN) {
            if (cols == 192) return launch_mid_mb<KIND, EPI, FMT, TB, UA, 3, 2, 3>(p, stream);
        }
    }
    return rows == 64 ? launch_mid_mb<KIND, EPI, FMT, TB, UA, 1, 2>(p, stream) : launch_mid_mb<KIND, EPI, FMT, TB, UA, 2, 2>(p, stream);
}

template <int KIND, int EPI, int FMT, int TB>
int launch_mid_t(const GemmProblem &p, int rows, int cols, hipStream_t stream)
{
    if constexpr (KIND != KIND_I8) {
        if ((p.sld & 3) != 0 || (p.sa_pitch & 3) != 0) return launch_mid_ua<KIND, EPI, FMT, TB, 1>(p, rows, cols, stream);
    }
    return launch_mid_ua<KIND, EPI, FMT, TB, 0>(p, rows, cols, stream);
}

}  // namespace cch
