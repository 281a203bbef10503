// What happens to eight neighbouring results of one row at the end of a tile: shared by the kernels whose accumulators pass
// through LDS as fp32 (int32) rows.
#pragma once
#include "gemm_mid.h"
#include "gemm_tail.h"

namespace cch {

// The raw sums v (and, with SwiGLU, those of the up columns) become the eight outputs: dequantisation, activation.  `ch` holds the
// per-channel factors (SwiGLU: gate columns, then up columns), `tok` the row's per-token factor.  FP16_STEP: GemmProblem::i8_fp16_step.
template <int EPI, bool FP16_STEP>
__device__ __forceinline__ void finish8(float (&v)[8], const float (&up)[8], const float *ch, float tok)
{
    constexpr bool SWIGLU = EPI == EPI_DEQUANT_SWIGLU || EPI == EPI_SWIGLU;
#pragma unroll
    for (int x = 0; x < 8; x++) {
        if constexpr (SWIGLU) {
            float gate = v[x], u = up[x];
            if constexpr (EPI == EPI_DEQUANT_SWIGLU) {
                gate *= ch[x];
                u *= ch[8 + x];
                if constexpr (FP16_STEP) {
                    // (two roundings, fp32 and then half: the compiler would otherwise fuse product and conversion)
                    asm volatile("" : "+v"(gate), "+v"(u));
                    gate = (float)(_Float16)gate;
                    u = (float)(_Float16)u;
                }
                gate *= tok;
                u *= tok;
            } else {
                gate = (float)(__bf16)gate;   // the up projection's result is a bf16 tile before the activation sees it
                u = (float)(__bf16)u;
            }
            v[x] = gate * __builtin_amdgcn_rcpf(1.0f + __expf(-gate)) * u;
        } else if constexpr (EPI == EPI_DEQUANT) {
            if constexpr (FP16_STEP) {
                float prod = v[x] * ch[x];
                asm volatile("" : "+v"(prod));
                v[x] = (float)(_Float16)prod * tok;
            } else {
                v[x] = v[x] * tok * ch[x];
            }
        }
    }
}

// Stores the eight outputs at row `row` (of the whole output; `mapped` where a row map redirects it) and columns col .. col+7.
// MX-quantised output: the four lanes of a quad hold one row's 32 columns, one MX block (all four must call).
template <int EPI, bool FP16>
__device__ __forceinline__ void store8(const GemmProblem &p, const float (&v)[8], bool ok, int row, int mapped, int col)
{
    constexpr bool SWIGLU = EPI == EPI_DEQUANT_SWIGLU || EPI == EPI_SWIGLU;
    uint32_t w[4];
#pragma unroll
    for (int x = 0; x < 4; x++) {
        if constexpr (FP16) w[x] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){v[2 * x], v[2 * x + 1]}, f16x2));
        else w[x] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){v[2 * x], v[2 * x + 1]}, bf16x2));
    }
    if constexpr (SWIGLU) {
        if (p.mx_out) {
            const uint32_t amax = block_amax_bits(w);
            uint32_t code[2], sbyte;
            int ex;
            bool is_nan;
            if (p.mx_out_fmt == CCH_FMT_E2M1) {
                sbyte = shared_exp_byte<CCH_FMT_E2M1>(amax, ex, is_nan);
                quant8_hw<CCH_FMT_E2M1>(w, ex, is_nan, code);
            } else if (p.mx_out_fmt == CCH_FMT_E5M2) {
                sbyte = shared_exp_byte<CCH_FMT_E5M2>(amax, ex, is_nan);
                quant8_hw<CCH_FMT_E5M2>(w, ex, is_nan, code);
            } else {
                sbyte = shared_exp_byte<CCH_FMT_E4M3>(amax, ex, is_nan);
                quant8_hw<CCH_FMT_E4M3>(w, ex, is_nan, code);
            }
            if (ok) {
                uint8_t *o = reinterpret_cast<uint8_t *>(p.out);
                const size_t elem = (size_t)row * p.n_out + col;
                if (p.mx_out_fmt == CCH_FMT_E2M1) *reinterpret_cast<uint32_t *>(o + elem / 2) = code[0];
                else *reinterpret_cast<v2u *>(o + elem) = (v2u){code[0], code[1]};
                if ((threadIdx.x & 3) == 0) {
                    uint8_t *s = p.out_scales + (size_t)row * p.mx_out_sld + (col >> 5);
                    s[0] = (uint8_t)sbyte;
                    if ((p.n_out & 32) != 0 && col >> 5 == (p.n_out >> 5) - 1) s[1] = 127;   // behind an odd count of blocks
                }
            }
            return;
        }
    }
    size_t out_row = (size_t)row;
    if constexpr (EPI == EPI_PLAIN) {
        if (p.out_row_map) {
            ok = ok && mapped >= 0 && mapped < p.out_rows;
            out_row = (size_t)mapped;
        }
    }
    if (ok) *reinterpret_cast<v4u *>(p.out + out_row * p.n_out + col) = (v4u){w[0], w[1], w[2], w[3]};
}

// Calls f(FP16_STEP, FP16) with what the problem asks for: a branch around the items of a tile instead of twelve inside each (they were
// a third of a small launch's epilogue).
template <int EPI, class F>
__device__ __forceinline__ void with_output_kind(const GemmProblem &p, F &&f)
{
    if constexpr (EPI == EPI_DEQUANT || EPI == EPI_DEQUANT_SWIGLU) {
        if (p.i8_fp16_step) {
            if (p.out_fp16) f(IC<1>{}, IC<1>{});
            else f(IC<1>{}, IC<0>{});
            return;
        }
    }
    if (p.out_fp16) f(IC<0>{}, IC<1>{});
    else f(IC<0>{}, IC<0>{});
}

// The arguments that a kernel needs at its start and those that its end needs lie in different lines of memory, and the compiler reads a line
// where it first needs one: three round trips to a launch's arguments before the first request and another in front of the epilogue.  This
// reads one word of every line at once; what is read later comes from the scalar cache.
__device__ __forceinline__ void touch_arguments(const GemmProblem &p)
{
    static_assert(sizeof(GemmProblem) <= 256, "four lines");
    asm volatile("" :: "s"((int)(uintptr_t)p.a), "s"((int)(uintptr_t)p.out_row_map), "s"(p.T), "s"(p.tile_order));
}

// Where a tile number lies among the groups of a problem.  Every wave finds it by itself from the prefix sums of the group
// sizes, 64 groups at a time; rows are clipped like the group table of the tiled kernel (once T rows are used up every later
// group is empty).
struct GroupPlace {
    bool found;
    int e, lo, hi;      // the group and its rows
    int rel, rt;        // the tile's number within the group, the group's row tiles
    int used, total;    // rows that belong to groups, tiles of all groups
};
__device__ __forceinline__ GroupPlace find_place(const GemmProblem &p, int tile, int tm, int n_tiles)
{
    const int lane = threadIdx.x & 63;
    GroupPlace g = {};
    uint32_t before = 0;
    int tiles_before = 0;
    for (int b = 0; b < p.num_groups; b += 64) {
        const uint32_t sz = b + lane < p.num_groups ? (uint32_t)min(max(p.group_sizes[b + lane], 0), p.T) : 0u;
        const uint32_t incl = sat_add(before, wave_scan_sat(sz));
        const int row_hi = (int)min(incl, (uint32_t)p.T);
        const uint32_t prev = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)incl, 0x138, 0xF, 0xF, false);   // wave_shr:1
        const int row_lo = (int)min(lane == 0 ? before : prev, (uint32_t)p.T);
        const int tiles = (row_hi - row_lo + tm - 1) / tm;
        const int tincl = (int)wave_scan_sat((uint32_t)tiles);
        const int start = (tiles_before + tincl - tiles) * n_tiles;
        const uint64_t hit = __ballot(tile >= start && tile < start + tiles * n_tiles);
        if (hit != 0) {
            const int l = __builtin_ctzll(hit);
            g.found = true;
            g.e = b + l;
            g.lo = __builtin_amdgcn_readlane(row_lo, l);
            g.hi = __builtin_amdgcn_readlane(row_hi, l);
            g.rel = tile - __builtin_amdgcn_readlane(start, l);
            g.rt = __builtin_amdgcn_readlane(tiles, l);
        }
        before = (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        tiles_before += __builtin_amdgcn_readlane(tincl, 63);
    }
    g.used = (int)min(before, (uint32_t)p.T);
    g.total = tiles_before * n_tiles;
    return g;
}

// The same for the second launch of a problem (gemm_tail.h): the groups' rows are those that the first left out.
template <bool SWIGLU>
__device__ __forceinline__ GroupPlace find_tail(const GemmProblem &p, int block, int tm, int n_tiles, int round_size)
{
    GroupPlace g = {};
    const GroupRows rows = group_rows(p);
    const uint32_t key = tail_key<SWIGLU>(p, rows);
    int tiles_before = 0, tiles[GroupRows::NB], start[GroupRows::NB];
#pragma unroll
    for (int b = 0; b < GroupRows::NB; b++) {
        tiles[b] = start[b] = 0;
        if (b * 64 < p.num_groups) {
            tiles[b] = in_tail(rows, b, key) ? (((rows.hi[b] - rows.lo[b]) & (BM - 1)) + tm - 1) / tm : 0;
            const int incl = (int)wave_scan_sat((uint32_t)tiles[b]);
            start[b] = (tiles_before + incl - tiles[b]) * n_tiles;
            tiles_before += __builtin_amdgcn_readlane(incl, 63);
        }
    }
    g.total = tiles_before * n_tiles;
    const int tile = mid_tile_of(block, g.total, round_size);
#pragma unroll
    for (int b = 0; b < GroupRows::NB; b++) {
        const uint64_t hit = __ballot(tile >= start[b] && tile < start[b] + tiles[b] * n_tiles);
        if (hit != 0) {
            const int l = __builtin_ctzll(hit);
            g.found = true;
            g.e = b * 64 + l;
            g.hi = __builtin_amdgcn_readlane(rows.hi[b], l);
            g.lo = g.hi - ((g.hi - __builtin_amdgcn_readlane(rows.lo[b], l)) & (BM - 1));
            g.rel = tile - __builtin_amdgcn_readlane(start[b], l);
            g.rt = __builtin_amdgcn_readlane(tiles[b], l);
        }
    }
    return g;
}

// Rows from `used` on belong to no group and are written as zeros by all workgroups together (usually there are none); with a
// row map they produce nothing.
template <int EPI>
__device__ __forceinline__ void zero_rest(const GemmProblem &p, int used)
{
    constexpr bool SWIGLU = EPI == EPI_DEQUANT_SWIGLU || EPI == EPI_SWIGLU;
    if (used >= p.T || (EPI == EPI_PLAIN && p.out_row_map)) return;
    const bool mx = SWIGLU && p.mx_out;
    const int out_row_bytes = mx ? (p.mx_out_fmt == CCH_FMT_E2M1 ? p.n_out / 2 : p.n_out) : p.n_out * 2;
    const size_t begin = (size_t)used * out_row_bytes / 16, end = (size_t)p.T * out_row_bytes / 16;
    v4u *o16 = reinterpret_cast<v4u *>(p.out);
    const size_t at = (size_t)blockIdx.x * blockDim.x + threadIdx.x, all = (size_t)gridDim.x * blockDim.x;
    for (size_t i = begin + at; i < end; i += all) o16[i] = (v4u){0, 0, 0, 0};
    if (mx)
        for (size_t i = (size_t)used * p.mx_out_sld + at; i < (size_t)p.T * p.mx_out_sld; i += all) p.out_scales[i] = 127;
}

}  // namespace cch
