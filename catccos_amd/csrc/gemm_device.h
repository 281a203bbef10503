// Device-side pieces that the MFMA GEMM kernels share: vector types, waits and barriers, the direct global -> LDS
// loads, LDS reads by address, the panel swizzle and the wave-wide prefix sum.
#pragma once
#include <type_traits>
#include <utility>

#include "common.h"
#include "gemm_common.h"
#include "gemm_tile_shape.h"
#include "mx_formats.h"
#include "mx_quant_block.h"

namespace cch {

typedef int v2i __attribute__((ext_vector_type(2)));
typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef int v16i __attribute__((ext_vector_type(16)));
typedef unsigned int v4u __attribute__((ext_vector_type(4)));
typedef unsigned int v2u __attribute__((ext_vector_type(2)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

template <int KIND> struct KindTraits;
template <> struct KindTraits<KIND_I8> { static constexpr int ELEMS_PER_BYTE = 1, SCALE_DW = 0; using Acc = v16i; };
template <> struct KindTraits<KIND_F8> { static constexpr int ELEMS_PER_BYTE = 1, SCALE_DW = 1; using Acc = v16f; };
template <> struct KindTraits<KIND_F4> { static constexpr int ELEMS_PER_BYTE = 2, SCALE_DW = 2; using Acc = v16f; };

extern __shared__ __attribute__((aligned(1024))) uint8_t smem[];

template <int N> using IC = std::integral_constant<int, N>;

// Calls f(IC<0>) ... f(IC<N-1>): loop indices that must be compile-time constants.
template <int... I, class F>
__device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F &&f)
{
    (f(IC<I>{}), ...);
}
template <int N, class F> __device__ __forceinline__ void static_for(F &&f)
{
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}

__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// s_waitcnt on gfx9: vmcnt in bits [3:0] and [15:14], expcnt [6:4], lgkmcnt [11:8].
#define CCH_WAIT_VM_LGKM0(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | (7 << 4))
// vmcnt only (lgkmcnt left at its maximum of 15)
#define CCH_WAIT_VM(n) __builtin_amdgcn_s_waitcnt(((n) & 15) | (((n) >> 4) << 14) | (7 << 4) | (15 << 8))
// s_waitcnt lgkmcnt(n) only (vmcnt left at its maximum of 63)
#define CCH_WAIT_LGKM(n) __builtin_amdgcn_s_waitcnt(0xC07F | ((n) << 8))
#define CCH_WAIT_LGKM0() __builtin_amdgcn_s_waitcnt(0xC07F)

// Workgroup barrier that the compiler moves no memory access across (the intrinsic alone is not a
// memory barrier to the optimiser) and that the instruction scheduler leaves where it is.
#define CCH_BARRIER()                                  \
    do {                                               \
        __builtin_amdgcn_sched_barrier(0);             \
        asm volatile("s_barrier" ::: "memory");        \
        __builtin_amdgcn_sched_barrier(0);             \
    } while (0)

// 16 / 4 bytes per lane, global -> LDS without passing through registers, as raw buffer loads:
// the descriptor holds the wave-uniform base, `voff` is the per-lane byte offset, `soff` a
// wave-uniform byte offset (the K position).  Lane l of the wave lands at LDS address
// lds_addr + size*l.  A lane whose offset lies at or past the descriptor's size fetches nothing
// and receives zeros.  Issued as inline assembly on purpose: the compiler's wait-count pass
// would otherwise drain every outstanding direct-to-LDS load before each LDS read;
// completion is tracked by the explicit vmcnt waits instead.
typedef int Rsrc __attribute__((ext_vector_type(4)));
__device__ __forceinline__ Rsrc make_rsrc(const void *base, uint32_t bytes)
{
    const uint64_t b = reinterpret_cast<uint64_t>(base);
    Rsrc rs;
    rs[0] = __builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    rs[1] = __builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32));  // stride 0, no swizzle
    rs[2] = __builtin_amdgcn_readfirstlane((int)bytes);                // num_records (bytes); reads past it return 0
    rs[3] = 0x00020000;                                                // raw 32-bit data format
    return rs;
}
// Descriptors are wave-uniform by construction; this pins them to scalar registers where the
// compiler has lost track of that (the 16-byte requests of the K loop take theirs as built).
__device__ __forceinline__ Rsrc scalar_rsrc(Rsrc rs)
{
    Rsrc u;
    u[0] = __builtin_amdgcn_readfirstlane(rs[0]);
    u[1] = __builtin_amdgcn_readfirstlane(rs[1]);
    u[2] = __builtin_amdgcn_readfirstlane(rs[2]);
    u[3] = 0x00020000;
    return u;
}
__device__ __forceinline__ void load16_to_lds(Rsrc rs, uint32_t voff, uint32_t soff, uint32_t lds_addr)
{
    soff = (uint32_t)__builtin_amdgcn_readfirstlane((int)soff);
    lds_addr = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(rs), "s"(soff)
                 : "memory", "m0");
}
// The same with the LDS address given as a scalar base plus a compile-time displacement (one scalar add
// straight into M0).
template <int DISP>
__device__ __forceinline__ void load16_to_lds_at(Rsrc rs, uint32_t voff, uint32_t soff, uint32_t lds_sbase)
{
    soff = (uint32_t)__builtin_amdgcn_readfirstlane((int)soff);
    lds_sbase = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_sbase);
    asm volatile("s_add_u32 m0, %0, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 :
                 : "s"(lds_sbase), "v"(voff), "s"(rs), "s"(soff), "i"(DISP)
                 : "memory", "m0", "scc");
}
__device__ __forceinline__ void load4_to_lds(Rsrc rs, uint32_t voff, uint32_t soff, uint32_t lds_addr)
{
    rs = scalar_rsrc(rs);
    soff = (uint32_t)__builtin_amdgcn_readfirstlane((int)soff);
    lds_addr = (uint32_t)__builtin_amdgcn_readfirstlane((int)lds_addr);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dword %1, %2, %3 offen lds"
                 :
                 : "s"(lds_addr), "v"(voff), "s"(rs), "s"(soff)
                 : "memory", "m0");
}

__device__ __forceinline__ v4i lds_read16(uint32_t off) { return *reinterpret_cast<const v4i *>(smem + off); }
__device__ __forceinline__ uint32_t lds_read4(uint32_t off) { return *reinterpret_cast<const uint32_t *>(smem + off); }
// The same reads from an absolute LDS address (a base that already holds the segment's start plus a
// compile-time displacement, which becomes the instruction's offset field).
__device__ __forceinline__ v4i lds_read16_abs(uint32_t addr)
{
    return *reinterpret_cast<const __attribute__((address_space(3))) v4i *>((uintptr_t)addr);
}
__device__ __forceinline__ uint32_t lds_read4_abs(uint32_t addr)
{
    return *reinterpret_cast<const __attribute__((address_space(3))) uint32_t *>((uintptr_t)addr);
}

// Panel layout: row pitch 128 B; 16-byte chunk c of row `row` sits at chunk position
// c ^ ((row >> 1) & 7), which spreads 16 consecutive rows over all 64 banks for 16-byte reads.
__device__ __forceinline__ uint32_t swizzle_of_row(int row) { return (uint32_t)((row >> 1) & 7); }

constexpr uint32_t NO_FETCH = 0xFFFFFFF0u;   // a lane offset past every descriptor: the lane fetches nothing

// Inclusive prefix sum over the 64 lanes of a wave with saturating unsigned adds (associative, and exact
// while no partial sum passes 2^32 - 1): four shifts inside each row of 16 lanes, then the last lane of row 0
// into row 1 and of row 2 into row 3, then the last lane of row 1 into rows 2 and 3 (data-parallel
// primitives of gfx9: no trip through LDS).
__device__ __forceinline__ uint32_t sat_add(uint32_t a, uint32_t b) { const uint32_t s = a + b; return s < a ? 0xFFFFFFFFu : s; }
__device__ __forceinline__ uint32_t wave_scan_sat(uint32_t v)
{
    v = sat_add(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, true));   // row_shr:1
    v = sat_add(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, true));   // row_shr:2
    v = sat_add(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, true));   // row_shr:4
    v = sat_add(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, true));   // row_shr:8
    v = sat_add(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false));  // row_bcast:15 into rows 1 and 3
    v = sat_add(v, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false));  // row_bcast:31 into rows 2 and 3
    return v;
}

}  // namespace cch
