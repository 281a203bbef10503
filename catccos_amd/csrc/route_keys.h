// Keys of the routing sort (routing.hip) and of the FFN's dispatch (moe_ffn.hip), which ranks routes the same way.
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

// Bits of a key below num_experts.
inline int route_key_bits(int num_experts)
{
    int bits = 0;
    while ((1 << bits) < num_experts) bits++;
    return bits;
}

}  // namespace cch
