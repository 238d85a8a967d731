// wave.h — reductions over a wavefront.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace larql {

// Reductions over the wavefront by data-parallel primitives (four steps inside the rows of 16 lanes, two row
// broadcasts, then lane 63 holds the result): a few cycles per step, where a cross-lane shuffle costs an LDS round trip.
template <int CTRL, int ROW_MASK, bool BOUND>
__device__ __forceinline__ uint32_t dpp_max_u32(uint32_t v) {  // lanes without a source read 0: the identity here
    const uint32_t other = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, ROW_MASK, 0xF, BOUND);
    return other > v ? other : v;
}
__device__ __forceinline__ uint32_t wave_max_u32(uint32_t v) {
    v = dpp_max_u32<0xB1, 0xF, true>(v);    // quad_perm [1,0,3,2]
    v = dpp_max_u32<0x4E, 0xF, true>(v);    // quad_perm [2,3,0,1]
    v = dpp_max_u32<0x141, 0xF, true>(v);   // row_half_mirror
    v = dpp_max_u32<0x140, 0xF, true>(v);   // row_mirror
    v = dpp_max_u32<0x142, 0xA, false>(v);  // row_bcast:15 into rows 1 and 3
    v = dpp_max_u32<0x143, 0xC, false>(v);  // row_bcast:31 into rows 2 and 3
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
template <int CTRL, int ROW_MASK, bool BOUND>
__device__ __forceinline__ float dpp_fmax(float v) {  // lanes without a source read -inf
    return fmaxf(v, __builtin_bit_cast(float, __builtin_amdgcn_update_dpp((int)0xFF800000u, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xF, BOUND)));
}
__device__ __forceinline__ float wave_fmax(float v) {
    v = dpp_fmax<0xB1, 0xF, false>(v);
    v = dpp_fmax<0x4E, 0xF, false>(v);
    v = dpp_fmax<0x141, 0xF, false>(v);
    v = dpp_fmax<0x140, 0xF, false>(v);
    v = dpp_fmax<0x142, 0xA, false>(v);
    v = dpp_fmax<0x143, 0xC, false>(v);
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), 63));
}
__device__ __forceinline__ float lane_value(float v, uint32_t lane_uniform) {  // the lane index must be the same in every lane
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), (int)lane_uniform));
}

// of values that are not negative: lanes without a source bring 0
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ float dpp_move(float v) {
    return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, ROW_MASK, 0xF, true));
}
template <int CTRL, int ROW_MASK = 0xF>
__device__ __forceinline__ float dpp_max(float v) { return fmaxf(v, dpp_move<CTRL, ROW_MASK>(v)); }
__device__ __forceinline__ float row16_max(float v) {
    v = dpp_max<0xB1>(v);     // quad_perm [1,0,3,2]
    v = dpp_max<0x4E>(v);     // quad_perm [2,3,0,1]
    v = dpp_max<0x141>(v);    // row_half_mirror
    return dpp_max<0x140>(v); // row_mirror
}

// inclusive sums
__device__ __forceinline__ uint32_t wave_inclusive_sum(uint32_t v) {
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xF, 0xF, false);  // row_shr:1
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xF, 0xF, false);  // row_shr:2
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xF, 0xF, false);  // row_shr:4
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xF, 0xF, false);  // row_shr:8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xA, 0xF, false);  // row_bcast:15 into rows 1 and 3
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xC, 0xF, false);  // row_bcast:31 into rows 2 and 3
    return v;
}

}  // namespace larql
