// kq.h — what the k-quant matrix-core kernels share: operand types, the f16 of a header, a wave-tile's size.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace larql {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
union Q4kOp { i32x4 v; uint32_t u[4]; };  // one MFMA operand: 16 int8 k-slots of a lane
constexpr uint32_t kQ4kTileBytes = 16 * 144;

__device__ __forceinline__ float half_bits_to_float(uint32_t lo16) {
    // hardware f16 -> f32 conversion; f16 subnormals are preserved (the f16
    // denormal mode is on for HIP kernels), which the Q4_K scales rely on.
    return (float)__builtin_bit_cast(_Float16, (uint16_t)lo16);
}

}  // namespace larql
