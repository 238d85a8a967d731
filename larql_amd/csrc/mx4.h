// mx4.h — what the MXFP4 expert kernels share: address-space pointers, the bf16 operand, the gate rule and the split of an
// f32 activation into bf16 terms.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace larql {

// Pointers that arrive inside a job record are generic; telling the compiler
// they are global memory turns flat_load into global_load.
#define GLOBAL_AS __attribute__((address_space(1)))
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef const GLOBAL_AS uint8_t *g_u8p;
typedef const GLOBAL_AS uint32_t *g_u32p;
typedef const GLOBAL_AS u32x4 *g_u4p;
typedef const GLOBAL_AS f32x4 *g_f4p;
typedef const GLOBAL_AS float *g_f32p;
typedef GLOBAL_AS float *g_f32wp;

typedef const GLOBAL_AS void *g_vp;
typedef __attribute__((address_space(3))) void *lds_vp;

// s_waitcnt vmcnt(n), n < 64, leaving the other counters alone (gfx9 encoding)
#define LARQL_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
union BfOp { bf16x8_t v; uint32_t u[4]; };

// MoeGateRule::ClampedGlu (larql-compute/src/pipeline/moe.rs:88-92): g = min(g, L); u = clamp(u, -L, L);
// (u + 1) * (g * sigmoid(alpha * g))
__device__ __forceinline__ float clamped_glu(float g, float u, float L, float al) {
    const float gc = fminf(g, L);
    const float uc = u < -L ? -L : (u > L ? L : u);
    return (uc + 1.0f) * (gc * (1.0f / (1.0f + expf(-(gc * al)))));
}

// The three bf16 terms of two activations, packed pairwise (a in the low half): x = t0 + t1 + t2 exactly.  An infinite
// or NaN activation stays in the first term alone (its residual would be a NaN of its own making).
__device__ __forceinline__ void mx4_terms(float a, float b, uint32_t (&t)[3]) {
    const uint32_t ab = __builtin_bit_cast(uint32_t, a), bb = __builtin_bit_cast(uint32_t, b);
    uint32_t a0 = ab & 0xFFFF0000u, b0 = bb & 0xFFFF0000u;
    float ra = a - __builtin_bit_cast(float, a0), rb = b - __builtin_bit_cast(float, b0);  // exact
    if ((ab & 0x7F800000u) == 0x7F800000u) { ra = 0.f; a0 = (ab & 0x007FFFFFu) ? (a0 | 0x00400000u) : a0; }
    if ((bb & 0x7F800000u) == 0x7F800000u) { rb = 0.f; b0 = (bb & 0x007FFFFFu) ? (b0 | 0x00400000u) : b0; }
    const uint32_t a1 = __builtin_bit_cast(uint32_t, ra) & 0xFFFF0000u, b1 = __builtin_bit_cast(uint32_t, rb) & 0xFFFF0000u;
    ra -= __builtin_bit_cast(float, a1);
    rb -= __builtin_bit_cast(float, b1);
    const uint32_t a2 = __builtin_bit_cast(uint32_t, ra) & 0xFFFF0000u, b2 = __builtin_bit_cast(uint32_t, rb) & 0xFFFF0000u;
    t[0] = (a0 >> 16) | b0;
    t[1] = (a1 >> 16) | b1;
    t[2] = (a2 >> 16) | b2;
}

}  // namespace larql
