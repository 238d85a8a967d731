// moe.hip — the small kernels around the MXFP4 expert matvecs of a MoE block:
// expert selection, the gate/up combine rule and the weighted sum.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "kernels.h"
#include "router.h"

namespace larql {

static_assert(kRouterMaxExperts == 64u * (uint32_t)kRouterWideSlots, "the wide selection holds kRouterMaxExperts logits");

// router::select for every token: one wavefront per token (router.h).
__global__ void __launch_bounds__(64) router_select_kernel(const float *__restrict__ logits, const float *__restrict__ bias, uint32_t n_experts,
                                                           uint32_t k, int policy, uint32_t *__restrict__ experts,
                                                           float *__restrict__ weights) {
    const uint32_t t = blockIdx.x, lane = threadIdx.x;
    uint32_t sel_idx[kRouterMaxK];
    float sel_w[kRouterMaxK];
    router_select_any(logits + (size_t)t * n_experts, bias, n_experts, k, policy, lane, sel_idx, sel_w);
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < kRouterMaxK; r++)
            if ((uint32_t)r < k) {
                experts[(size_t)t * k + r] = sel_idx[r];
                weights[(size_t)t * k + r] = sel_w[r];
            }
    }
}

// MoeGateRule::ClampedGlu — larql-compute/src/pipeline/moe.rs:88-92:
// g = min(g, L); u = clamp(u, -L, L); (u + 1) * (g * sigmoid(alpha * g)).
__global__ void clamped_glu_kernel(const float *__restrict__ g, const float *__restrict__ u, float *__restrict__ h, size_t n,
                                   float limit, float alpha) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float gv = fminf(g[i], limit);
    float uv = u[i];
    uv = uv < -limit ? -limit : (uv > limit ? limit : uv);
    const float sig = 1.0f / (1.0f + expf(-(gv * alpha)));
    h[i] = (uv + 1.0f) * (gv * sig);
}

// the same on the interleaved result of a fused gate_up matrix: g = gu[2i], u = gu[2i+1]
__global__ void clamped_glu_interleaved_kernel(const float *__restrict__ gu, float *__restrict__ h, size_t n, float limit, float alpha) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    float gv = fminf(gu[2 * i], limit);
    float uv = gu[2 * i + 1];
    uv = uv < -limit ? -limit : (uv > limit ? limit : uv);
    const float sig = 1.0f / (1.0f + expf(-(gv * alpha)));
    h[i] = (uv + 1.0f) * (gv * sig);
}

// weights[i] *= scale[experts[i]] — MoeExpertScalePolicy::PerExpert (larql-compute/src/cpu/ops/moe/mod.rs:168-176);
// a selected id outside the scale table keeps its weight, as the reference leaves it.
__global__ void expert_scale_kernel(float *__restrict__ weights, const uint32_t *__restrict__ experts, const float *__restrict__ scale,
                                    uint32_t n, uint32_t n_scale) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint32_t e = experts[i];
    if (e < n_scale) weights[i] *= scale[e];
}

// out[t] = sum over the token's k slots, in selection order, of w * (down output + the expert's down bias, where there is one)
// (larql-compute/src/cpu/ops/moe/forward.rs:220-228, 266-270: add_down_bias, then `*a += w * v`).  A slot whose expert id lies
// outside the bank adds nothing (forward.rs:203-208): its row of `d` holds nothing, and its bias is the bank's first.
// Bound: latency.  K is the number of slots (0: any, four at a time), so that the ids and weights come in one scalar read each and
// all rows of `d` are asked for together.  Four at a time / K at once, one token of 2816, us: one slot 2.4 / 2.1, six 2.55 / 2.2, eight
// 2.35 / 2.1; two to four slots 2.1 to 2.3 either way, and from 16 tokens on there is no difference.
template <int K, bool BIAS>
__global__ void __launch_bounds__(256) weighted_sum_kernel(const float *__restrict__ d, const float *__restrict__ weights, const uint32_t *__restrict__ experts,
                                                          float *__restrict__ out, uint32_t n_experts, uint32_t k_any, uint32_t hidden,
                                                          const float *__restrict__ bias) {
    const uint32_t t = blockIdx.y, k = K ? (uint32_t)K : k_any;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= hidden) return;
    constexpr int C = K ? K : 4;
    float acc = 0.0f;
    for (uint32_t r0 = 0; r0 < k; r0 += C) {
        uint32_t e[C];
        float w[C], v[C];
#pragma unroll
        for (int q = 0; q < C; q++) {
            const size_t s = (size_t)t * k + (K ? (uint32_t)q : min(r0 + q, k - 1));
            e[q] = experts[s];
            w[q] = weights[s];
            v[q] = d[s * hidden + i];
        }
#pragma unroll
        for (int q = 0; q < C; q++) {
            if (BIAS) v[q] += bias[(size_t)(e[q] < n_experts ? e[q] : 0u) * hidden + i];
            const float with = acc + w[q] * v[q];
            acc = (K || r0 + q < k) && e[q] < n_experts ? with : acc;
        }
    }
    out[(size_t)t * hidden + i] = acc;
}

// ---- the k-quant expert path (cpu_moe_forward over Q4_K / Q6_K banks: cpu/ops/moe/forward.rs:160-330) ----------------

// quantize_x_to_q8k (cpu/ops/q4k_q8k_dot/q8k_activation.rs:84-109) of one 256-element super-block that a wavefront
// holds four elements per lane: d = amax / 127, codes round(x * (1/d)) clamped to +-127, NaN -> 0.  `sum` ends, in the
// lanes 8s, as the sum of sub-block s's 32 codes.
__device__ __forceinline__ int q8k_code(float t) {
    float r = roundf(t);
    r = r < -127.0f ? -127.0f : (r > 127.0f ? 127.0f : r);
    return r != r ? 0 : (int)r;
}
__device__ __forceinline__ void q8k_block(const float (&v)[4], uint32_t &codes, float &scale, int &sum) {
    const float amax = wave_fmax(fmaxf(fmaxf(fabsf(v[0]), fabsf(v[1])), fmaxf(fabsf(v[2]), fabsf(v[3]))));  // fmaxf ignores a NaN operand, as f32::max does
    scale = amax > 0.0f ? amax / 127.0f : 0.0f;
    const float inv = scale > 0.0f ? 1.0f / scale : 0.0f;
    const int q0 = q8k_code(v[0] * inv), q1 = q8k_code(v[1] * inv), q2 = q8k_code(v[2] * inv), q3 = q8k_code(v[3] * inv);
    sum = q0 + q1 + q2 + q3;
    sum += __builtin_amdgcn_update_dpp(0, sum, 0xB1, 0xF, 0xF, true);   // quad_perm [1,0,3,2]
    sum += __builtin_amdgcn_update_dpp(0, sum, 0x4E, 0xF, 0xF, true);   // quad_perm [2,3,0,1]
    sum += __builtin_amdgcn_update_dpp(0, sum, 0x141, 0xF, 0xF, true);  // row_half_mirror: the other quad of the eight
    codes = ((uint32_t)q0 & 0xFFu) | (((uint32_t)q1 & 0xFFu) << 8) | (((uint32_t)q2 & 0xFFu) << 16) | (((uint32_t)q3 & 0xFFu) << 24);
}
// four elements of a row of `n` floats from j on, zeros past its end; `vec`: every row starts at 16 bytes and n % 4 == 0
__device__ __forceinline__ void load4(float (&v)[4], const float *row, uint32_t j, uint32_t n, bool vec) {
    if (vec) {
        const float4 f = j < n ? *reinterpret_cast<const float4 *>(row + j) : make_float4(0.f, 0.f, 0.f, 0.f);
        v[0] = f.x; v[1] = f.y; v[2] = f.z; v[3] = f.w;
    } else {
#pragma unroll
        for (uint32_t i = 0; i < 4; i++) v[i] = j + i < n ? row[j + i] : 0.0f;
    }
}
// the device layout of a Q8_K activation of `cols` elements at `o`: [cols codes | cols/256 f32 scales | cols/32 i16 sums]
__device__ __forceinline__ void q8k_store(uint8_t *o, uint32_t cols, uint32_t sb, uint32_t lane, uint32_t codes, float scale, int sum) {
    const uint32_t nb = cols / 256;
    reinterpret_cast<uint32_t *>(o)[sb * 64 + lane] = codes;
    if (lane == 0) reinterpret_cast<float *>(o + cols)[sb] = scale;
    if ((lane & 7u) == 0) reinterpret_cast<int16_t *>(o + cols + (size_t)nb * 4)[sb * 8 + (lane >> 3)] = (int16_t)sum;
}

// Row `blockIdx.y` of src ([rows, src_cols] floats, src_stride apart), zero-padded to `cols` (a multiple of 256: the
// stored row width of the gate/up matrices, forward.rs:176-184), as a Q8_K activation of its own at dst + row * dst_stride.
// One wavefront per super-block.
__global__ void __launch_bounds__(256) quantize_rows_to_q8k_kernel(const float *__restrict__ src, size_t src_stride, uint32_t src_cols, uint32_t cols,
                                                                  uint8_t *__restrict__ dst, size_t dst_stride) {
    const uint32_t sb = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (sb >= cols / 256) return;
    const float *s = src + (size_t)blockIdx.y * src_stride;
    const uint32_t j = sb * 256 + 4 * lane;
    float v[4];
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) v[i] = j + i < src_cols ? s[j + i] : 0.0f;
    uint32_t codes; float scale; int sum;
    q8k_block(v, codes, scale, sum);
    q8k_store(dst + (size_t)blockIdx.y * dst_stride, cols, sb, lane, codes, scale, sum);
}

// Token `blockIdx.x`'s route and its expert input in one launch (they do not depend on one another): wavefront 0 selects
// as router_select_kernel does and applies MoeExpertScalePolicy::PerExpert where a scale table is given (as
// expert_scale_kernel does) while the others, a wavefront per super-block up to eleven, quantise the token's row as
// quantize_rows_to_q8k_kernel does (four wavefronts, the first of them after its selection: 9.0 -> 6.1 us for 16 tokens of 2816).
// Where the matvecs run as a job per slot (rows or calls beyond the grouped kernel), the workgroups behind the tokens write the job
// tables of the two launches that follow, a thread per job and per share: they are uniform, so the host need not build and upload
// them (two copies of 70 and 35 KB that the stream waited for, 22 us each with 16 tokens, 128 experts and top-8).
constexpr uint32_t kRouteQuantWaves = 12;
struct JobTables { JobTableSpec t[2]; };
__device__ __forceinline__ void write_job_table(const JobTableSpec &T, uint32_t i) {
    if (!T.jobs) return;
    if (i < T.n_jobs) {
        const uint32_t slot = i / T.per_slot, second = i % T.per_slot;
        GemvJob j = T.base;
        j.w += second * T.w_second;
        j.x = reinterpret_cast<const float *>(reinterpret_cast<const uint8_t *>(j.x) + (slot / T.x_div) * T.x_step);
        j.out += slot * T.out_step + second * T.out_second;
        j.sel += slot;
        j.pass_begin = i * T.base.n_pass;
        T.jobs[i] = j;
    }
    if (T.first && i < T.grid) {  // (as the kernels cut the passes)
        const uint32_t total = (uint32_t)T.total, pass = total / T.grid * i + min(i, total % T.grid);
        T.first[i] = min(pass / T.base.n_pass, T.n_jobs - 1);
    }
}

__global__ void __launch_bounds__(kRouteQuantWaves * 64) moe_kq_route_quant_kernel(const float *__restrict__ logits, const float *__restrict__ bias, uint32_t n_experts, uint32_t k,
                                                                int policy, const float *__restrict__ scale, uint32_t *__restrict__ experts,
                                                                float *__restrict__ weights, const float *__restrict__ src, size_t src_stride,
                                                                uint32_t src_cols, uint32_t cols, uint8_t *__restrict__ dst, size_t dst_stride, uint32_t tokens,
                                                                const JobTables tables) {
    if (blockIdx.x >= tokens) {
        const uint32_t i = (blockIdx.x - tokens) * blockDim.x + threadIdx.x;
        write_job_table(tables.t[0], i);
        write_job_table(tables.t[1], i);
        return;
    }
    const uint32_t t = blockIdx.x, wave = threadIdx.x >> 6, lane = threadIdx.x & 63u;
    if (wave == 0) {
        uint32_t sel_idx[kRouterMaxK];
        float sel_w[kRouterMaxK];
        router_select_any(logits + (size_t)t * n_experts, bias, n_experts, k, policy, lane, sel_idx, sel_w);
        if (lane == 0) {
#pragma unroll
            for (int r = 0; r < kRouterMaxK; r++)
                if ((uint32_t)r < k) {
                    const uint32_t e = sel_idx[r];
                    experts[(size_t)t * k + r] = e;
                    weights[(size_t)t * k + r] = (scale && e < n_experts) ? sel_w[r] * scale[e] : sel_w[r];
                }
        }
    }
    const float *s = src + (size_t)t * src_stride;
    const bool vec = ((src_stride | src_cols) & 3u) == 0 && ((uintptr_t)src & 15u) == 0;
    if (wave > 0)
        for (uint32_t sb = wave - 1; sb < cols / 256; sb += (blockDim.x >> 6) - 1) {
            float v[4];
            load4(v, s, sb * 256 + 4 * lane, src_cols, vec);
            uint32_t codes; float sc; int sum;
            q8k_block(v, codes, sc, sum);
            q8k_store(dst + (size_t)t * dst_stride, cols, sb, lane, codes, sc, sum);
        }
}

// Row `blockIdx.y` of src ([rows, src_cols] floats, src_stride apart) zero-padded to `cols` floats at dst + row * cols:
// the expert input of a float bank whose rows are stored wider than hidden (forward.rs:176-184).
__global__ void __launch_bounds__(256) pad_rows_f32_kernel(const float *__restrict__ src, size_t src_stride, uint32_t src_cols, uint32_t cols,
                                                          float *__restrict__ dst) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= cols) return;
    dst[(size_t)blockIdx.y * cols + j] = j < src_cols ? src[(size_t)blockIdx.y * src_stride + j] : 0.0f;
}

// math::silu / math::gelu_tanh (cpu/ops/moe/math.rs:54-65) and MoeGateRule::combine (pipeline/moe.rs:73-118)
__device__ __forceinline__ float moe_combine(int rule, float g, float u, float limit, float alpha) {
    if (rule == 1) {
        const float c = 0.7978846f;
        return 0.5f * g * (1.0f + tanhf(c * (g + 0.044715f * g * g * g))) * u;
    }
    if (rule == 2) return g / (1.0f + expf(-g)) * u;
    if (rule == 3) {  // SituGlu { beta = limit, linear_beta = alpha, 0 for None }
        const float situ_a = limit * tanhf(g / limit) * (1.0f / (1.0f + expf(-g)));
        const float uc = alpha != 0.0f ? alpha * tanhf(u / alpha) : u;
        return situ_a * uc;
    }
    const float gv = fminf(g, limit);
    const float uv = u < -limit ? -limit : (u > limit ? limit : u);
    if (rule == 4) return 0.5f * gv * (1.0f + tanhf(0.7978846f * (gv + 0.044715f * gv * gv * gv))) * uv;  // ClampedGated { limit, gelu_tanh }
    if (rule == 5) return gv / (1.0f + expf(-gv)) * uv;                                                    // ClampedGated { limit, silu }
    return (uv + 1.0f) * (gv * (1.0f / (1.0f + expf(-(gv * alpha)))));
}

// Slot `blockIdx.y`'s activation: act[j] = combine(g[j] + gate bias, u[j] + up bias) for j < inter (the fused bias row
// of the slot's expert is interleaved: gate at 2j, up at 2j+1 — ExpertMlp::gate_bias / up_bias, pipeline/moe.rs:150-170),
// zeros up to inter_padded, quantised to a Q8_K activation of inter_padded elements at dst + slot * dst_stride
// (run_single_expert_kq_q8k_into, cpu/ops/moe/expert/q4k.rs:300-325).  A slot whose expert lies outside the bank gets
// no bias; its result is never read.
__global__ void __launch_bounds__(256) moe_kq_act_q8k_kernel(const float *__restrict__ g, const float *__restrict__ u, uint32_t inter, uint32_t inter_padded,
                                                            const uint32_t *__restrict__ experts, uint32_t n_experts, const float *__restrict__ gub,
                                                            int rule, float limit, float alpha, uint8_t *__restrict__ dst, size_t dst_stride) {
    const uint32_t sb = blockIdx.x * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63u;
    if (sb >= inter_padded / 256) return;
    const uint32_t slot = blockIdx.y;
    const uint32_t e = experts[slot];
    const float *b = (gub && e < n_experts) ? gub + (size_t)e * 2 * inter : nullptr;
    const uint32_t j = sb * 256 + 4 * lane;
    const bool vec = (inter & 3u) == 0 && (((uintptr_t)g | (uintptr_t)u | (uintptr_t)gub) & 15u) == 0;
    float v[4], gv[4], uv[4], b0[4] = {0.f, 0.f, 0.f, 0.f}, b1[4] = {0.f, 0.f, 0.f, 0.f};
    load4(gv, g + (size_t)slot * inter, j, inter, vec);
    load4(uv, u + (size_t)slot * inter, j, inter, vec);
    if (b) {
        load4(b0, b, 2 * j, 2 * inter, vec);
        load4(b1, b, 2 * j + 4, 2 * inter, vec);
    }
    const float bias[8] = {b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
#pragma unroll
    for (uint32_t i = 0; i < 4; i++) v[i] = j + i < inter ? moe_combine(rule, gv[i] + bias[2 * i], uv[i] + bias[2 * i + 1], limit, alpha) : 0.0f;
    uint32_t codes; float scale; int sum;
    q8k_block(v, codes, scale, sum);
    q8k_store(dst + (size_t)slot * dst_stride, inter_padded, sb, lane, codes, scale, sum);
}

// The same activation kept as f32 (a float bank: cpu_moe_forward's f32 arm, forward.rs:262-267): slot `blockIdx.y`'s row
// of `inter` floats at act + slot * act_stride.
__global__ void __launch_bounds__(256) moe_act_f32_kernel(const float *__restrict__ g, const float *__restrict__ u, uint32_t inter,
                                                         const uint32_t *__restrict__ experts, uint32_t n_experts, const float *__restrict__ gub, int rule,
                                                         float limit, float alpha, float *__restrict__ act, size_t act_stride) {
    const uint32_t j = blockIdx.x * blockDim.x + threadIdx.x, slot = blockIdx.y;
    if (j >= inter) return;
    const uint32_t e = experts[slot];
    const float *b = (gub && e < n_experts) ? gub + (size_t)e * 2 * inter : nullptr;
    const float gv = g[(size_t)slot * inter + j] + (b ? b[2 * j] : 0.0f);
    const float uv = u[(size_t)slot * inter + j] + (b ? b[2 * j + 1] : 0.0f);
    act[(size_t)slot * act_stride + j] = moe_combine(rule, gv, uv, limit, alpha);
}

hipError_t router_select_launch(hipStream_t s, const float *logits, const float *bias, uint32_t tokens, uint32_t n_experts, uint32_t k,
                                int policy, uint32_t *experts, float *weights) {
    if (tokens == 0) return hipSuccess;
    hipLaunchKernelGGL(router_select_kernel, dim3(tokens), dim3(64), 0, s, logits, bias, n_experts, k, policy, experts, weights);
    return hipGetLastError();
}
hipError_t clamped_glu_interleaved_launch(hipStream_t s, const float *gu, float *h, size_t n, float limit, float alpha) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(clamped_glu_interleaved_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, gu, h, n, limit, alpha);
    return hipGetLastError();
}
hipError_t clamped_glu_launch(hipStream_t s, const float *g, const float *u, float *h, size_t n, float limit, float alpha) {
    if (n == 0) return hipSuccess;
    hipLaunchKernelGGL(clamped_glu_kernel, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, g, u, h, n, limit, alpha);
    return hipGetLastError();
}
hipError_t expert_scale_launch(hipStream_t s, float *weights, const uint32_t *experts, const float *scale, uint32_t n, uint32_t n_scale) {
    if (n == 0 || n_scale == 0) return hipSuccess;
    hipLaunchKernelGGL(expert_scale_kernel, dim3((n + 255) / 256), dim3(256), 0, s, weights, experts, scale, n, n_scale);
    return hipGetLastError();
}

hipError_t quantize_rows_to_q8k_launch(hipStream_t s, const float *src, size_t src_stride, uint32_t src_cols, uint32_t cols, uint32_t rows,
                                       uint8_t *dst, size_t dst_stride) {
    if (rows == 0 || cols < 256) return hipSuccess;
    hipLaunchKernelGGL(quantize_rows_to_q8k_kernel, dim3((cols / 256 + 3) / 4, rows), dim3(256), 0, s, src, src_stride, src_cols, cols, dst, dst_stride);
    return hipGetLastError();
}
hipError_t moe_kq_act_q8k_launch(hipStream_t s, const float *g, const float *u, uint32_t inter, uint32_t inter_padded, uint32_t slots,
                                 const uint32_t *experts, uint32_t n_experts, const float *gub, int rule, float limit, float alpha, uint8_t *dst,
                                 size_t dst_stride) {
    if (slots == 0 || inter_padded < 256) return hipSuccess;
    hipLaunchKernelGGL(moe_kq_act_q8k_kernel, dim3((inter_padded / 256 + 3) / 4, slots), dim3(256), 0, s, g, u, inter, inter_padded, experts, n_experts,
                       gub, rule, limit, alpha, dst, dst_stride);
    return hipGetLastError();
}
hipError_t moe_kq_route_quant_launch(hipStream_t s, const float *logits, const float *bias, uint32_t tokens, uint32_t n_experts, uint32_t k, int policy,
                                     const float *scale, uint32_t *experts, float *weights, const float *src, size_t src_stride, uint32_t src_cols,
                                     uint32_t cols, uint8_t *dst, size_t dst_stride,
                                     const JobTableSpec (&tables)[2]) {
    if (tokens == 0) return hipSuccess;
    const JobTables T = {{tables[0], tables[1]}};
    uint32_t writers = 0;
    for (const JobTableSpec &t : T.t)
        if (t.jobs) writers = std::max(writers, std::max(t.n_jobs, t.first ? t.grid : 0u));
    const uint32_t threads = 64 * std::min(kRouteQuantWaves, 1 + cols / 256);
    hipLaunchKernelGGL(moe_kq_route_quant_kernel, dim3(tokens + (writers + threads - 1) / threads), dim3(threads), 0, s, logits, bias, n_experts, k, policy, scale, experts, weights, src,
                       src_stride, src_cols, cols, dst, dst_stride, tokens, T);
    return hipGetLastError();
}
hipError_t pad_rows_f32_launch(hipStream_t s, const float *src, size_t src_stride, uint32_t src_cols, uint32_t cols, uint32_t rows, float *dst) {
    if (rows == 0 || cols == 0) return hipSuccess;
    hipLaunchKernelGGL(pad_rows_f32_kernel, dim3((cols + 255) / 256, rows), dim3(256), 0, s, src, src_stride, src_cols, cols, dst);
    return hipGetLastError();
}
hipError_t moe_act_f32_launch(hipStream_t s, const float *g, const float *u, uint32_t inter, uint32_t slots, const uint32_t *experts, uint32_t n_experts,
                              const float *gub, int rule, float limit, float alpha, float *act, size_t act_stride) {
    if (slots == 0 || inter == 0) return hipSuccess;
    hipLaunchKernelGGL(moe_act_f32_kernel, dim3((inter + 255) / 256, slots), dim3(256), 0, s, g, u, inter, experts, n_experts, gub, rule, limit, alpha,
                       act, act_stride);
    return hipGetLastError();
}
hipError_t weighted_sum_launch(hipStream_t s, const float *d, const float *weights, const uint32_t *experts, uint32_t n_experts, const float *bias, float *out,
                               uint32_t tokens, uint32_t k, uint32_t hidden) {
    if (tokens == 0 || hidden == 0) return hipSuccess;
    const dim3 grid((hidden + 255) / 256, tokens);
#define LARQL_WSUM(K) \
    if (bias) hipLaunchKernelGGL((weighted_sum_kernel<K, true>), grid, dim3(256), 0, s, d, weights, experts, out, n_experts, k, hidden, bias); \
    else hipLaunchKernelGGL((weighted_sum_kernel<K, false>), grid, dim3(256), 0, s, d, weights, experts, out, n_experts, k, hidden, bias)
    switch (k) {
        case 1: LARQL_WSUM(1); break;
        case 6: LARQL_WSUM(6); break;
        case 8: LARQL_WSUM(8); break;
        default: LARQL_WSUM(0);
    }
#undef LARQL_WSUM
    return hipGetLastError();
}

}  // namespace larql
