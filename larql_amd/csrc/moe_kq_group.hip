// moe_kq_group.hip — a bank of Q4_K experts against Q8_K activations: every expert's weights are read once per group of up to
// eight of the slots (token, rank) that chose it.
//
// Bound: HBM on the distinct experts' bytes.  The arithmetic is the integer path of gemv_q4k_q8k_kernel (gemv.hip), result for
// result: A row m of an operand is sub-block m's 32 codes in the k-slots where B carries that sub-block's nibbles, four
// v_mfma_i32_16x16x64_i8 per 16 rows x 256 weights, sums in integers, d_w d_y sum1 - dmin_w d_y sum2 once per (row, super-block)
// without contraction, super-blocks added in order by one lane: bit for bit the reference's q4k_q8k_matvec_scalar.  One activation
// fills eight of the sixteen A rows, so two of a group share an operand: lanes kq = 0, 1 end with the dots of the first, kq = 2, 3
// with those of the second, and the same ~45 vector instructions serve both.  Four such operands share a tile's copy, its nibbles
// and its header.  (At HBM's pace a compute unit gets a 2304-byte wave-tile every ~216 cycles, 864 of a SIMD's.)
// FIGURES
//
// A wavefront owns one super-block column of every ways-th tile (rows of three super-blocks: twelve wavefronts, four ways; one
// workgroup per compute unit, so that its groups are found once); its tiles stream global -> LDS through a private ring; partials
// [column][slot][row] of four tiles per way meet in LDS.  A workgroup finds the groups and its share of their tiles for itself (expert_groups.h).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>

#include "expert_groups.h"
#include "kernels.h"
#include "kq.h"
#include "mx4.h"

namespace larql {

constexpr int kKgStages = 4, kKgTiles = 4, kKgSlots = 8;  // ring slots, 16-row tiles of a wavefront between two folds, slots of a group
constexpr uint32_t kKgMaxWaves = 12;                      // and super-blocks of a row: a wavefront each

struct KgCol {  // two slots' super-block: lanes whose A row (r = lane % 16) is below eight carry the first's codes
    Q4kOp xm[4];
    uint32_t bs[2];  // sub-block sums (i16) of the slot and half that this lane adds up: slot kq / 2, sub-blocks 4 (kq % 2) ..
    float dy;
};

__device__ __forceinline__ KgCol kg_load_col(const uint8_t *first, const uint8_t *second, uint32_t k, uint32_t c, uint32_t lane) {
    const uint32_t r = lane & 15u, kq = lane >> 4;
    const GLOBAL_AS uint8_t *mine = (const GLOBAL_AS uint8_t *)(r < 8 ? first : second), *sums_of = (const GLOBAL_AS uint8_t *)(kq < 2 ? first : second);
    const u32x2 codes = *(const GLOBAL_AS u32x2 *)(mine + (size_t)c * 256 + (r & 7u) * 32 + kq * 8);
    const u32x2 sums = *(const GLOBAL_AS u32x2 *)(sums_of + k + (k / 256) * 4 + (size_t)c * 16 + (kq & 1u) * 8);
    KgCol col;
    col.dy = *(const GLOBAL_AS float *)(sums_of + k + (size_t)c * 4);
    col.bs[0] = sums.x; col.bs[1] = sums.y;
#pragma unroll
    for (int g = 0; g < 4; g++) {
        const bool lo = (r & 7u) == (uint32_t)(2 * g), hi = (r & 7u) == (uint32_t)(2 * g + 1);
        col.xm[g].u[0] = lo ? codes.x : 0u; col.xm[g].u[1] = lo ? codes.y : 0u;
        col.xm[g].u[2] = hi ? codes.x : 0u; col.xm[g].u[3] = hi ? codes.y : 0u;
    }
    return col;
}

__global__ void __launch_bounds__(kKgMaxWaves * 64) moe_kq_group_kernel(const MoeKqGroupArgs A, const uint32_t ways) {
#pragma clang fp contract(off)
    extern __shared__ __attribute__((aligned(16))) uint8_t kg_lds[];
    constexpr int NS = kKgStages, R = kKgTiles, NPAIR = kKgSlots / 2;
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wv = __builtin_amdgcn_readfirstlane(tid >> 6), cols = A.cols, nw = cols * ways;
    const uint32_t col_i = wv % cols, way = wv / cols, kRows = ways * (kKgTiles * 16);
    const uint32_t jr = lane & 15u, kq = lane >> 4;
    const uint32_t nE = A.n_experts, slots = A.slots, rows = A.rows, row_bytes = cols * 144;
    uint8_t *ring = kg_lds + wv * (NS * kQ4kTileBytes);
    float *part = reinterpret_cast<float *>(kg_lds + nw * (NS * kQ4kTileBytes));  // [2][column][slot][kRows]
    const uint32_t part_floats = cols * kKgSlots * kRows;
    ExpertGroups G;
    G.cnt = reinterpret_cast<uint32_t *>(part + 2 * part_floats);
    G.before = G.cnt + nE;
    uint16_t *list = reinterpret_cast<uint16_t *>(G.before + nE + 1);  // [2][8]
    G.ex = list + 2 * kKgSlots;
    expert_groups_count<kKgSlots>(G, A.experts, slots, nE, tid, lane, wv);

    // this workgroup's share of the list (group, 16-row tile); a group opens with kStart units of its own, what its start costs
    constexpr uint32_t kStart = 3;
    const uint32_t tpm = (rows + 15) / 16, per_group = tpm * A.n_mats + kStart, units = G.before[nE] * per_group, grid = gridDim.x;
    const uint32_t share = (grid & 7u) ? blockIdx.x : (blockIdx.x & 7u) * (grid >> 3) + (blockIdx.x >> 3);  // neighbours on one XCD
    uint32_t v = (uint32_t)((uint64_t)units * share / grid);
    const uint32_t v_end = (uint32_t)((uint64_t)units * (share + 1) / grid);

    // lane's pieces of a wave-tile: 16-byte unit u = row * 9 + piece, the last 256 bytes dword by dword
    const uint32_t u1 = 64 + lane, u2 = 128 + (lane >> 2);
    const uint32_t r0 = lane / 9, r1 = u1 / 9, r2 = u2 / 9;
    const uint32_t w0 = (lane - r0 * 9) * 16, w1 = (u1 - r1 * 9) * 16, w2 = (u2 - r2 * 9) * 16 + (lane & 3u) * 4;

    uint32_t parity = 0, lpar = 0, slot_i = 0, use_i = 0;
    while (v < v_end) {
        const uint32_t gi = v / per_group, a0 = v - gi * per_group, a1 = min(a0 + (v_end - v), per_group);
        v += a1 - a0;
        if (a1 <= kStart) continue;
        const uint32_t t0 = max(a0, kStart) - kStart, t1 = a1 - kStart;
        const uint32_t e = expert_of_group(G, nE, gi, lane);
        const uint32_t lo = (gi - G.before[e]) * kKgSlots, ns = __builtin_amdgcn_readfirstlane(min(G.cnt[e] - lo, (uint32_t)kKgSlots));

        // the first tiles leave
        uint32_t it = t0 + way, flying = 0;
        auto issue = [&]() {
            const uint32_t m = it >= tpm ? 1u : 0u, rb = (it - m * tpm) * 16, lim = min(15u, rows - 1 - rb);  // (rows past the end: the last again)
            const uint8_t *gp = (m ? A.w[1] : A.w[0]) + (size_t)e * A.w_stride + (size_t)rb * row_bytes + col_i * 144;
            uint8_t *lp = ring + slot_i * kQ4kTileBytes;
            __builtin_amdgcn_global_load_lds((g_vp)(gp + min(r0, lim) * row_bytes + w0), (lds_vp)lp, 16, 0, 0);
            __builtin_amdgcn_global_load_lds((g_vp)(gp + min(r1, lim) * row_bytes + w1), (lds_vp)(lp + 1024), 16, 0, 0);
            __builtin_amdgcn_global_load_lds((g_vp)(gp + min(r2, lim) * row_bytes + w2), (lds_vp)(lp + 2048), 4, 0, 0);
            slot_i = slot_i + 1 == NS ? 0u : slot_i + 1;
            it += ways;
            flying++;
        };
#pragma unroll
        for (int q = 0; q < NS - 1; q++)
            if (it < t1) issue();

        uint16_t *const gl = list + lpar * kKgSlots;
        expert_group_slots<kKgSlots>(G, slots, e, lo, gl, lane);
        KgCol col[NPAIR];  // (of slots that there are not: the group's first again, not stored)
#pragma unroll
        for (int p = 0; p < NPAIR; p++) {
            const uint32_t a = gl[2 * p < (int)ns ? 2 * p : 0], b = gl[2 * p + 1 < (int)ns ? 2 * p + 1 : 0];
            if (2 * p < (int)ns) col[p] = kg_load_col(A.x + (a / A.x_div) * A.x_stride, A.x + (b / A.x_div) * A.x_stride, cols * 256, col_i, lane);
        }

        for (uint32_t tb = t0; tb < t1; tb += R * ways) {
            float *pb = part + parity * part_floats;
            for (uint32_t tl = 0; tl < (uint32_t)R && tb + tl * ways + way < t1; tl++) {
                if (it < t1) issue();
                const uint32_t younger = --flying;  // tiles requested after this one
                if (younger >= 3) LARQL_WAIT_VMCNT(9);
                else if (younger == 2) LARQL_WAIT_VMCNT(6);
                else if (younger == 1) LARQL_WAIT_VMCNT(3);
                else LARQL_WAIT_VMCNT(0);
                asm volatile("" ::: "memory");
                const uint8_t *sp = ring + use_i * kQ4kTileBytes + jr * 144;
                use_i = use_i + 1 == NS ? 0u : use_i + 1;
                const u32x4 hdr = *reinterpret_cast<const u32x4 *>(sp);
                Q4kOp b[4];
#pragma unroll
                for (int g = 0; g < 4; g++) {
                    const u32x2 q = *reinterpret_cast<const u32x2 *>(sp + 16 + 32 * g + 8 * kq);
                    b[g].u[0] = q.x & 0x0F0F0F0Fu; b[g].u[1] = q.y & 0x0F0F0F0Fu;
                    b[g].u[2] = (q.x >> 4) & 0x0F0F0F0Fu; b[g].u[3] = (q.y >> 4) & 0x0F0F0F0Fu;
                }
                // this lane's four sub-blocks: 4 (kq % 2) .. + 3
                const bool upper = (kq & 1u) != 0;
                const uint32_t sc4 = upper ? ((hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u)) : (hdr.y & 0x3F3F3F3Fu);
                const uint32_t mn4 = upper ? (((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u)) : (hdr.z & 0x3F3F3F3Fu);
                const float d_w = half_bits_to_float(hdr.x & 0xFFFFu), dmin_w = half_bits_to_float(hdr.x >> 16);
                float *pr = pb + (col_i * kKgSlots + (kq >> 1)) * kRows + (tl * ways + way) * 16 + jr;
#pragma unroll
                for (int p = 0; p < NPAIR; p++) {
                    if (2 * p < (int)ns) {
                        i32x4 D = {0, 0, 0, 0};
#pragma unroll
                        for (int g = 0; g < 4; g++) D = __builtin_amdgcn_mfma_i32_16x16x64_i8(col[p].xm[g].v, b[g].v, D, 0, 0, 0);
                        // |dot| <= 32*15*127 and |bsum| <= 32*127: the products fit 24-bit multiplies
                        int s1 = __mul24((int)(sc4 & 0xFFu), D[0]) + __mul24((int)((sc4 >> 8) & 0xFFu), D[1]) +
                                 __mul24((int)((sc4 >> 16) & 0xFFu), D[2]) + __mul24((int)(sc4 >> 24), D[3]);
                        const int b0 = (int)(int16_t)(col[p].bs[0] & 0xFFFFu), b1 = (int)col[p].bs[0] >> 16;
                        const int b2 = (int)(int16_t)(col[p].bs[1] & 0xFFFFu), b3 = (int)col[p].bs[1] >> 16;
                        int s2 = __mul24((int)(mn4 & 0xFFu), b0) + __mul24((int)((mn4 >> 8) & 0xFFu), b1) +
                                 __mul24((int)((mn4 >> 16) & 0xFFu), b2) + __mul24((int)(mn4 >> 24), b3);
                        s1 += __shfl_xor(s1, 16);  // sub-blocks 0..3 + 4..7
                        s2 += __shfl_xor(s2, 16);
                        float p1 = d_w * col[p].dy;
                        p1 = p1 * (float)s1;
                        float p2 = dmin_w * col[p].dy;
                        p2 = p2 * (float)s2;
                        if (!upper) pr[2 * p * kRows] = p1 - p2;
                    }
                }
                asm volatile("" ::: "memory");  // (the slot's reads are done before the next copies into it are asked for)
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            // a lane per (slot, row): super-blocks in order.  `ways` wavefronts hold the rows of a batch, so the slots go round `cols`
            // sets of them
            const uint32_t rr = (wv % ways) * 64 + lane, tile = tb + rr / 16, m = tile >= tpm ? 1u : 0u, row = (tile - m * tpm) * 16 + (rr & 15u);
            for (uint32_t s = wv / ways; s < ns; s += cols) {
                const float *pv = pb + s * kRows + rr;
                float acc = 0.f;
#pragma unroll 4
                for (uint32_t c = 0; c < cols; c++) acc += pv[c * (kKgSlots * kRows)];
                if (tile < t1 && row < rows) ((g_f32wp)(m ? A.out[1] : A.out[0]))[(size_t)gl[s] * rows + row] = acc;
            }
            parity ^= 1u;
        }
        lpar ^= 1u;
    }
    LARQL_WAIT_VMCNT(0);
}

static size_t kg_lds_bytes(uint32_t cols, uint32_t ways, uint32_t n_experts, uint32_t slots) {
    return (size_t)cols * ways * (kKgStages * kQ4kTileBytes + 2 * kKgSlots * kKgTiles * 16 * sizeof(float)) +
           (2 * (size_t)n_experts + 1) * sizeof(uint32_t) + (2 * kKgSlots + (size_t)slots) * sizeof(uint16_t);
}
static uint32_t kg_ways(uint32_t cols, uint32_t n_experts, uint32_t slots) {  // 0: not served
    for (uint32_t ways = cols ? kKgMaxWaves / cols : 0; ways > 0; ways--)
        if (kg_lds_bytes(cols, ways, n_experts, slots) <= 160 * 1024) return ways;
    return 0;
}

bool moe_kq_group_serves(uint32_t rows, uint32_t cols, uint32_t n_experts, uint32_t slots) {
    return rows >= 1 && rows < (1u << 22) && slots >= 1 && slots <= kMoeGroupMaxSlots && n_experts >= 1 && n_experts <= kMoeGroupMaxExperts &&
           kg_ways(cols, n_experts, slots) != 0;
}

hipError_t moe_kq_group_launch(hipStream_t s, const MoeKqGroupArgs &A, uint32_t cu_count) {
    if (!moe_kq_group_serves(A.rows, A.cols, A.n_experts, A.slots) || A.n_mats < 1 || A.n_mats > 2) return hipErrorInvalidValue;
    static std::atomic<bool> allowed{false};  // dynamic LDS above 64 KB has to be allowed once per kernel
    if (!allowed) {
        const hipError_t e = hipFuncSetAttribute((const void *)moe_kq_group_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
        allowed = true;
    }
    const uint32_t ways = kg_ways(A.cols, A.n_experts, A.slots);
    hipLaunchKernelGGL(moe_kq_group_kernel, dim3(cu_count), dim3(A.cols * ways * 64), kg_lds_bytes(A.cols, ways, A.n_experts, A.slots), s, A, ways);
    return hipGetLastError();
}

}  // namespace larql
