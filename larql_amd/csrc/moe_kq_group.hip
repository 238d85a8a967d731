// moe_kq_group.hip — a bank of Q4_K or Q6_K experts against Q8_K activations: every expert's weights are read once per group of
// up to eight of the slots (token, rank) that chose it.
//
// Bound: HBM on the distinct experts' bytes.  The arithmetic is the integer path of the per-slot kernels (gemv.hip), result for
// result: sums in integers, the reference's float expression once per (row, super-block) without contraction, super-blocks added in
// order by one lane: bit for bit q4k_q8k_matvec_scalar / q6k_q8k_matvec_scalar.
//   * Q4_K: A row m of an operand is sub-block m's 32 codes in the k-slots where B carries that sub-block's nibbles, four
//     v_mfma_i32_16x16x64_i8 per 16 rows x 256 weights.  One activation fills eight of the sixteen A rows, so two of a group share
//     an operand: lanes kq = 0, 1 end with the dots of the first, kq = 2, 3 with those of the second, and the same ~45 vector
//     instructions serve both.  Four such operands share a tile's copy, its nibbles and its header.
//   * Q6_K: one MFMA covers 64 weights = four scale groups; A row 4g + a is activation a's codes of group g in that group's k-slots,
//     so four activations share an operand, lane (row, rq) ends with the four dots of group rq, the -32 comes in as the MFMA's
//     third operand, and three lane swaps leave lane group a with activation a's sum over all sixteen groups.
// (At HBM's pace a compute unit gets a 2304-byte wave-tile every ~216 cycles, 864 of a SIMD's.)
// Layer calls with a matvec per slot / with groups, us, all else equal.  Q4_K, 128 experts, top-8, 2816 x 704: 1 token 32.3 / 29.4, 4
// 45.4 / 42.3, 16 88.1 / 80.2, 64 281 / 142; 32 tokens of 64 experts, top-8, 2048 x 512 90.4 / 60.6, 2560 x 640 121 / 74.0; 64 tokens of 32
// experts, top-8, 3072 x 768 252 / 99.6, of 64 experts, top-4, 1024 x 256 47.3 / 40.3; 1 token of 32 experts, top-4, 1536 x 256 28.8 / 26.1.
// Q6_K (K-slice kernel), the same: 33.6 / 31.7, 49.2 / 49.8, 132 / 110, 421 / 182; 111 / 56.7, 180 / 77.2; 400 / 100, 49.1 / 42.4; 25.5 / 24.0.
//
// A wavefront owns one super-block column of every ways-th tile (rows of three super-blocks: twelve wavefronts, four ways; one
// workgroup per compute unit, so that its groups are found once); its tiles stream global -> LDS through a private ring; partials
// [column][slot][row] of a few tiles per way meet in LDS.  A workgroup finds the groups and its share of their tiles for itself
// (expert_groups.h).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "expert_groups.h"
#include "kernels.h"
#include "kq.h"
#include "mx4.h"

namespace larql {

constexpr int kKgSlots = 8;               // slots of a group
constexpr uint32_t kKgMaxWaves = 12;      // and super-blocks of a row: a wavefront each
template <bool Q6> struct KgFormat;       // ring slots, 16-row tiles of a wavefront between two folds (what LDS has room for), bytes, copies
template <> struct KgFormat<false> { static constexpr int kStages = 4, kTiles = 4, kCopies = 3; static constexpr uint32_t kBlock = 144, kTileBytes = kQ4kTileBytes; };
// (the pieces of a Q6_K tile as gemv_q6k_mfma_kernel copies them: 13 sixteen-byte pieces per row, and the block's last 16 bytes for d)
template <> struct KgFormat<true> { static constexpr int kStages = 3, kTiles = 2, kCopies = 4; static constexpr uint32_t kBlock = 210, kTileBytes = 16 * 208 + 256; };

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

struct KgCol6 {  // four slots' super-block: A row 4g + a holds slot a's codes of group 4m + g (m: the MFMA)
    Q4kOp xm[4];
    i32x4 c[4];  // -32 * the sums of the four slots' codes over this lane's group 4m + kq
    float dy;    // of slot kq
};

__device__ __forceinline__ KgCol6 kg_load_col6(const uint8_t *const (&of)[4], uint32_t k, uint32_t c, uint32_t lane) {
    const uint32_t r = lane & 15u, kq = lane >> 4, a = r & 3u;
    const uint8_t *mine = a == 0 ? of[0] : a == 1 ? of[1] : a == 2 ? of[2] : of[3];
    const uint8_t *scale_of = kq == 0 ? of[0] : kq == 1 ? of[1] : kq == 2 ? of[2] : of[3];
    KgCol6 col;
    col.dy = *(const GLOBAL_AS float *)(scale_of + k + (size_t)c * 4);
    u32x4 codes[4];
#pragma unroll
    for (int m = 0; m < 4; m++) codes[m] = *(const GLOBAL_AS u32x4 *)(mine + (size_t)c * 256 + 64 * m + 16 * kq);
#pragma unroll
    for (int m = 0; m < 4; m++) {
        const bool here = (r >> 2) == kq;
        int sum = 0;
#pragma unroll
        for (int i = 0; i < 4; i++) {
            col.xm[m].u[i] = here ? codes[m][i] : 0u;
            sum = __builtin_amdgcn_sdot4(0x01010101, (int)codes[m][i], sum, false);
        }
#pragma unroll
        for (int q = 0; q < 4; q++) col.c[m][q] = -32 * __shfl(sum, (int)(kq * 20 + q), 64);  // (lane 16 kq + 4 kq + q: slot q, group kq)
    }
    return col;
}

template <bool Q6>
__global__ void __launch_bounds__(kKgMaxWaves * 64)
    moe_kq_group_kernel(const uint32_t *experts, uint32_t slots, uint32_t nE, uint32_t cols, uint32_t ways, uint32_t rows,
                        uint32_t grid,  // (in registers when the wavefront starts: the way to the experts' ids)
                        const MoeKqGroupArgs A) {
#pragma clang fp contract(off)
    extern __shared__ __attribute__((aligned(16))) uint8_t kg_lds[];
    typedef KgFormat<Q6> F;
    constexpr int NS = F::kStages, R = F::kTiles, L = F::kCopies, SET = Q6 ? 4 : 2, NSET = kKgSlots / SET;  // SET: slots that share an operand
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wv = __builtin_amdgcn_readfirstlane(tid >> 6), nw = cols * ways;
    const uint32_t kRows = ways * (R * 16);
    uint32_t col_i = wv, way = 0;
    while (col_i >= cols) { col_i -= cols; way++; }
    const uint32_t jr = lane & 15u, kq = lane >> 4;
    const uint32_t row_bytes = cols * F::kBlock;
    uint8_t *ring = kg_lds + wv * (NS * F::kTileBytes);
    float *part = reinterpret_cast<float *>(kg_lds + nw * (NS * F::kTileBytes));  // [2][column][slot][kRows]
    const uint32_t part_floats = cols * kKgSlots * kRows;
    ExpertGroups G;
    G.cnt = reinterpret_cast<uint32_t *>(part + 2 * part_floats);
    G.before = G.cnt + nE;
    uint16_t *list = reinterpret_cast<uint16_t *>(G.before + nE + 1);  // [2][8]
    G.ex = list + 2 * kKgSlots;
    expert_groups_count<kKgSlots>(G, experts, slots, nE, tid, lane, wv);

    // this workgroup's share of the list (group, 16-row tile); a group opens with kStart units of its own, what its start costs
    // (42 layer calls a format, with 1 / 3 / 6 of them: Q4_K 1.02 / 1 / 1.00, Q6_K 1.03 / 1 / 0.99 of the time)
    constexpr uint32_t kStart = 3;
    const uint32_t tpm = (rows + 15) / 16, per_group = tpm * A.n_mats + kStart, units = __builtin_amdgcn_readfirstlane(G.before[nE]) * per_group;
    const uint32_t share = (grid & 7u) ? blockIdx.x : (blockIdx.x & 7u) * (grid >> 3) + (blockIdx.x >> 3);  // neighbours on one XCD
    uint32_t v, v_end;
    expert_group_share(units, share, grid, v, v_end);

    // lane's pieces of a wave-tile: row and place there.  Q4_K: 16-byte unit u = row * 9 + piece, the last 256 bytes dword by dword;
    // Q6_K: u = row * 13 + piece (u < 208), and lanes 16..31 of the fourth copy bring the end of row lane - 16
    uint32_t pr[L], po[L];
#pragma unroll
    for (int i = 0; i < L; i++) {
        if (Q6) {
            const uint32_t u = min(64u * i + lane, 207u);
            pr[i] = u / 13;
            po[i] = (u - pr[i] * 13) * 16;
            if (i == 3 && lane >= 16) { pr[i] = lane & 15u; po[i] = 194; }
        } else {
            const uint32_t u = i < 2 ? 64u * i + lane : 128 + (lane >> 2);
            pr[i] = u / 9;
            po[i] = (u - pr[i] * 9) * 16 + (i < 2 ? 0u : (lane & 3u) * 4);
        }
    }

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
            const uint8_t *gp = (m ? A.w[1] : A.w[0]) + (size_t)e * A.w_stride + (size_t)rb * row_bytes + col_i * F::kBlock;
            uint8_t *lp = ring + slot_i * F::kTileBytes;
            __builtin_amdgcn_global_load_lds((g_vp)(gp + min(pr[0], lim) * row_bytes + po[0]), (lds_vp)lp, 16, 0, 0);
            __builtin_amdgcn_global_load_lds((g_vp)(gp + min(pr[1], lim) * row_bytes + po[1]), (lds_vp)(lp + 1024), 16, 0, 0);
            const uint8_t *g2 = gp + min(pr[2], lim) * row_bytes + po[2];
            if constexpr (Q6) {
                __builtin_amdgcn_global_load_lds((g_vp)g2, (lds_vp)(lp + 2048), 16, 0, 0);
                if (lane < 32) __builtin_amdgcn_global_load_lds((g_vp)(gp + min(pr[L - 1], lim) * row_bytes + po[L - 1]), (lds_vp)(lp + 3072), 16, 0, 0);
            } else {
                __builtin_amdgcn_global_load_lds((g_vp)g2, (lds_vp)(lp + 2048), 4, 0, 0);
            }
            slot_i = slot_i + 1 == NS ? 0u : slot_i + 1;
            it += ways;
            flying++;
        };
#pragma unroll
        for (int q = 0; q < NS - 1; q++)
            if (it < t1) issue();

        uint16_t *const gl = list + lpar * kKgSlots;
        expert_group_slots<kKgSlots>(G, slots, e, lo, gl, lane);
        std::conditional_t<Q6, KgCol6, KgCol> col[NSET];  // (of slots that there are not: the group's first again, not stored)
#pragma unroll
        for (int p = 0; p < NSET; p++) {
            if (SET * p < (int)ns) {
                const uint8_t *of[SET];
#pragma unroll
                for (int q = 0; q < SET; q++) of[q] = A.x + (gl[SET * p + q < (int)ns ? SET * p + q : 0] / A.x_div) * A.x_stride;
                if constexpr (Q6) col[p] = kg_load_col6(of, cols * 256, col_i, lane);
                else col[p] = kg_load_col(of[0], of[1], cols * 256, col_i, lane);
            }
        }

        for (uint32_t tb = t0; tb < t1; tb += R * ways) {
            float *pb = part + parity * part_floats;
            for (uint32_t tl = 0; tl < (uint32_t)R && tb + tl * ways + way < t1; tl++) {
                if (it < t1) issue();
                const uint32_t younger = --flying;  // tiles requested after this one
                if (NS > 3 && younger >= 3) LARQL_WAIT_VMCNT(3 * L);
                else if (younger >= 2) LARQL_WAIT_VMCNT(2 * L);
                else if (younger == 1) LARQL_WAIT_VMCNT(L);
                else LARQL_WAIT_VMCNT(0);
                asm volatile("" ::: "memory");
                const uint8_t *slot = ring + use_i * F::kTileBytes, *sp = slot + jr * (Q6 ? 208 : 144);
                use_i = use_i + 1 == NS ? 0u : use_i + 1;
                if constexpr (Q6) {
                    u32x4 ql[2], qh[2];
#pragma unroll
                    for (int h = 0; h < 2; h++) {
                        ql[h] = *reinterpret_cast<const u32x4 *>(sp + 64 * h + 16 * kq);
                        qh[h] = *reinterpret_cast<const u32x4 *>(sp + 128 + 32 * h + 16 * (kq & 1u));
                    }
                    const u32x4 scs = *reinterpret_cast<const u32x4 *>(sp + 192);
                    const float d_w = half_bits_to_float(*reinterpret_cast<const uint32_t *>(slot + 16 * 208 + 16 * jr + 12) >> 16);
                    // (nibbles and top bits as in q6k_mfma_dot)
                    const uint32_t s0 = 2u * (kq >> 1), sl = 4u - s0;
                    Q4kOp b[4];
                    int sc[4];
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        const int h = m >> 1;
#pragma unroll
                        for (int i = 0; i < 4; i++)
                            b[m].u[i] = (m & 1) ? ((qh[h][i] >> s0) & 0x30303030u) | ((ql[h][i] >> 4) & 0x0F0F0F0Fu)
                                                : ((qh[h][i] << sl) & 0x30303030u) | (ql[h][i] & 0x0F0F0F0Fu);
                        sc[m] = (int)(int8_t)(scs[m] >> (8u * kq));
                    }
                    float *pw = pb + (col_i * kKgSlots + kq) * kRows + (tl * ways + way) * 16 + jr;
#pragma unroll
                    for (int p = 0; p < NSET; p++) {
                        if (SET * p < (int)ns) {
                            // |sum (q-32)*y| <= 16*32*127 over a group: the products with the int8 scales fit 24-bit multiplies
                            int s1[4] = {0, 0, 0, 0};
#pragma unroll
                            for (int m = 0; m < 4; m++) {
                                const i32x4 D = __builtin_amdgcn_mfma_i32_16x16x64_i8(col[p].xm[m].v, b[m].v, col[p].c[m], 0, 0, 0);
#pragma unroll
                                for (int q = 0; q < 4; q++) s1[q] += __mul24(sc[m], D[q]);
                            }
                            // over the four lane groups: halves of slots 0, 2 and of 1, 3 change places, then rows of 16
                            const auto x = __builtin_amdgcn_permlane32_swap((uint32_t)s1[0], (uint32_t)s1[2], false, false);
                            const auto y = __builtin_amdgcn_permlane32_swap((uint32_t)s1[1], (uint32_t)s1[3], false, false);
                            const auto z = __builtin_amdgcn_permlane16_swap(x[0] + x[1], y[0] + y[1], false, false);
                            float term = d_w * col[p].dy;
                            term = term * (float)(int)(z[0] + z[1]);
                            pw[4 * p * kRows] = term;
                        }
                    }
                } else {
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
                    float *pw = pb + (col_i * kKgSlots + (kq >> 1)) * kRows + (tl * ways + way) * 16 + jr;
#pragma unroll
                    for (int p = 0; p < NSET; p++) {
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
                            if (!upper) pw[2 * p * kRows] = p1 - p2;
                        }
                    }
                }
                asm volatile("" ::: "memory");  // (the slot's reads are done before the next copies into it are asked for)
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            // A lane per (slot, row): super-blocks in order.  A batch has kRows rows, R * 16 per way; a wavefront takes 64 / (R * 16)
            // slots of one way's rows (Q4_K: one slot; Q6_K: two of 32 rows each), and the slots go round `cols` sets of wavefronts.
            constexpr uint32_t kWayRows = R * 16, kFoldSlots = 64 / kWayRows;
            const uint32_t rr = (wv % ways) * kWayRows + lane % kWayRows, tile = tb + rr / 16, m = tile >= tpm ? 1u : 0u, row = (tile - m * tpm) * 16 + (rr & 15u);
            for (uint32_t s = (wv / ways) * kFoldSlots + lane / kWayRows; s < ns; s += cols * kFoldSlots) {
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

template <bool Q6>
static size_t kg_lds_bytes(uint32_t cols, uint32_t ways, uint32_t n_experts, uint32_t slots) {
    typedef KgFormat<Q6> F;
    return (size_t)cols * ways * (F::kStages * F::kTileBytes + 2 * kKgSlots * F::kTiles * 16 * sizeof(float)) +
           (2 * (size_t)n_experts + 1) * sizeof(uint32_t) + (2 * kKgSlots + (size_t)slots) * sizeof(uint16_t);
}
template <bool Q6>
static uint32_t kg_ways(uint32_t cols, uint32_t n_experts, uint32_t slots) {  // 0: not served
    for (uint32_t ways = cols ? kKgMaxWaves / cols : 0; ways > 0; ways--)
        if (kg_lds_bytes<Q6>(cols, ways, n_experts, slots) <= 160 * 1024) return ways;
    return 0;
}

// Rows of up to twelve super-blocks (a wavefront each) and as many slots as the lists have LDS for: kMoeGroupMaxSlots with fewer ways
// where that helps, but Q4_K rows of twelve super-blocks leave room for 1518 slots of 128 experts, 1006 of 256.  Beyond, every slot
// reads its expert again: 128 experts, top-8, 3072 x 256, 189 / 190 tokens 138 / 342 us (Q6_K 142 / 143).
bool moe_kq_group_serves(bool q6, uint32_t rows, uint32_t cols, uint32_t n_experts, uint32_t slots) {
    return rows >= 1 && rows < (1u << 22) && slots >= 1 && slots <= kMoeGroupMaxSlots && n_experts >= 1 && n_experts <= kMoeGroupMaxExperts &&
           (q6 ? kg_ways<true>(cols, n_experts, slots) : kg_ways<false>(cols, n_experts, slots)) != 0;
}

template <bool Q6>
static hipError_t kg_launch(hipStream_t s, const MoeKqGroupArgs &A, uint32_t cu_count) {
    static std::atomic<bool> allowed{false};  // dynamic LDS above 64 KB has to be allowed once per kernel
    if (!allowed) {
        const hipError_t e = hipFuncSetAttribute((const void *)moe_kq_group_kernel<Q6>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
        allowed = true;
    }
    const uint32_t ways = kg_ways<Q6>(A.cols, A.n_experts, A.slots);
    hipLaunchKernelGGL(moe_kq_group_kernel<Q6>, dim3(cu_count), dim3(A.cols * ways * 64), kg_lds_bytes<Q6>(A.cols, ways, A.n_experts, A.slots), s, A.experts, A.slots,
                       A.n_experts, A.cols, ways, A.rows, cu_count, A);
    return hipGetLastError();
}

hipError_t moe_kq_group_launch(hipStream_t s, bool q6, const MoeKqGroupArgs &A, uint32_t cu_count) {
    if (!moe_kq_group_serves(q6, A.rows, A.cols, A.n_experts, A.slots) || A.n_mats < 1 || A.n_mats > 2) return hipErrorInvalidValue;
    return q6 ? kg_launch<true>(s, A, cu_count) : kg_launch<false>(s, A, cu_count);
}

}  // namespace larql
