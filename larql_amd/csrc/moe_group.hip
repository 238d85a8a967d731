// moe_group.hip — several tokens through a bank of MXFP4 experts: every expert's weights are read once per group of up to
// sixteen of the tokens that chose it.
//
// Bound: HBM on the distinct experts' bytes while a group is at most full (16 tokens x 3 terms are 12 MFMAs of 16 cycles per
// 16 x 128 weights: 0.48 us of matrix pipe per 16-row tile of 2880 elements, whose 24.5 KB take 0.85 us of a CU's share of
// HBM).  The arithmetic is the matrix-core scheme of the one-token kernels (gemv.hip): the 16 "B" columns are weight rows
// converted from FP4 exactly, the "A" rows are activations as three exact bf16 terms, a wavefront owns a K-range of CW
// 128-element steps, its weight tiles stream global -> LDS through a private ring, the row partials of the wavefronts meet
// in LDS and are added in wavefront order.  A token's additions are those of a group of any size, so a result does not
// depend on who else is in the block, bit for bit.
//   * TG = 16: one A operand per term, 16 tokens each: three MFMAs share a converted weight operand.  The operands of all
//     steps stay in registers (12 CW times 4 VGPRs; with four steps, rows of 3073 to 4096 elements, all 256 are taken and 9 or 12
//     values go through scratch: its loads and stores only make the counted waits stricter).
//   * TG = 4: one A operand holds four tokens' terms (row 4t + i = term i of token t): a third of the MFMAs and operand
//     loads, for blocks whose experts have few tokens each.
// The activations arrive as terms, split once (moe_route_terms_kernel, and this kernel's gate/up stage for the down stage):
// splitting them in every share cost a share of a four-token job ~3000 instructions before its first tile.
//
// No job table: a workgroup counts the slots (token, rank) per expert in LDS from the router's choice (at most 4096 ids),
// which gives it the list of groups and its share of their row tiles; a planning launch on one workgroup took 43 us for 512
// slots.  Figures: see mg_launch_stage.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>

#include "expert_groups.h"
#include "kernels.h"
#include "mx4.h"
#include "router.h"

namespace larql {

// Weight tiles in the ring of a wavefront.  (Four with half the tiles between folds: 5 % slower; it is not the depth that bounds.)
constexpr int kMgStages = 3;
constexpr uint32_t kMgStepBytes = 1024;
typedef float float2_t __attribute__((ext_vector_type(2)));
constexpr int mg_tiles(int cw, int tg) { return tg == 4 ? (cw <= 4 ? 8 : 2) : (cw <= 3 ? 4 : 2); }  // 16-row tiles between two folds (what LDS has room for)
constexpr uint32_t mg_slot_bytes(int cw) { return (uint32_t)cw * kMgStepBytes + (cw > 4 ? 512u : 256u); }
__device__ const uint32_t kMgZeros[4] = {0u, 0u, 0u, 0u};  // what an operand lane without an activation loads

// Where element e of a row of terms stands: within a step of 128 elements, in the order in which the operand loads want them —
// load m takes elements 32kg + 8m .. + 7 from the four lanes kg of a row, which then are 64 neighbouring bytes.  (In plain
// order a load touched 64 different lines: 8 us per start of a 16-token group instead of 2.)
__device__ __forceinline__ uint32_t moe_term_at(uint32_t e) { return (e & ~127u) | ((e & 24u) << 2) | ((e & 96u) >> 2) | (e & 7u); }

template <bool DOWN, int CW, int TG>
__global__ void __launch_bounds__(512)
    moe_group_kernel(const uint32_t *experts, uint32_t slots, uint32_t nE, uint32_t kdim, uint32_t rows,
                     uint32_t grid,  // (in registers when the wavefront starts: the way to the experts' ids)
                     const MoeGroupArgs A) {
    extern __shared__ __attribute__((aligned(16))) uint8_t mg_lds[];
    constexpr int NS = kMgStages, R = mg_tiles(CW, TG), NT = TG == 16 ? 3 : 1, TP = TG / 2;  // NT: A operands, TP: pairs of tokens
    constexpr uint32_t slot_bytes = mg_slot_bytes(CW);
    constexpr int L = CW + 1 + (CW > 4);  // copies per tile
    const uint32_t tid = threadIdx.x, lane = tid & 63u, wv = __builtin_amdgcn_readfirstlane(tid >> 6), nw = blockDim.x >> 6;
    const uint32_t jr = lane & 15u, kg = lane >> 4;
    const uint32_t nb = kdim / 32, row_bytes = nb * 16, steps = (kdim + 127) / 128;
    const uint32_t tpm = rows / 16;
    uint8_t *ring = mg_lds + wv * (NS * slot_bytes);
    float *part = reinterpret_cast<float *>(mg_lds + nw * (NS * slot_bytes));  // [2][R][nw][16 rows][TG tokens]
    const uint32_t part_floats = R * nw * 16 * TG;
    float *lbias = part + 2 * part_floats;                                    // [2][R * 16]: the biases of a batch's rows
    ExpertGroups G;
    G.cnt = reinterpret_cast<uint32_t *>(lbias + 2 * R * 16);
    G.before = G.cnt + nE;
    uint16_t *list = reinterpret_cast<uint16_t *>(G.before + nE + 1);         // [2][16]: the slots of a group
    G.ex = list + 32;
    const uint32_t step0 = wv * CW;  // (below `steps`: the launch has no more wavefronts than K-ranges)

    // 1. slots per expert, groups before each expert
    expert_groups_count<TG>(G, experts, slots, nE, tid, lane, wv);

    // 2. this workgroup's share of the list (group, 16-row tile).  Workgroups are dealt to the eight XCDs in turn: an XCD
    //    takes neighbouring shares, whose groups' operands then sit in its L2.
    //    A group opens with kStart units of its own: who meets a second group in its share starts twice (list, operands, first
    //    tiles), so it gets that many tiles fewer.
    constexpr uint32_t kStart = TG == 16 ? 6 : 4;
    const uint32_t per_group = tpm + kStart, units = __builtin_amdgcn_readfirstlane(G.before[nE]) * per_group;
    const uint32_t share = (grid & 7u) ? blockIdx.x : (blockIdx.x & 7u) * (grid >> 3) + (blockIdx.x >> 3);
    uint32_t v, v_end;
    expert_group_share(units, share, grid, v, v_end);

    // per-lane parts of a tile's addresses: the block of each step, clamped into the row (a step past the row end meets
    // zero activations), and where its scale byte lies in the slot
    uint32_t blk[CW], sc_at[CW];
#pragma unroll
    for (int s = 0; s < CW; s++) {
        const uint32_t b = min((step0 + s) * 4 + kg, nb - 1);
        blk[s] = b * 16;
        sc_at[s] = (16u * s + jr) * 4 + (b - min((step0 + s) * 4, nb - 4));
    }
    const uint32_t sc_dw = min((step0 + kg) * 4, nb - 4), sc_dw4 = min((step0 + 4) * 4, nb - 4);
    // virtual row r of a gate/up pair kept apart: gate row r/2 (r even) or up row r/2 (r odd), as a fused matrix interleaves them
    const uint32_t lane_row = A.split ? jr >> 1 : jr, tile_rows = A.split ? 8u : 16u;
    const uint8_t *mat = A.split && (jr & 1u) ? A.w[1] : A.w[0], *smat = A.split && (jr & 1u) ? A.aux[1] : A.aux[0];

    const uint32_t fold_at = wv < 4 ? 0u : (uint32_t)R / 2;
    uint32_t parity = 0, lpar = 0, turn = 0, slot_i = 0, use_i = 0;
    while (v < v_end) {
        const uint32_t gi = v / per_group, a0 = v - gi * per_group, a1 = min(a0 + (v_end - v), per_group);
        v += a1 - a0;
        if (a1 <= kStart) continue;
        const uint32_t t0 = max(a0, kStart) - kStart, nt = a1 - kStart - t0;
        const uint32_t e = expert_of_group(G, nE, gi, lane);
        const uint32_t lo = (gi - G.before[e]) * TG, ntok = min(G.cnt[e] - lo, (uint32_t)TG);

        // 3. the first tiles leave
        const uint8_t *wp = mat + (size_t)e * A.w_stride + (size_t)(t0 * tile_rows + lane_row) * row_bytes;
        const uint8_t *sp = smat + (size_t)e * A.aux_stride + (size_t)(t0 * tile_rows + lane_row) * nb;
        const uint32_t w_adv = tile_rows * row_bytes, s_adv = tile_rows * nb;
        uint32_t left = nt;
        auto issue = [&]() {
            uint8_t *lp = ring + slot_i * slot_bytes;
#pragma unroll
            for (int s = 0; s < CW; s++) __builtin_amdgcn_global_load_lds((g_vp)(wp + blk[s]), (lds_vp)(lp + s * kMgStepBytes), 16, 0, 0);
            // the scale bytes of all steps: lane (row, step) brings the dword of its row and step
            __builtin_amdgcn_global_load_lds((g_vp)(sp + sc_dw), (lds_vp)(lp + CW * kMgStepBytes), 4, 0, 0);
            if (CW > 4) __builtin_amdgcn_global_load_lds((g_vp)(sp + sc_dw4), (lds_vp)(lp + CW * kMgStepBytes + 256), 4, 0, 0);
            slot_i = slot_i + 1 == NS ? 0u : slot_i + 1;
            wp += w_adv;
            sp += s_adv;
            left--;
        };
#pragma unroll
        for (int q = 0; q < NS - 1; q++)
            if (left) issue();

        // 4. the group's slots: those of rank lo .. lo+TG-1 among the expert's, in slot order (every wavefront finds them
        //    for itself and writes the same list)
        uint16_t *const gl = list + lpar * 16;
        expert_group_slots<TG>(G, slots, e, lo, gl, lane);

        // 5. the A operands of the wavefront's K-range
        BfOp a[NT][CW][4];
        {
            const uint32_t token = TG == 16 ? jr : jr >> 2, slot = token < ntok ? gl[token] : 0u;
            const uint32_t src_row = DOWN ? slot : slot / A.k;
#pragma unroll
            for (int t = 0; t < NT; t++) {
                const uint32_t term = TG == 16 ? (uint32_t)t : jr & 3u;
                const bool mine = token < ntok && term < 3u;
                const uint16_t *tp = A.terms_in + ((size_t)min(term, 2u) * A.in_rows + src_row) * (steps * 128);
#pragma unroll
                for (int s = 0; s < CW; s++)
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        const uint32_t el = (step0 + s) * 128 + 32 * kg + 8 * m;  // (kdim % 32 == 0: eight elements are inside or outside)
                        const uint16_t *src = mine && el < kdim ? tp + moe_term_at(el) : reinterpret_cast<const uint16_t *>(kMgZeros);
                        const u32x4 o = *(const GLOBAL_AS u32x4 *)src;
                        a[t][s][m].u[0] = o.x; a[t][s][m].u[1] = o.y; a[t][s][m].u[2] = o.z; a[t][s][m].u[3] = o.w;
                    }
            }
        }

        // 6. The row partials of a finished batch meet: a thread per (tile, row, pair of tokens), every wavefront its share.
        //    A wavefront does so somewhere inside the next batch — the two of a SIMD at different tiles — so that the other one
        //    has the matrix pipe meanwhile; all of them folding right behind the barrier cost 0.8 us a batch.
        uint32_t f_nbt = 0, f_tile = 0;
        const float *f_part = nullptr, *f_bias = nullptr;
        auto fold = [&]() {
            for (uint32_t i = tid; i < f_nbt * 16 * TP; i += blockDim.x) {
                const uint32_t p = i % TP, r = (i / TP) & 15u, tile = i / (16 * TP);
                const float *pr = f_part + (tile * nw * 16 + r) * TG + 2 * p;
                float2_t pw[8];
#pragma unroll
                for (uint32_t w = 0; w < 8; w++) pw[w] = *reinterpret_cast<const float2_t *>(pr + min(w, nw - 1) * 16 * TG);
                float2_t s = pw[0];
#pragma unroll
                for (uint32_t w = 1; w < 8; w++) {
                    s.x = w < nw ? s.x + pw[w].x : s.x;
                    s.y = w < nw ? s.y + pw[w].y : s.y;
                }
                const uint32_t row = (f_tile + tile) * 16 + r;
                if (A.bias) { const float bv = f_bias[tile * 16 + r]; s.x += bv; s.y += bv; }
                if (DOWN) {
                    if (2 * p < ntok) ((g_f32wp)A.out)[(size_t)gl[2 * p] * rows + row] = s.x;
                    if (2 * p + 1 < ntok) ((g_f32wp)A.out)[(size_t)gl[2 * p + 1] * rows + row] = s.y;
                } else {
                    // the thread of a gate row (even) gates its first token, the one of the up row, TP lanes on, the second
                    constexpr int CTRL = TP == 8 ? 0x128 : 0x4E;  // row_ror:8 / quad_perm [2,3,0,1]
                    const bool odd = r & 1u;
                    const float in = __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, odd ? s.x : s.y), CTRL, 0xF, 0xF, false));
                    const uint32_t token = 2 * p + (odd ? 1u : 0u);
                    float act = clamped_glu(odd ? in : s.x, odd ? s.y : in, A.glu_limit, A.glu_alpha);
                    // (the terms are those of the f32 value, as in the one-token kernels: its last product would else be fused
                    // into their first subtraction)
                    asm volatile("" : "+v"(act));
                    uint32_t t3[3];
                    mx4_terms(act, 0.0f, t3);
                    if (token < ntok) {
                        const size_t opad = moe_terms_pad(rows / 2), plane = slots * opad;
                        GLOBAL_AS uint16_t *tp = (GLOBAL_AS uint16_t *)A.terms_out + gl[token] * opad + moe_term_at(row >> 1);
                        tp[0] = (uint16_t)t3[0]; tp[plane] = (uint16_t)t3[1]; tp[2 * plane] = (uint16_t)t3[2];
                    }
                }
            }
            f_nbt = 0;
        };
        // 7. the tiles
        for (uint32_t tb = 0; tb < nt; tb += R) {
            float *pb = part + parity * part_floats, *bb = lbias + parity * (R * 16);
            const uint32_t nbt = min((uint32_t)R, nt - tb);
            // The biases of the batch's rows come through LDS as well (the wavefronts take turns): a load into a register
            // would be waited for behind every tile in flight.  This copy is older than the tiles that may still fly when
            // the batch's last tile is waited for, so it has landed by then; anywhere else it only makes a wait stricter.
            if (A.bias && wv == turn) {
                const float *bp = A.bias + (size_t)e * rows + (t0 + tb) * 16;
#pragma unroll
                for (int q = 0; q < (R * 16 + 63) / 64; q++)
                    if (q * 64 + lane < (uint32_t)R * 16)
                        __builtin_amdgcn_global_load_lds((g_vp)(bp + min(q * 64 + lane, nbt * 16 - 1)), (lds_vp)(bb + q * 64), 4, 0, 0);
            }
            for (uint32_t tl = 0; tl < nbt; tl++) {
                if (left) issue();
                const uint32_t younger = nt - left - (tb + tl) - 1;  // tiles requested after this one
                if (younger >= 2) LARQL_WAIT_VMCNT(2 * L);
                else if (younger == 1) LARQL_WAIT_VMCNT(L);
                else LARQL_WAIT_VMCNT(0);
                asm volatile("" ::: "memory");
                const uint8_t *slot = ring + use_i * slot_bytes;
                use_i = use_i + 1 == NS ? 0u : use_i + 1;
                f32x4 D[NT];
#pragma unroll
                for (int t = 0; t < NT; t++) D[t] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
                for (int s = 0; s < CW; s++) {
                    const u32x4 q = *reinterpret_cast<const u32x4 *>(slot + s * kMgStepBytes + lane * 16);
                    const uint32_t sc = slot[CW * kMgStepBytes + sc_at[s]];
                    float scale = __builtin_bit_cast(float, sc << 23);                    // 2^(sc-127); 0 -> 0.0
                    scale = sc == 255u ? __builtin_bit_cast(float, 0x7FC00000u) : scale;  // 255 -> NaN
                    const uint32_t w4[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
                    for (int m = 0; m < 4; m++) {
                        BfOp b;
                        b.u[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w4[m], scale, 0));
                        b.u[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w4[m], scale, 1));
                        b.u[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w4[m], scale, 2));
                        b.u[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp4(w4[m], scale, 3));
#pragma unroll
                        for (int t = 0; t < NT; t++) D[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t][s][m].v, b.v, D[t], 0, 0, 0);
                    }
                }
                // lane (weight row jr, kg): TG = 16: D[t] = term t of tokens 4kg .. 4kg+3; TG = 4: D[0] = the three terms of token kg
                float *pr = pb + ((tl * nw + wv) * 16 + jr) * TG;
                if (TG == 16) *reinterpret_cast<f32x4 *>(pr + 4 * kg) = (D[0] + D[NT > 1 ? 1 : 0]) + D[NT > 2 ? 2 : 0];
                else pr[kg] = (D[0][0] + D[0][1]) + D[0][2];
                // (the sums depend on every read of the slot: nothing of it is outstanding when the next copies are asked for)
                asm volatile("" ::: "memory");
                if (f_nbt && tl == fold_at) fold();
            }
            if (f_nbt) fold();  // (a batch too short to reach the place for it)
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            __builtin_amdgcn_s_barrier();
            asm volatile("" ::: "memory");
            f_nbt = nbt; f_tile = t0 + tb; f_part = pb; f_bias = bb;
            parity ^= 1u;
            turn = turn + 1 == nw ? 0u : turn + 1;
        }
        if (f_nbt) fold();
        lpar ^= 1u;
    }
    LARQL_WAIT_VMCNT(0);
}

// Token `blockIdx.x`'s selection (with `logits`: Router::select by wavefront 0) and, by the other four wavefronts beside it, its
// activation as three bf16 terms, terms[term][token][moe_terms_pad(hidden)].  (The selection behind its wavefront's share of the
// terms: 6.1 us for 128 tokens of 2880, so 4.8.)
__global__ void __launch_bounds__(320) moe_route_terms_kernel(const float *__restrict__ logits, const float *__restrict__ bias, uint32_t n_experts,
                                                             uint32_t k, int policy, uint32_t tokens, uint32_t *__restrict__ experts,
                                                             float *__restrict__ weights, const float *__restrict__ x, uint16_t *__restrict__ terms, uint32_t hidden) {
    const uint32_t t = blockIdx.x, lane = threadIdx.x & 63u;
    if (threadIdx.x >= 64) {
        const size_t pad = moe_terms_pad(hidden), plane = tokens * pad;
        for (uint32_t i = (threadIdx.x - 64) * 4; i < hidden; i += 1024) {  // (hidden % 32 == 0)
            const f32x4 v = *reinterpret_cast<const f32x4 *>(x + (size_t)t * hidden + i);
            uint32_t a[3], b[3];
            mx4_terms(v.x, v.y, a);
            mx4_terms(v.z, v.w, b);
#pragma unroll
            for (int q = 0; q < 3; q++) *reinterpret_cast<uint2 *>(terms + q * plane + t * pad + moe_term_at(i)) = make_uint2(a[q], b[q]);
        }
    } else if (logits) {
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
}

hipError_t moe_route_terms_launch(hipStream_t s, const float *logits, const float *bias, uint32_t tokens, uint32_t n_experts, uint32_t k, int policy,
                                  uint32_t *experts, float *weights, const float *x, uint32_t hidden, uint16_t *terms) {
    hipLaunchKernelGGL(moe_route_terms_kernel, dim3(tokens), dim3(320), 0, s, logits, bias, n_experts, k, policy, tokens, experts, weights, x, terms, hidden);
    return hipGetLastError();
}

static uint32_t mg_steps_per_wave(uint32_t kdim) {  // 128-element steps per wavefront: at most eight wavefronts cover a row
    const uint32_t steps = (kdim + 127) / 128;
    for (uint32_t cw = 1; cw <= 5; cw++)
        if ((steps + cw - 1) / cw <= 8) return cw;
    return 0;
}

bool moe_group_serves(uint32_t rows, uint32_t kdim) {
    return kdim >= 128 && kdim % 32 == 0 && rows % 16 == 0 && rows < (1u << 22) && mg_steps_per_wave(kdim) != 0;
}

template <bool DOWN, int CW, int TG>
static hipError_t mg_launch(hipStream_t s, const MoeGroupArgs &A, uint32_t cu_count) {
    static std::atomic<bool> allowed{false};  // dynamic LDS above 64 KB has to be allowed once per kernel
    if (!allowed) {
        hipError_t e = hipFuncSetAttribute((const void *)moe_group_kernel<DOWN, CW, TG>, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
        allowed = true;
    }
    const uint32_t nw = ((A.kdim + 127) / 128 + CW - 1) / CW;
    const size_t lds = (size_t)nw * kMgStages * mg_slot_bytes(CW) + 2 * (size_t)mg_tiles(CW, TG) * 16 * (nw * TG + 1) * sizeof(float) +
                       (2 * (size_t)A.n_experts + 1) * sizeof(uint32_t) + (32 + (size_t)A.slots) * sizeof(uint16_t);
    if (lds > 160 * 1024) return hipErrorInvalidValue;
    const uint32_t per_cu = std::max<uint32_t>(1, std::min<uint32_t>((160 * 1024) / (uint32_t)lds, 8 / nw));
    hipLaunchKernelGGL((moe_group_kernel<DOWN, CW, TG>), dim3(cu_count * per_cu), dim3(nw * 64), lds, s, A.experts, A.slots, A.n_experts, A.kdim, A.rows,
                       cu_count * per_cu, A);
    return hipGetLastError();
}

// Groups of sixteen tokens once an expert has more than four on average, five with four steps per wavefront.  Same block with
// groups of four / of sixteen, us (routing included; biases), by slots per expert:
//   1024 x 1024, 32 experts, top-4   4: 32.6 / 32.9    5: 34.7 / 33.5    6: 37.1 / 34.0    8: 43.8 / 36.0
//   2048 x 2048, 32 experts, top-4   4: 63.3 / 61.9    5: 74.4 / 62.5    6: 80.1 / 63.9    8: 96.1 / 68.2
//   2880 x 2880, 32 experts, top-4   2: 93.4 / 107.0   4: 120.3 / 122.8  5: 131.2 / 124.2  6: 144.3 / 125.6   8: 179.8 / 126.1
//   3328 x 3328, 16 experts, top-2   5: 86.1 / 93.1    6: 100.7 / 94.7   7: 105.7 / 97.6
//   4096 x 4096, 16 experts, top-2   2: 85.6 / 107.9   4: 107.7 / 118.4  5: 119.4 / 122.6  5.5: 128.4 / 121.8  8: 171.4 / 133.5
// The job tables before, where four tokens shared a job (2880 / 4096 as above): 2 tokens 47.1 -> 33.4 / 47.2 -> 32.2, 8 tokens
// 95.0 -> 74.5 / 80.0 -> 58.3, 16 tokens 118.7 -> 93.9 / 114.7 -> 84.8, 64 tokens - / 234.8 -> 133.2, 128 tokens 400 -> 164 / 375.9 -> 169.1;
// 5120 x 5120, 16 experts, top-4, groups of four only: 2 tokens 85.6 -> 74.2, 16 213.9 -> 196.5, 64 582.9 -> 591.1, 128 1054 -> 996.
template <bool DOWN>
static hipError_t mg_launch_stage(hipStream_t s, const MoeGroupArgs &A, uint32_t cu_count) {
    const uint32_t cw = mg_steps_per_wave(A.kdim);
    const bool wide = A.slots > (cw == 4 ? 5u : 4u) * A.n_experts;
    switch (cw) {
        case 1: return wide ? mg_launch<DOWN, 1, 16>(s, A, cu_count) : mg_launch<DOWN, 1, 4>(s, A, cu_count);
        case 2: return wide ? mg_launch<DOWN, 2, 16>(s, A, cu_count) : mg_launch<DOWN, 2, 4>(s, A, cu_count);
        case 3: return wide ? mg_launch<DOWN, 3, 16>(s, A, cu_count) : mg_launch<DOWN, 3, 4>(s, A, cu_count);
        case 4: return wide ? mg_launch<DOWN, 4, 16>(s, A, cu_count) : mg_launch<DOWN, 4, 4>(s, A, cu_count);
        case 5: return mg_launch<DOWN, 5, 4>(s, A, cu_count);  // (sixteen tokens' operands of five steps: 240 registers)
        default: return hipErrorInvalidValue;
    }
}

hipError_t moe_group_launch(hipStream_t s, const MoeGroupArgs &A, bool down, uint32_t cu_count) {
    if (!moe_group_serves(A.rows, A.kdim) || A.slots == 0 || A.slots > kMoeGroupMaxSlots || A.n_experts == 0 || A.n_experts > kMoeGroupMaxExperts)
        return hipErrorInvalidValue;
    return down ? mg_launch_stage<true>(s, A, cu_count) : mg_launch_stage<false>(s, A, cu_count);
}

}  // namespace larql
