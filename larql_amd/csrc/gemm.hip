// gemm.hip — batched-prefill Q4_K GEMM on the gfx950 matrix cores.
//
//   out[s, r] = sum_k W[r, k] * X[s, k]      W: [rows, hidden] Q4_K,  X: [seq, hidden] bf16 or f32
//
// the contraction q4k_matmul_into computes (larql-compute/src/cpu/ops/q4_common/
// matmul.rs:20-139; `out` is [seq, rows] row-major), on f16 MFMA over operands made
// from the stored nibbles (see the formulation below).
#include <hip/hip_runtime.h>

#include <atomic>
#include <type_traits>
#include <stdint.h>
#include <stdlib.h>

#include "kernels.h"
#include "wave.h"

namespace larql {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// ---------------------------------------------------------------------------
// The formulation: a sub-block's scale term and its offset are separate operands.
//
//   out[s, r] = sum over super-blocks of  d[r] * (sum_k (sc6*q)[r,k] * x[s,k])  -  dmin[r] * (sum_sub mn6[r,sub] * Sx[s,sub])
//
// The activations are prepared once per call (q4k_gemm_prep_kernel): per token a power-of-two scale brings
// max|x| to [2^13, 2^14) and x/scale is stored as f16 (exact for bf16 inputs; f32 inputs add a second f16 term
// and a second pass).  The weight operand is made from the raw nibbles (mask into the mantissa of an f16, packed f16
// instructions) and never stored in memory.  Two kernels:
//   * q4k_gemm_exact_kernel (host tier): the operand is sc6*q <= 945, exact in f16; per super-block a wavefront keeps
//     the integer sums apart (D), gets sum_sub mn6*Sx from one more MFMA per block (A slots 2*sub+h = 32 mn6,
//     B slots = Sx_h/32; Sx, the sum of the represented activations over each 32-element sub-block, comes with the
//     preparation as an f16 pair, divided by 32 to stay inside f16), and folds both into the f32 result with the row's
//     d and dmin.
//   * q4k_gemm_pair_kernel (device tier): the operand is f16(d sc6 (q - 7.5)), sc6 (q - 7.5) exact in f16 and the product with d
//     rounded once; the offsets 7.5 d sc6 - dmin mn6 are an f16 pair of their own (22 bits) against the Sx pair, one more MFMA per block
//     and super-block.  All times the row's 2^E; 2^-E and the token's scale are applied once at the end, no folds.
//     So the only error above f32 is one f16 rounding per nibble value, at the size of d sc6 |q - 7.5|: a sub-block's mean and the
//     activations' do not enter.  Relative to the f64 product, 203 x 2560, 33 tokens (in brackets: the whole weight in one f16 |
//     f16(s (q - 8)) with s = f16(d sc6) and one f16 per offset):
//       weights N(0,1), activations N(0,1) 2.2e-4 (2.2e-4 | 3.1e-4), with mean 5 2.1e-4 (4.7e-4 | 5.8e-4);  |N(0,1)|, N(0,1) 1.6e-4
//       (3.3e-4 | 2.7e-4);  1 + N/20 against activations whose neighbours cancel 1.3e-3 (3.3e-3 | 1.5e-3);  offsets 60 times the scales,
//       against the same 2.1e-4 (2.5e-3 | 2.8e-4)
// ---------------------------------------------------------------------------
__device__ __forceinline__ float half_to_float(uint32_t lo16) { return (float)__builtin_bit_cast(_Float16, (uint16_t)lo16); }

typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x4 __attribute__((ext_vector_type(4)));

// one block per token: scale, f16 terms, sub-block sums.  `x_is_bf16`: 16-bit inputs (exact in one term).
// A thread takes 8 consecutive elements at a time (one or two 16-byte loads); four neighbouring threads hold a
// 32-element sub-block.
// (The arguments that a block's first loads wait for are the first fourteen dwords, which are in registers when it starts.)
__global__ void __launch_bounds__(1024) q4k_gemm_prep_kernel(const void *__restrict__ x, uint32_t hidden, uint32_t seq, int x_is_bf16, int swap12,
                                                            uint16_t *__restrict__ xh, uint16_t *__restrict__ sx, float *__restrict__ tok_scale,
                                                            uint16_t *__restrict__ xl, int *__restrict__ any_lo,
                                                            const uint8_t *__restrict__ w, uint32_t rows, int *__restrict__ rexp) {
    __shared__ float red[16];
    const uint32_t t = threadIdx.x, nvec = hidden >> 3;  // hidden % 256 == 0
    if (blockIdx.x >= seq) {
        // the blocks behind the tokens: 16 lanes per weight row, E with max(|d|, |dmin|/16) * 2^E in [0.5, 1) over the row,
        // so that 2^15 d 2^E < 2^15 and |32 (7.5 d sc6 - dmin mn6) 2^E| <= 32 (7.5 + 16) 63 = 47376 stay well inside f16
        const uint32_t row = (blockIdx.x - seq) * (blockDim.x >> 4) + (t >> 4), nsb = hidden >> 8;
        float m = 0.f;
        if (row < rows) {
            const uint8_t *p = w + (size_t)row * nsb * 144;
            for (uint32_t sb0 = t & 15u; sb0 < nsb; sb0 += 64) {  // four independent loads in flight per lane
                uint32_t h[4];
#pragma unroll
                for (int u = 0; u < 4; u++) h[u] = sb0 + 16 * u < nsb ? *reinterpret_cast<const uint32_t *>(p + (size_t)(sb0 + 16 * u) * 144) : 0u;
#pragma unroll
                for (int u = 0; u < 4; u++)
                    m = fmaxf(m, fmaxf(fabsf(half_to_float(h[u] & 0xFFFFu)), 0.0625f * fabsf(half_to_float(h[u] >> 16))));
            }
        }
        m = row16_max(m);
        if (row < rows && (t & 15u) == 0) {
            int e = 0;
            if (m > 0.f && m < __builtin_inff()) (void)frexpf(m, &e);
            rexp[row] = -e;
        }
        return;
    }
    const uint32_t tok = blockIdx.x;
    const u32x4 *xb = reinterpret_cast<const u32x4 *>((const uint16_t *)x + (size_t)tok * hidden);
    const f32x4 *xf = reinterpret_cast<const f32x4 *>((const float *)x + (size_t)tok * hidden);
    auto load8 = [&](uint32_t v, float (&o)[8], const u32x4 *kept = nullptr) {
        if (x_is_bf16) {
            const u32x4 r = kept ? *kept : xb[v];
            const uint32_t w[4] = {r.x, r.y, r.z, r.w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
                o[2 * i] = __builtin_bit_cast(float, w[i] << 16);
                o[2 * i + 1] = __builtin_bit_cast(float, w[i] & 0xFFFF0000u);
            }
        } else {
            const f32x4 a = xf[2 * v], b = xf[2 * v + 1];
            o[0] = a.x; o[1] = a.y; o[2] = a.z; o[3] = a.w; o[4] = b.x; o[5] = b.y; o[6] = b.z; o[7] = b.w;
        }
    };
    // KEEP vectors of a bf16 token stay in the thread's registers from the maximum to the conversion, requested together (the
    // launch is a chain of round trips; 77 tokens of 15360: 5.9 us)
    constexpr uint32_t KEEP = 2;
    u32x4 kept[KEEP] = {};
    float mx = 0.f;
    if (x_is_bf16) {
#pragma unroll
        for (uint32_t u = 0; u < KEEP; u++) kept[u] = xb[min(t + u * blockDim.x, nvec - 1)];
    }
    auto max8 = [&](uint32_t v, const u32x4 *k) {
        float o[8];
        load8(v, o, k);
#pragma unroll
        for (int i = 0; i < 8; i++) mx = fmaxf(mx, fabsf(o[i]));
    };
    if (x_is_bf16) {  // (a clamped vector is the token's own: it does not change the maximum)
#pragma unroll
        for (uint32_t u = 0; u < KEEP; u++) max8(0, &kept[u]);
    }
    for (uint32_t v = t + (x_is_bf16 ? KEEP * blockDim.x : 0u); v < nvec; v += blockDim.x) max8(v, nullptr);
    mx = row16_max(mx);
    mx = dpp_max<0x142, 0xA>(mx);  // row_bcast:15 into rows 1 and 3
    mx = dpp_max<0x143, 0xC>(mx);  // row_bcast:31 into rows 2 and 3: lane 63 holds the wavefront's
    if ((t & 63u) == 63) red[t >> 6] = mx;
    __syncthreads();
    mx = 0.f;
    for (uint32_t wv = 0; wv < (blockDim.x >> 6); wv++) mx = fmaxf(mx, red[wv]);
    int ex = 0;
    if (mx > 0.f && mx < __builtin_inff()) (void)frexpf(mx, &ex);
    ex = max(-100, min(110, ex));
    const float to_h = ldexpf(1.f, 14 - ex);
    if (t == 0) tok_scale[tok] = ldexpf(1.f, ex - 14);
    int lo_seen = 0;
    // the f16 terms are kept as [token][hidden] (a step's 128 bytes of a token are one cache line; a [step][token] order
    // was measured: no faster for the GEMM, slower here) and the sums as [super-block][token][8], so that what a GEMM
    // workgroup copies of them for a super-block is one contiguous run
    u32x4 *oh = reinterpret_cast<u32x4 *>(xh);
    u32x4 *ol = xl ? reinterpret_cast<u32x4 *>(xl) : nullptr;
    auto convert = [&](uint32_t v, const u32x4 *k) {  // nvec % 32 == 0: the four threads of a sub-block run together
        float o[8];
        load8(v, o, k);
        uint32_t hw[4] = {0u, 0u, 0u, 0u}, lw[4] = {0u, 0u, 0u, 0u};
        float sm = 0.f;
#pragma unroll
        for (int i = 0; i < 8; i++) {
            const float sv = o[i] * to_h;
            const _Float16 h = (_Float16)sv;
            const _Float16 l = (_Float16)(sv - (float)h);
            const uint32_t hb = __builtin_bit_cast(uint16_t, h), lb = __builtin_bit_cast(uint16_t, l);
            // `swap12`: elements 1 and 2 of every four change places (the pipelined GEMM's weight operand comes out of
            // its nibble masks as the pairs (k0, k2), (k1, k3); the MFMA only needs both operands to agree)
            const int pos = swap12 ? ((i & 4) | ((i & 1) << 1) | ((i >> 1) & 1)) : i;
            if (pos & 1) { hw[pos >> 1] |= hb << 16; lw[pos >> 1] |= lb << 16; } else { hw[pos >> 1] |= hb; lw[pos >> 1] |= lb; }
            lo_seen |= (ol && (float)l != 0.f) ? 1 : 0;
            sm += (float)h + (ol ? (float)l : 0.f);  // the activation as the MFMAs will see it
        }
        const size_t at = (size_t)tok * nvec + v;
        oh[at] = (u32x4){hw[0], hw[1], hw[2], hw[3]};
        if (ol) ol[at] = (u32x4){lw[0], lw[1], lw[2], lw[3]};
        sm += dpp_move<0xB1>(sm);  // quad_perm [1,0,3,2]
        sm += dpp_move<0x4E>(sm);  // quad_perm [2,3,0,1]
        sm *= 0.03125f;  // stored as Sx/32 so that 32 x 2^14 stays inside f16; the min operand carries the 32
        if ((t & 3u) == 0) {
            const _Float16 sh = (_Float16)sm;
            const _Float16 sl = (_Float16)(sm - (float)sh);
            const uint32_t pair = (uint32_t)__builtin_bit_cast(uint16_t, sh) | ((uint32_t)__builtin_bit_cast(uint16_t, sl) << 16);
            reinterpret_cast<uint32_t *>(sx)[((size_t)(v >> 5) * seq + tok) * 8 + ((v >> 2) & 7u)] = pair;
        }
    };
    if (x_is_bf16) {
#pragma unroll
        for (uint32_t u = 0; u < KEEP; u++)
            if (t + u * blockDim.x < nvec) convert(t + u * blockDim.x, &kept[u]);
    }
    for (uint32_t v = t + (x_is_bf16 ? KEEP * blockDim.x : 0u); v < nvec; v += blockDim.x) convert(v, nullptr);
    if (lo_seen && any_lo) *any_lo = 1;
}

// adds the partial slabs of a K-split in slab order and applies the token scale; VEC elements per thread.  Four may lie in two tokens and at any
// multiple of four bytes (a 16-byte access needs no more).
// Bound: latency, then memory (the slabs come out of the last-level cache).  Eight slabs are requested together, so that a
// launch costs splits / 8 round trips instead of `splits`; a request past the last slab reads the last one and is not added.
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
template <int VEC>
__global__ void __launch_bounds__(256) q4k_gemm_reduce_kernel(const float *__restrict__ partial, uint32_t splits, const float *__restrict__ tok_scale,
                                                              float *__restrict__ out, uint32_t rows, uint32_t seq, int accumulate) {
    typedef std::conditional_t<VEC == 4, f32x4_a4, float> vec;
    const size_t n = (size_t)rows * seq, i = ((size_t)blockIdx.x * blockDim.x + threadIdx.x) * VEC;
    if (i >= n) return;
    if (i + VEC > n) {  // the last one to three elements
        for (size_t k = i; k < n; k++) {
            float s = 0.f;
            for (uint32_t z = 0; z < splits; z++) s += partial[z * n + k];
            s *= tok_scale[k / rows];
            out[k] = accumulate ? out[k] + s : s;
        }
        return;
    }
    const size_t tok = i / rows;
    const uint32_t left = (uint32_t)min((size_t)VEC, (tok + 1) * rows - i);  // elements of this token
    float ts[VEC], s[VEC];
#pragma unroll
    for (int e = 0; e < VEC; e++) { ts[e] = tok_scale[(uint32_t)e < left ? tok : (i + e) / rows]; s[e] = 0.f; }
    for (uint32_t z0 = 0; z0 < splits; z0 += 8) {
        vec v[8];
#pragma unroll
        for (uint32_t u = 0; u < 8; u++) v[u] = *reinterpret_cast<const vec *>(partial + (size_t)min(z0 + u, splits - 1) * n + i);
#pragma unroll
        for (uint32_t u = 0; u < 8; u++)
#pragma unroll
            for (int e = 0; e < VEC; e++) s[e] = z0 + u < splits ? s[e] + reinterpret_cast<const float *>(&v[u])[e] : s[e];
    }
    vec r, *o = reinterpret_cast<vec *>(out + i);
#pragma unroll
    for (int e = 0; e < VEC; e++) reinterpret_cast<float *>(&r)[e] = s[e] * ts[e];
    if (accumulate) r += *o;
    *o = r;
}

// ---------------------------------------------------------------------------
// The host tier's kernel: the weight operand is the integer sc6*q, a super-block's sums are kept apart (D) and folded
// into the result with the row's f32 d / dmin, so the only roundings are the f32 accumulations (the trait's callers
// compare a row of the matmul with the CPU matvec at 1e-4 absolute).
// with_mins = 0: the activation term carries no offset part (second pass over the lo terms).
//
// One workgroup of 4 wavefronts per CU owns a 256-row x 128-token tile; a wavefront owns 64 of the rows against
// all 128 tokens (2 x 4 blocks of v_mfma_f32_32x32x16_f16: an operand read from LDS feeds two MFMAs of 32 cycles).
// Everything a step (64 k) needs from global memory was copied global -> LDS (global_load_lds, 16 bytes per lane,
// no registers involved) at least two steps before:
//   * the f16 activations of a step, into a ring of four stages.  Rows are 128 bytes (64 f16) without
//     padding; the 16-byte chunk c of row r is kept at position c ^ ((r >> 1) & 7), chosen on the global side of
//     the copy, so that sixteen neighbouring lanes of an operand read (sixteen rows, one chunk) cover the 64 banks;
//   * the weights a super-block at a time (144 bytes per row, header included: a row's two or three cache lines
//     are asked for once, not once per step), into two stages (a wavefront copies its own rows);
//   * per super-block the Sx of the tile's tokens.
// A wavefront turns the headers of its rows into two small LDS tables once per super-block (one thread per row):
// per sub-block the packed-FMA operands (scale, -1024 * scale) and the offsets' MFMA operand.
// The f16 weight operand never exists in memory: lane (row32, kgrp) of an MFMA holds 8 k of row row32.  The k
// of a step are dealt so that a lane needs 16 consecutive raw bytes of its row: MFMA j of half h takes the
// nibbles h of bytes 16*kgrp + 8j .. +7, i.e. k 32h + 16kgrp + 8j .. +7 (the activations' chunk 4h + 2kgrp + j).
// The lane reads those 16 bytes of its two rows once per step and converts them, in the MFMAs' shadow, into the
// operand of the next half.  Only the activations cross wavefronts: one barrier per step, in the middle of it, so
// that the operand reads of the next step's first MFMAs are already issued when the step ends.  No global load
// returns into a register inside the loop, so the compiler places no vmcnt waits of its own (it would wait for
// *all* outstanding loads as soon as register loads and LDS copies are in flight together); outstanding copies
// are counted by hand: at the barrier only the requests made at the barrier before may still fly.  For the same
// reason (an LDS copy in flight makes the compiler wait for lgkmcnt(0) at every LDS read) the operand reads of
// the loop are written as instructions with counted waits, G_LA reads ahead of the MFMA group that consumes them.
// ---------------------------------------------------------------------------
constexpr int GM = 256, GN = 128, GTHREADS = 256;
constexpr int G_LA = 4;                                                         // operand reads in flight ahead of the MFMAs
constexpr int G_NB = 4, G_NR = 2;                                               // ring depths: activations (steps), weights (super-blocks)
constexpr int G_B_STAGE = GN * 128, G_R_STAGE = GM * 144;                       // bytes
constexpr int G_B_OFF = 0, G_R_OFF = G_B_OFF + G_NB * G_B_STAGE,
              G_BM_OFF = G_R_OFF + G_NR * G_R_STAGE, G_SC_OFF = G_BM_OFF + GN * 32, G_AM_OFF = G_SC_OFF + GM * 32,
              G_D_OFF = G_AM_OFF + GM * 32, G_DMIN_OFF = G_D_OFF + 2 * GM * 4, G_LOOP_BYTES = G_DMIN_OFF + 2 * GM * 4;
constexpr int G_EP_LD = 68, G_EP_BYTES = 4 * GN * G_EP_LD * 4;                  // the results leave through LDS (see the epilogue)
constexpr int G_LDS_BYTES = G_LOOP_BYTES > G_EP_BYTES ? G_LOOP_BYTES : G_EP_BYTES;
static_assert(G_LDS_BYTES <= 160 * 1024, "one workgroup per CU");
static_assert(G_NB == 4 && G_NR == 2, "ring slots are named by the step's position in its super-block and the super-block's parity");
typedef __attribute__((address_space(3))) void *p_lds_vp;
typedef const __attribute__((address_space(1))) void *p_g_vp;
typedef float f32x16 __attribute__((ext_vector_type(16)));
#define GEMM_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0xF << 8))

__global__ void __launch_bounds__(GTHREADS, 1) q4k_gemm_exact_kernel(const uint8_t *w, const uint16_t *xh, const uint16_t *sx,
                                                               const float *__restrict__ tok_scale, float *__restrict__ out,
                                                               uint32_t rows, uint32_t hidden, uint32_t seq, int with_mins,
                                                               int accumulate, uint32_t sb_per_split, float *__restrict__ partial) {
    extern __shared__ __attribute__((aligned(16))) uint8_t glds[];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t row0 = blockIdx.x * GM, tok0 = blockIdx.y * GN;
    const uint32_t nsb = hidden >> 8, row_bytes = nsb * 144;
    const uint32_t sb_begin = blockIdx.z * sb_per_split, sb_end = min(nsb, sb_begin + sb_per_split);
    if (sb_begin >= sb_end) return;
    const uint32_t nsteps = (sb_end - sb_begin) * 4;

    // copy roles.  Weights: a super-block of the wavefront's 64 rows (144 bytes each, header included) is nine copies;
    // piece p, lane l brings 16-byte chunk (64p + l) % 9 of row (64p + l) / 9, so that the rows lie in LDS one after the
    // other and a row's two or three cache lines are asked for by neighbouring lanes of one instruction.
    const uint8_t *wt = w + (size_t)row0 * row_bytes;                                          // uniform
    uint32_t r_off[9];
#pragma unroll
    for (int p9 = 0; p9 < 9; p9++) {
        const uint32_t idx = p9 * 64 + lane;
        r_off[p9] = (min(row0 + wave * 64 + idx / 9, rows - 1) - row0) * row_bytes + (idx % 9) * 16;
    }
    // activations ([token][hidden] f16): wavefront -> tokens 32w .. 32w+31 (four copies of 8 tokens x 128 bytes), lane -> (token, chunk)
    const uint8_t *xt = (const uint8_t *)xh;                                                   // uniform
    uint32_t b_off[4];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const uint32_t r = (wave * 4 + q) * 8 + (lane >> 3);
        b_off[q] = min(tok0 + r, seq - 1) * hidden * 2 + (((lane & 7u) ^ ((r >> 1) & 7u)) * 16);
    }
    // Sx ([super-block][token][8 pairs]): wavefront -> tokens 32w .. 32w+31 (two 16-byte halves each)
    const uint8_t *st = (const uint8_t *)sx;                                                   // uniform
    const uint32_t m_off = min(tok0 + wave * 32 + (lane >> 1), seq - 1) * 32 + (lane & 1u) * 16;

    // compute role: a wavefront owns the 64 rows it converts, against all 128 tokens: the weight operand, the raw
    // bytes, the headers and the per-row tables never cross wavefronts, only the activations (and Sx) do
    const uint32_t wm = wave * 64;
    const uint32_t row32 = lane & 31u, kgrp = lane >> 5;

    // (requests past the end are clamped: same number of copies in flight, results unused)
    auto issue_raw = [&](uint32_t sb, int p9) {  // one of the nine pieces of a super-block
        const uint8_t *src = wt + (size_t)min(sb, sb_end - 1) * 144;
        uint8_t *dst = glds + G_R_OFF + ((sb - sb_begin) & 1u) * G_R_STAGE + wave * 9216;
        __builtin_amdgcn_global_load_lds((p_g_vp)(src + r_off[p9]), (p_lds_vp)(dst + p9 * 1024), 16, 0, 0);
    };
    auto issue_b = [&](uint32_t s, uint32_t slot, int q) {  // one of the four pieces of a step
        const uint32_t sc = min(s, nsteps - 1);
        const uint8_t *src = xt + ((size_t)sb_begin * 4 + sc) * 128;
        uint8_t *dst = glds + G_B_OFF + slot * G_B_STAGE + wave * 4096;
        __builtin_amdgcn_global_load_lds((p_g_vp)(src + b_off[q]), (p_lds_vp)(dst + q * 1024), 16, 0, 0);
    };
    auto issue_sx = [&](uint32_t sb) {  // Sx of a super-block
        const uint32_t sbc = min(sb, sb_end - 1);
        __builtin_amdgcn_global_load_lds((p_g_vp)((st + (size_t)sbc * seq * 32) + m_off), (p_lds_vp)(glds + G_BM_OFF + wave * 1024), 16, 0, 0);
    };
    // a super-block's header -> this row's tables.  Scales: per sub-block the pair (sc6, -1024 sc6) for the packed FMA
    // that turns a masked nibble 1024 + q into sc6*q.  Odd sub-blocks are the high nibbles, whose masked value is
    // 1024 + 16q, so they carry sc6/16.  Offsets: 32 mn6 twice, for the two f16 halves of Sx/32.
    auto stage_sb = [&](uint32_t par) {
        const u32x4 hdr = *reinterpret_cast<const u32x4 *>(glds + G_R_OFF + par * G_R_STAGE + wave * 9216 + lane * 144);
        const float d = half_to_float(hdr.x & 0xFFFFu), dmin = half_to_float(hdr.x >> 16);
        uint32_t mnw[8];
#pragma unroll
        for (int sub = 0; sub < 8; sub++) {
            const uint32_t sh = 8u * (sub & 3u);
            const uint32_t pa = (hdr.y >> sh) & 0xFFu, pb = (hdr.z >> sh) & 0xFFu, pc = (hdr.w >> sh) & 0xFFu;
            const uint32_t sc6 = sub < 4 ? (pa & 63u) : ((pc & 0x0Fu) | ((pa >> 6) << 4));
            const uint32_t mn6 = sub < 4 ? (pb & 63u) : ((pc >> 4) | ((pb >> 6) << 4));
            const float sf = (float)sc6 * ((sub & 1) ? 0.0625f : 1.f);
            const _Float16 s16 = (_Float16)sf, o16 = (_Float16)(-1024.f * sf);
            *reinterpret_cast<uint32_t *>(glds + G_SC_OFF + wave * 2048 + sub * 256 + lane * 4) =
                (uint32_t)__builtin_bit_cast(uint16_t, s16) | ((uint32_t)__builtin_bit_cast(uint16_t, o16) << 16);
            const uint32_t hb = __builtin_bit_cast(uint16_t, (_Float16)(32.f * (float)mn6));
            mnw[sub] = hb | (hb << 16);
        }
        *reinterpret_cast<u32x4 *>(glds + G_AM_OFF + (wm + lane) * 32) = (u32x4){mnw[0], mnw[1], mnw[2], mnw[3]};
        *reinterpret_cast<u32x4 *>(glds + G_AM_OFF + (wm + lane) * 32 + 16) = (u32x4){mnw[4], mnw[5], mnw[6], mnw[7]};
        reinterpret_cast<float *>(glds + G_D_OFF)[par * GM + wm + lane] = d;
        reinterpret_cast<float *>(glds + G_DMIN_OFF)[par * GM + wm + lane] = dmin;
    };
    // 4 raw bytes (nibble h) -> two dwords of f16(sc6*q), exact (sc6*q <= 945), as the pairs (k0, k2) and (k1, k3): the
    // nibbles of bytes 0 and 2 are masked in place into the mantissas of two f16 (1024 + q, or 1024 + 16q for the high
    // nibbles), those of bytes 1 and 3 after one shift; one packed FMA takes the 1024 away and applies sc6.
    // `magic` is 0x64006400 held in a register so that mask-and-or is one instruction; `sp` is a table entry (s, -1024 s).
    uint32_t magic;
    asm volatile("v_mov_b32 %0, 0x64006400" : "=v"(magic));
    auto convert4 = [&](uint32_t raw, uint32_t h, uint32_t sp, uint32_t &o0, uint32_t &o1) {
        const f16x2 p = __builtin_bit_cast(f16x2, sp);
        const f16x2 sc2 = {p[0], p[0]}, off2 = {p[1], p[1]};  // (broadcast by the instruction's operand selects, not by a pack)
        const uint32_t mask = h ? 0x00F000F0u : 0x000F000Fu;
        const f16x2 m02 = __builtin_bit_cast(f16x2, (raw & mask) | magic);
        const f16x2 m13 = __builtin_bit_cast(f16x2, ((raw >> 8) & mask) | magic);
        o0 = __builtin_bit_cast(uint32_t, m02 * sc2 + off2);
        o1 = __builtin_bit_cast(uint32_t, m13 * sc2 + off2);
    };
    // The reads of the main loop are written as instructions with hand-counted waits: while LDS copies are in flight
    // the compiler's own wait for an LDS read is lgkmcnt(0), i.e. it would drain the reads issued ahead with the one
    // that is needed.  LDS reads return in order, so "all but the last n" is exact.
    const uint32_t lds0 = (uint32_t)(uintptr_t)(p_lds_vp)glds;
    const uint32_t raw_lane = lds0 + G_R_OFF + wave * 9216 + row32 * 144 + 16 + kgrp * 16;
    auto raw_of = [&](uint32_t par, uint32_t g4, u32x4 (&rq)[2]) {  // step g4 of the super-block in slot `par`
        const uint32_t a = raw_lane + par * G_R_STAGE + g4 * 32;
        asm volatile("ds_read_b128 %0, %1" : "=v"(rq[0]) : "v"(a));
        asm volatile("ds_read_b128 %0, %1 offset:4608" : "=v"(rq[1]) : "v"(a));
    };
    const uint32_t sc_lane = lds0 + G_SC_OFF + wave * 2048 + row32 * 4;
    auto scales_of = [&](uint32_t sub, uint32_t (&sp)[2]) {  // the table entries of sub-block `sub` for this lane's two rows
        const uint32_t a = sc_lane + sub * 256;
        asm volatile("ds_read_b32 %0, %1" : "=v"(sp[0]) : "v"(a));
        asm volatile("ds_read_b32 %0, %1 offset:128" : "=v"(sp[1]) : "v"(a));
    };
    const uint32_t b_lane = lds0 + G_B_OFF + row32 * 128;
    uint32_t b_col[4];  // byte position of this lane's chunk in a token's row, for the four MFMA depths (h, j) of a step
#pragma unroll
    for (int c = 0; c < 4; c++) b_col[c] = (((uint32_t)(c >> 1) * 4 + 2 * kgrp + (c & 1)) ^ ((row32 >> 1) & 7u)) << 4;

    f32x16 acc[2][4], D[2][4];  // the result; the integer sums of the current super-block
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int jj = 0; jj < 4; jj++)
#pragma unroll
            for (int e = 0; e < 16; e++) {
                acc[i][jj][e] = 0.f;
                D[i][jj][e] = 0.f;
            }

    // ---- prologue: the first super-block's weights and Sx, six pieces of the second's, activation steps 0..2; k 0..31 of step 0 converted ----
    issue_sx(sb_begin);
#pragma unroll
    for (int p9 = 0; p9 < 9; p9++) issue_raw(sb_begin, p9);
#pragma unroll
    for (int p9 = 0; p9 < 6; p9++) issue_raw(sb_begin + 1, p9);
#pragma unroll
    for (int q = 0; q < 4; q++) { issue_b(0, 0, q); issue_b(1, 1, q); issue_b(2, 2, q); }
    GEMM_WAIT_VMCNT(0);
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    stage_sb(0);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    u32x4 rq[2];        // this lane's raw bytes of the step whose halves are being converted
    uint32_t an[2][2][4];  // the operand of the coming half: [row block][j][dword]
    uint32_t scn[2];    // table entries for the conversions of the coming half
    u32x4 pf[4];        // the first G_LA operand reads of the coming step
    {
        uint32_t sp0[2];
        raw_of(0, 0, rq);
        scales_of(0, sp0);
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(rq[0]), "+v"(rq[1]), "+v"(sp0[0]), "+v"(sp0[1]));
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < 2; j++) {
                convert4(rq[i][2 * j], 0, sp0[i], an[i][j][0], an[i][j][1]);
                convert4(rq[i][2 * j + 1], 0, sp0[i], an[i][j][2], an[i][j][3]);
            }
        scales_of(1, scn);
#pragma unroll
        for (int G = 0; G < G_LA; G++) {
            const uint32_t a = b_lane + b_col[0] + G * 4096;
            asm volatile("ds_read_b128 %0, %1" : "=v"(pf[G]) : "v"(a));
        }
    }

    uint32_t s = 0;
    for (uint32_t sb = sb_begin; sb < sb_end; sb++) {
        const uint32_t par = (sb - sb_begin) & 1u;
#pragma unroll
        for (int g = 0; g < 4; g++, s++) {
            // ---- top of the step: (g = 3) the next super-block's tables, (g = 0) this one's offsets ----
            if (g == 3) {
                stage_sb(par ^ 1u);  // (its weights landed before the barrier of g = 2; the entries still needed of this one are in registers)
                asm volatile("" ::: "memory");
            }
            if (g == 0 && with_mins) {
                // sum_sub mn6 * Sx as one 16-deep MFMA per block (A slots 2*sub+h = the offsets' operand, B slots = Sx_h/32:
                // lane (row32, kgrp) holds slots 8kgrp .. 8kgrp+7)
                f16x8 amf[2], bmf[4];
#pragma unroll
                for (int i = 0; i < 2; i++) amf[i] = *reinterpret_cast<const f16x8 *>(glds + G_AM_OFF + (wm + i * 32 + row32) * 32 + kgrp * 16);
#pragma unroll
                for (int jj = 0; jj < 4; jj++) bmf[jj] = *reinterpret_cast<const f16x8 *>(glds + G_BM_OFF + (jj * 32 + row32) * 32 + kgrp * 16);
                // (D is free here: the products go there, then they are folded in with the rows' dmin)
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int jj = 0; jj < 4; jj++) {
                        f32x16 z;
#pragma unroll
                        for (int e = 0; e < 16; e++) z[e] = 0.f;
                        D[i][jj] = __builtin_amdgcn_mfma_f32_32x32x16_f16(amf[i], bmf[jj], z, 0, 0, 0);
                    }
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const f32x4 mv = *reinterpret_cast<const f32x4 *>(glds + G_DMIN_OFF + (par * GM + wm + i * 32 + q * 8 + kgrp * 4) * 4);
#pragma unroll
                        for (int jj = 0; jj < 4; jj++)
#pragma unroll
                            for (int e = 0; e < 4; e++)
                                acc[i][jj][4 * q + e] = __builtin_fmaf(-mv[e], D[i][jj][4 * q + e], acc[i][jj][4 * q + e]);
                    }
            }
            // ---- the step's sixteen operand reads (four depths x four token blocks) run G_LA groups ahead of the MFMAs that
            //      use them, into the next step at the end; the raw bytes of the next step are requested first ----
            u32x4 bf[16];
            u32x4 rqn[2];
            uint32_t b_addr[4];
#pragma unroll
            for (int c = 0; c < 4; c++) b_addr[c] = b_lane + (uint32_t)g * G_B_STAGE + b_col[c];
            const uint32_t b_next = b_lane + (uint32_t)((g + 1) & 3) * G_B_STAGE + b_col[0];
#define LARQL_RD(G) case G: asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(bf[G]) : "v"(b_addr[(G) >> 2]), "n"(((G) & 3) * 4096)); break;
#define LARQL_RN(G) case 16 + G: asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(pf[G]) : "v"(b_next), "n"((G) * 4096)); break;
            auto b_read = [&](int G) {
                switch (G) { LARQL_RD(4) LARQL_RD(5) LARQL_RD(6) LARQL_RD(7) LARQL_RD(8) LARQL_RD(9) LARQL_RD(10) LARQL_RD(11)
                             LARQL_RD(12) LARQL_RD(13) LARQL_RD(14) LARQL_RD(15) LARQL_RN(0) LARQL_RN(1) LARQL_RN(2) LARQL_RN(3) default: break; }
            };
#undef LARQL_RD
#undef LARQL_RN
            asm volatile("" ::: "memory");  // (nothing of the above sinks below the counted reads)
            __builtin_amdgcn_sched_barrier(0);
            raw_of(g == 3 ? par ^ 1u : par, (uint32_t)((g + 1) & 3), rqn);  // (own rows, own copies, landed before the barrier of the step before)
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int h = 0; h < 2; h++) {
                if (h == 1) {
                    // ---- middle of the step: everything requested before the last barrier has landed (after it: the step's 4
                    //      activation copies, plus 3 weight pieces and Sx at g = 0, 3 weight pieces at g = 2 and 3); after this
                    //      barrier everybody's activations of step s+1 are visible and everybody is done with step s-1, whose
                    //      slot the activations of step s+3 take.  The next super-block's weights are complete with the pieces
                    //      of g = 0, two barriers before their first use at the top of g = 3; the slot of the one after is free
                    //      from the top of g = 2.  The requests themselves go out one per MFMA group of the second half (a
                    //      burst of eight here costs the matrix cores 0.1-0.2 us) ----
                    if (g == 1) GEMM_WAIT_VMCNT(8);
                    else if (g == 2) GEMM_WAIT_VMCNT(4);
                    else GEMM_WAIT_VMCNT(7);
                    __builtin_amdgcn_s_barrier();
                    asm volatile("" ::: "memory");
                    __builtin_amdgcn_sched_barrier(0);
                }
                // ---- half h: the matrix cores take k 32h .. 32h+31 of step s; the threads convert, for h = 0, this step's
                //      high nibbles and, for h = 1, the next step's low nibbles.  Both halves of the operand belong to this
                //      wavefront alone ----
                if (h == 1) { rq[0] = rqn[0]; rq[1] = rqn[1]; }
                uint32_t scv[2] = {scn[0], scn[1]};
                // table entries for the conversions of the half after this one
                scales_of(h == 0 ? 2u * ((g + 1) & 3) : (g == 3 ? 1u : 2u * (g + 1) + 1u), scn);
                const uint32_t nib = 1 - h;                                 // nibble of the half being converted
                f16x8 af[2][2];
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int j = 0; j < 2; j++) af[i][j] = __builtin_bit_cast(f16x8, (u32x4){an[i][j][0], an[i][j][1], an[i][j][2], an[i][j][3]});
                __builtin_amdgcn_sched_barrier(0);
                // eight groups of two MFMAs; each carries one piece of the conversion
#pragma unroll
                for (int jj = 0; jj < 8; jj++) {
                    const int G = h * 8 + jj;
                    if (h == 1) {  // this group's copy request
                        if (jj < 4) issue_b(s + 3, (uint32_t)((g + 3) & 3), jj);
                        else if (jj < 7) {
                            if (g == 0) issue_raw(sb + 1, 6 + jj - 4);
                            if (g == 2) issue_raw(sb + 2, jj - 4);
                            if (g == 3) issue_raw(sb + 2, 3 + jj - 4);
                        } else if (g == 0) issue_sx(sb + 1);  // (everybody took this super-block's Sx before the barrier)
                    }
                    b_read(G + G_LA);
                    // operand G has arrived when at most the G_LA reads issued after it are outstanding (reads return in order;
                    // anything else issued in between only makes the wait stricter)
                    if (G < 4) asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(pf[G < 4 ? G : 0]));
                    else asm volatile("s_waitcnt lgkmcnt(4)" : "+v"(bf[G]));
                    // (these name what came back before this group's operand: they keep each piece of the conversion between
                    // two groups instead of wherever its first use is)
                    if (jj == 0) asm volatile("" : "+v"(scv[0]), "+v"(scv[1]), "+v"(rq[0]), "+v"(rq[1]));
                    {
                        const int i = jj >> 2, j = (jj >> 1) & 1, dd = jj & 1;
                        if (jj > 0) asm volatile("" : "+v"(an[(jj - 1) >> 2][((jj - 1) >> 1) & 1][2 * ((jj - 1) & 1)]), "+v"(an[(jj - 1) >> 2][((jj - 1) >> 1) & 1][2 * ((jj - 1) & 1) + 1]));
                        convert4(rq[i][2 * j + dd], nib, scv[i], an[i][j][2 * dd], an[i][j][2 * dd + 1]);
                    }
                    const f16x8 bv = __builtin_bit_cast(f16x8, G < 4 ? pf[G < 4 ? G : 0] : bf[G]);
                    const int j = (G >> 2) & 1, tb = G & 3;
#pragma unroll
                    for (int i = 0; i < 2; i++) {  // (a super-block's first MFMAs start from zero: D is never cleared)
                        f32x16 z;
#pragma unroll
                        for (int e = 0; e < 16; e++) z[e] = 0.f;
                        D[i][tb] = __builtin_amdgcn_mfma_f32_32x32x16_f16(af[i][j], bv, (g == 0 && h == 0 && j == 0) ? z : D[i][tb], 0, 0, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                asm volatile("" ::: "memory");
            }
            if (g == 3) {
                // ---- end of the super-block: acc += d * D ----
#pragma unroll
                for (int i = 0; i < 2; i++)
#pragma unroll
                    for (int q = 0; q < 4; q++) {
                        const f32x4 dv = *reinterpret_cast<const f32x4 *>(glds + G_D_OFF + (par * GM + wm + i * 32 + q * 8 + kgrp * 4) * 4);
#pragma unroll
                        for (int jj = 0; jj < 4; jj++)
#pragma unroll
                            for (int e = 0; e < 4; e++)
                                acc[i][jj][4 * q + e] = __builtin_fmaf(dv[e], D[i][jj][4 * q + e], acc[i][jj][4 * q + e]);
                    }
                asm volatile("" ::: "memory");
            }
        }
    }
    // the clamped requests past the end and the operand reads issued for a step that does not exist
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(pf[0]), "+v"(pf[1]), "+v"(pf[2]), "+v"(pf[3]), "+v"(scn[0]), "+v"(scn[1]));
    GEMM_WAIT_VMCNT(0);

    // Results leave through LDS so that a store instruction writes whole lines: each wavefront parks its 64-row x
    // 128-token block as [token][row] (token rows padded to 68 floats: the 8 lanes of a write phase hit 8 bank
    // groups) in its own 34 KB, then every lane stores 16 bytes of a 256-byte run of one token.
    __builtin_amdgcn_s_barrier();  // nobody's copies are still landing in what becomes another wavefront's block
    asm volatile("" ::: "memory");
    constexpr uint32_t EP_LD = G_EP_LD;
    float *blk = reinterpret_cast<float *>(glds) + wave * (GN * EP_LD);
#pragma unroll
    for (int i = 0; i < 2; i++)
#pragma unroll
        for (int jj = 0; jj < 4; jj++)
#pragma unroll
            for (int q = 0; q < 4; q++)  // registers 4q .. 4q+3 of a block: rows 8q + 4kgrp .. +3, token row32
                *reinterpret_cast<f32x4 *>(blk + (jj * 32 + row32) * EP_LD + i * 32 + q * 8 + kgrp * 4) =
                    (f32x4){acc[i][jj][4 * q], acc[i][jj][4 * q + 1], acc[i][jj][4 * q + 2], acc[i][jj][4 * q + 3]};
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // own writes, own reads
    const bool vec_ok = (rows & 3u) == 0 && (((uintptr_t)(partial ? partial : out)) & 15u) == 0;
    const uint32_t rc = (lane & 15u) * 4, r = row0 + wm + rc;
#pragma unroll 4
    for (int it = 0; it < 32; it++) {
        const uint32_t tl = it * 4 + (lane >> 4), tok = tok0 + tl;
        if (tok >= seq) continue;
        f32x4 v = *reinterpret_cast<const f32x4 *>(blk + tl * EP_LD + rc);
        float *o = partial ? partial + ((size_t)blockIdx.z * seq + tok) * rows + r : out + (size_t)tok * rows + r;
        // (partial sums stay without the token's scale; q4k_gemm_reduce_kernel adds the slabs in order and applies it)
        const float ts = partial ? 1.f : tok_scale[tok];
#pragma unroll
        for (int e = 0; e < 4; e++) v[e] *= ts;
        if (vec_ok && r + 3 < rows) {
            f32x4 *ov = reinterpret_cast<f32x4 *>(o);
            if (!partial && accumulate) { const f32x4 old = *ov; v += old; }
            *ov = v;
        } else {
#pragma unroll
            for (int e = 0; e < 4; e++)
                if (r + e < rows) o[e] = (!partial && accumulate) ? o[e] + v[e] : v[e];
        }
    }
}

// ---------------------------------------------------------------------------
// The device tier's kernel: one workgroup of 8 wavefronts, two per SIMD, owns 256 rows against a tile of tokens.  The two
// wavefronts of a SIMD (w and w + 4) share 64 rows and either
//   * split every step's k (KS; 16 TB <= 128 tokens): wavefront kh takes the nibbles kh of the same raw bytes against all of
//     the tile's tokens: no weight converted twice; the pair adds its sums through LDS at the end; or
//   * split the tokens (128 each of 256): each converts all weights of the rows, but copies, super-block tables, prologue and
//     end serve twice the tokens and nothing is added at the end.
// A step is 64 k, half a step 32 (one nibble of 32 raw bytes per row = one sub-block).  In half a step a wavefront
// *prepares* (the activation operands from LDS into registers, the weight operand converted in registers: lane (row r16, kq)
// needs the nibbles of 8 consecutive raw bytes) and *multiplies* (4 x TB v_mfma_f32_16x16x32_f16).  One wavefront of the pair
// prepares first and one multiplies first, with one barrier per half step, so that one's vector instructions fall
// into the other's MFMAs.  (A barrier after each of the two, the form before, makes a half step twice the longer of the two:
// 1931 cycles per step of 128 tokens where the MFMAs take 1024; with one 1689, with table entries and raw bytes read ahead
// 1614, with the copies asked for between MFMAs 1541; without the offsets, all four.)
// Everything comes into LDS by global_load_lds: the f16 activations of a step into a ring (128 bytes per token; chunk c
// of token r at position c ^ ((r >> 1) & 7), chosen on the global side of the copy: no bank conflicts), the weights a super-block at a
// time (144 bytes per row: a row's two or three cache lines are asked for once) into two stages.  kh = 0 asks for
// the activations, kh = 1 for the weights, between its MFMAs: a copy instruction whose lanes lie in many cache lines holds up
// the wavefront that issues it (nine in a row: 0.4 us).  Per super-block two threads per row turn the header into table entries:
// the scales for the lanes that convert, and the offsets' operand.
// The offsets are one MFMA of depth 32 per block and super-block (an eighth of the MFMAs more, and half a kilobyte of Sx per 16 tokens),
// at the super-block's first half step; timing-only builds, 15360 x 3840 with 512 tokens (72.4 us a call): without
// the offsets' MFMAs 69.1, without their table entries 69.4, without the sums' copies 72.2.
// Bound by the schedule, then by power: a wavefront's two phases are a chain, which leaves the matrix pipe busy 53 % of the cycles of a call of 2048
// tokens (40 % with 512), and the clock is 2.1 GHz under operands of normal values, 2.4 under zeros (232 and 197 us).  16 x 16 x 32 MFMAs because a loop
// of them ran at a 10 % higher clock than the same work in 32 x 32 x 16, which read and write twice the accumulators per operation.
// Measured on one GPU, us per call with the exponents given: two barriers per half step, 32 x 32 x 16 MFMAs and one f16 per offset | the whole
// weight in one f16, no offsets | this: 15360 x 3840 with 2048 tokens 279 | 218 | 237, 512 74.2 | 64.5 | 71.4; 3840 x 15360 with 77 35.0 | 31.8 | 33.9,
// 16 25.0 | 20.8 | 21.9; 13270 x 3840 with 1783 234 | 188 | 203; 12607 x 1280 with 1817 118 | 88 | 94 (rows no multiple of four: the results in
// four-byte stores in the first).
// ---------------------------------------------------------------------------
constexpr int QTHREADS = 512;
constexpr uint32_t Q_B_BYTES = 65536, Q_R_STAGE = GM * 144;  // activation ring; weights of a super-block, two of them
constexpr uint32_t Q_R_OFF = Q_B_BYTES, Q_O_OFF = Q_R_OFF + 2 * Q_R_STAGE, Q_M_OFF = Q_O_OFF + GM * 32;  // offsets of a super-block, the activations' sums
constexpr uint32_t Q_D_OFF = Q_M_OFF + 2 * GN * 32, Q_E_OFF = Q_D_OFF + 2 * GM * 4, Q_S_OFF = Q_E_OFF + GM * 4, Q_LDS_BYTES = Q_S_OFF + 2 * GN * 4;
static_assert(Q_LDS_BYTES <= 160 * 1024, "one workgroup per CU");
// one global -> LDS copy of 16 bytes per lane: uniform base + per-lane 32-bit offset on the global side (no 64-bit
// address registers), uniform LDS address (the lanes' 16-byte slots follow one another from there)
__device__ __forceinline__ void copy16_to_lds(const void *base, uint32_t lane_off, uint32_t lds_addr) {
    const uint64_t b = (uint64_t)(uintptr_t)base;  // (uniform by construction: told to the compiler, which otherwise may keep them in vector registers)
    const uint64_t bs = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(lane_off), "s"(bs) : "memory");  // (m0 is not the compiler's to allocate; nothing else in these kernels uses it)
}

// four bytes per lane, likewise
__device__ __forceinline__ void copy4_to_lds(const void *base, uint32_t lane_off, uint32_t lds_addr) {
    const uint64_t b = (uint64_t)(uintptr_t)base;
    const uint64_t bs = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(b >> 32)) << 32) | (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)b);
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dword %1, %2" ::"s"(__builtin_amdgcn_readfirstlane((int)lds_addr)), "v"(lane_off), "s"(bs) : "memory");
}

// up to four neighbouring results; `left` of them are inside the matrix.  (A 16-byte store needs four-byte alignment only.)
__device__ __forceinline__ void store4(float *o, f32x4 v, uint32_t left) {
    if (left >= 4) {
        *reinterpret_cast<f32x4_a4 *>(o) = v;
    } else {
        if (left > 0) o[0] = v[0];
        if (left > 1) o[1] = v[1];
        if (left > 2) o[2] = v[2];
    }
}

template <int TB, bool KS>
__global__ void __launch_bounds__(QTHREADS) q4k_gemm_pair_kernel(const uint8_t *w, const uint16_t *xh, const uint16_t *sx, const int *__restrict__ rexp,
                                                                  const float *__restrict__ tok_scale, float *__restrict__ out,
                                                                  uint32_t rows, uint32_t hidden, uint32_t seq, uint32_t row_tiles, uint32_t tok_tiles,
                                                                  uint32_t sb_per_split, float *__restrict__ partial) {
    static_assert(TB % 2 == 0 && TB <= 8 && (KS || TB == 8), "");
    constexpr uint32_t NT = KS ? 16 * TB : 32 * TB;                // tokens of the tile
    constexpr uint32_t B_STAGE = KS ? 16384 : 32768, NB = Q_B_BYTES / B_STAGE;  // a step's activations (128 bytes a token), and how many of them
    constexpr int CP = NT / 32;                                    // activation copies of a wavefront kh = 0 for a step
    extern __shared__ __attribute__((aligned(16))) uint8_t glds[];
    const uint32_t t = threadIdx.x, lane = t & 63u, wave = __builtin_amdgcn_readfirstlane(t >> 6);
    const uint32_t wq = wave & 3u, kh = wave >> 2;  // row group; which of the pair: wavefronts w and w + 4 run on one SIMD
    // which tile: workgroups are dealt to the eight XCDs in turn; each takes a contiguous part of the list of tiles, in which four
    // token tiles of a row tile follow one another (an XCD's 32 workgroups then share 8 row tiles and 4 token tiles in its L2)
    uint32_t id = blockIdx.x;
    {
        const uint32_t total = gridDim.x, q = total >> 3, r = total & 7u, xcd = id & 7u, ix = id >> 3;
        id = xcd * q + min(xcd, r) + ix;
    }
    const uint32_t per_range = row_tiles * tok_tiles, range = __builtin_amdgcn_readfirstlane(id / per_range);
    id -= range * per_range;
    constexpr uint32_t TG = 4;
    const uint32_t tg = id / (row_tiles * TG), in = id - tg * row_tiles * TG, tw = min(TG, tok_tiles - tg * TG);
    const uint32_t row0 = __builtin_amdgcn_readfirstlane((in / tw) * GM), tok0 = __builtin_amdgcn_readfirstlane((tg * TG + in % tw) * NT);
    const uint32_t nsb = hidden >> 8, row_bytes = nsb * 144;
    const uint32_t sb_begin = range * sb_per_split, sb_end = min(nsb, sb_begin + sb_per_split);
    if (sb_begin >= sb_end) return;
    const uint32_t nsteps = (sb_end - sb_begin) * 4;
    const uint32_t wm = wq * 64;
    const uint32_t lds0 = (uint32_t)(uintptr_t)(p_lds_vp)glds;

    // copies.  kh = 1: a super-block of the pair's 64 rows is nine pieces; piece p, lane l brings 16-byte chunk (64p + l) % 9 of row
    // (64p + l) / 9, so that the rows lie in LDS one after the other.  kh = 0: a step's activations, CP pieces of 8 tokens
    const uint8_t *wt = w + (size_t)row0 * row_bytes;                                          // uniform
    const uint8_t *xt = (const uint8_t *)xh + (size_t)tok0 * hidden * 2;                       // uniform
    const uint8_t *st = (const uint8_t *)sx + (size_t)tok0 * 32;                               // uniform
    uint32_t c_off[9], m_off[2];
    if (kh) {
#pragma unroll
        for (int p = 0; p < 9; p++) {
            const uint32_t idx = p * 64 + lane;
            c_off[p] = (min(row0 + wm + idx / 9, rows - 1) - row0) * row_bytes + (idx % 9) * 16;
        }
    } else {
#pragma unroll
        for (int q = 0; q < 9; q++) {
            const uint32_t r = (wq + 4 * (q < CP ? q : 0)) * 8 + (lane >> 3);
            c_off[q] = (min(tok0 + r, seq - 1) - tok0) * hidden * 2 + (((lane & 7u) ^ ((r >> 1) & 7u)) * 16);
        }
    }
    // and kh = 0 a super-block's sums Sx/32 ([token][8 pairs]), MP pieces of 32 tokens
    constexpr int MP = KS ? 1 : 2;
#pragma unroll
    for (int q = 0; q < 2; q++) m_off[q] = (min(tok0 + q * 128 + wq * 32 + (lane >> 1), seq - 1) - tok0) * 32 + (lane & 1u) * 16;
    // (requests past the end are clamped: same number of copies in flight, results unused)
    auto issue_raw = [&](uint32_t sb, int p) {  // one of the nine pieces of a super-block
        copy16_to_lds(wt + (size_t)min(sb, sb_end - 1) * 144, c_off[p], lds0 + Q_R_OFF + ((sb - sb_begin) & 1u) * Q_R_STAGE + wq * 9216 + p * 1024);
    };
    auto issue_b = [&](uint32_t s, uint32_t slot, int q) {  // one of the CP pieces of a step
        copy16_to_lds(xt + ((size_t)sb_begin * 4 + min(s, nsteps - 1)) * 128, c_off[q], lds0 + slot * B_STAGE + (wq + 4 * q) * 1024);
    };
    auto issue_sx = [&](uint32_t sb, int q) {
        copy16_to_lds(st + (size_t)min(sb, sb_end - 1) * seq * 32, m_off[q], lds0 + Q_M_OFF + wq * 1024 + q * 4096);
    };

    // A super-block's header -> table entries, 32 rows of the pair's per wavefront: lane l takes the sub-blocks 4 (l / 32) .. + 3 of a row.
    //   part 0: the offsets' operand v = 32 (7.5 d sc6 - dmin mn6) 2^E as an f16 pair, [row][4 x high of the sub-blocks 0 .. 3 | 4 .. 7 | 4 x low ..]
    //           (both cut off, not rounded: one instruction for two; the pair has v to 2^-21)
    //   part 1: the scales 32 sc6 as f16 in the header's own 16 bytes (no other wavefront reads them as a header), and 2^15 d 2^E
    const uint32_t srow = wm + kh * 32 + (lane & 31u), sub4 = lane >> 5;
    float row_f = 0.f;  // 2^(E + 5), max(|d|, |dmin|/16) 2^E < 1 over the whole row srow
    auto header_of = [&](const uint32_t par) { return *reinterpret_cast<const u32x4 *>(glds + Q_R_OFF + par * Q_R_STAGE + srow * 144); };
    auto stage = [&](const uint32_t par, const int part, u32x4 hdr) {
        uint8_t *const hp = glds + Q_R_OFF + par * Q_R_STAGE + srow * 144;
        asm volatile("" : "+v"(hdr) :: "memory");  // (both lanes of a row have read it before either writes, and in one piece)
        const float df = half_to_float(hdr.x & 0xFFFFu) * row_f;
        // the 6-bit scales and mins of the four sub-blocks, a byte each
        const uint32_t m = 0u - sub4;  // (selected by masks: the compiler makes branches of ?:)
        const uint32_t sc4 = (((hdr.w & 0x0F0F0F0Fu) | ((hdr.y >> 2) & 0x30303030u)) & m) | (hdr.y & 0x3F3F3F3Fu & ~m);
        if (part) {
            // (bytes under the exponent of 1024: 1024 + sc6, times 32 less 32768)
            const f16x2 c = {(_Float16)-32768.f, (_Float16)-32768.f}, k = {(_Float16)32.f, (_Float16)32.f};
            const f16x2 s01 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(sc4, 0x64646464u, 0x00050004u)), s23 = __builtin_bit_cast(f16x2, __builtin_amdgcn_perm(sc4, 0x64646464u, 0x00070006u));
            *reinterpret_cast<u32x2 *>(hp + sub4 * 8) = (u32x2){__builtin_bit_cast(uint32_t, __builtin_elementwise_fma(s01, k, c)), __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(s23, k, c))};
            *reinterpret_cast<uint32_t *>(glds + Q_D_OFF + par * GM * 4 + srow * 4) = (uint32_t)__builtin_bit_cast(uint16_t, (_Float16)(1024.f * df));
        } else {
            const uint32_t mn4 = ((((hdr.w >> 4) & 0x0F0F0F0Fu) | ((hdr.z >> 2) & 0x30303030u)) & m) | (hdr.z & 0x3F3F3F3Fu & ~m);
            const float ds = 7.5f * df, dm = half_to_float(hdr.x >> 16) * row_f;
            u32x2 hi, lo;
#pragma unroll
            for (int k = 0; k < 2; k++) {
                const float v0 = ds * (float)((sc4 >> (16 * k)) & 0xFFu) - dm * (float)((mn4 >> (16 * k)) & 0xFFu);
                const float v1 = ds * (float)((sc4 >> (16 * k + 8)) & 0xFFu) - dm * (float)((mn4 >> (16 * k + 8)) & 0xFFu);
                const f16x2 h = __builtin_bit_cast(f16x2, __builtin_amdgcn_cvt_pkrtz(v0, v1));
                hi[k] = __builtin_bit_cast(uint32_t, h);
                lo[k] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_pkrtz(v0 - (float)h[0], v1 - (float)h[1]));
            }
            *reinterpret_cast<u32x2 *>(glds + Q_O_OFF + srow * 32 + sub4 * 8) = hi;
            *reinterpret_cast<u32x2 *>(glds + Q_O_OFF + srow * 32 + 16 + sub4 * 8) = lo;
        }
    };
    // 4 raw bytes, nibble h -> two dwords of f16(d sc6 (q - 7.5)) as the pairs (k0, k2) and (k1, k3).  The nibbles go to bits 4 .. 7 of
    // two f16, subnormals of the value q 2^-20 (f16 subnormals cost nothing here); times 32 sc6 less 7.5 sc6 2^-15 is sc6 (q - 7.5) 2^-15,
    // exact; the product with 2^15 d rounds once
    auto convert4 = [&](uint32_t raw, const int h, f16x2 sc, f16x2 c, f16x2 d, uint32_t &o0, uint32_t &o1) {
        const f16x2 m02 = __builtin_bit_cast(f16x2, (h ? raw : raw << 4) & 0x00F000F0u);
        const f16x2 m13 = __builtin_bit_cast(f16x2, (h ? raw >> 8 : raw >> 4) & 0x00F000F0u);
        o0 = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(m02, sc, c) * d);
        o1 = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(m13, sc, c) * d);
    };
    const uint32_t r16 = lane & 15u, kq = lane >> 4;
    const uint32_t raw_lane = lds0 + Q_R_OFF + wq * 9216 + r16 * 144 + 16 + kq * 8;
    const uint32_t tab_lane = lds0 + Q_R_OFF + (wm + r16) * 144, d_lane = lds0 + Q_D_OFF + (wm + r16) * 4;
    // offsets: a lane's eight products of the 16 x 16 x 32 MFMA are v_high (kq = 0, 1) or v_low (2, 3) of four sub-blocks, each twice,
    // against those sub-blocks' Sx/32 pairs.  KS: each of the pair adds them for the half of the rows that it stores
    constexpr int OI = KS ? 2 : 4;  // row blocks that this wavefront stores
    const uint32_t i0 = KS ? 2 * kh : 0;
    const uint32_t o_lane = lds0 + Q_O_OFF + (wm + i0 * 16 + r16) * 32 + kq * 8;
    const uint32_t m_lane = lds0 + Q_M_OFF + (KS ? 0u : kh * 4096) + r16 * 32 + (kq & 1u) * 16;
    uint32_t b_lane[2];  // for the two halves of a step
#pragma unroll
    for (int h = 0; h < 2; h++)
        b_lane[h] = lds0 + (KS ? 0u : kh * 16384) + r16 * 128 + ((((uint32_t)h * 4 + kq) ^ ((r16 >> 1) & 7u)) << 4);

    f32x4 acc[4][TB];
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < TB; j++) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
    u32x4 an[4] = {};      // the weight operand being prepared / multiplied, by row blocks
    u32x4 breg[8] = {};    // its activation operands
    u32x2 rq[4];
    uint32_t sp[4];        // raw bytes and table entries (two scales) of the step
    uint32_t dd[4];        // d of the super-block

    // raw bytes and table entries of a step, read while the half step before it multiplies.  (Written as instructions, as all
    // LDS reads of the loop: the wait for them stands behind the MFMAs, tied to their registers.)
    auto fetch = [&](auto GG, const uint32_t sb) {
        constexpr int g = decltype(GG)::value;
        uint32_t (&dr)[4] = dd;
        uint32_t (&spr)[4] = sp;
        const uint32_t par = (sb - sb_begin) & 1u;
        const uint32_t ra = raw_lane + par * Q_R_STAGE, ta = tab_lane + par * Q_R_STAGE;
#define LARQL_RS(i) asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(spr[i]) : "v"(ta), "n"(g * 4 + (i) * 2304)); \
                    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(rq[i]) : "v"(ra), "n"(g * 32 + (i) * 2304));
        LARQL_RS(0) LARQL_RS(1) LARQL_RS(2) LARQL_RS(3)
#undef LARQL_RS
        if (g == 0) {
            const uint32_t da = d_lane + par * GM * 4;
            asm volatile("ds_read_b32 %0, %1" : "=v"(dr[0]) : "v"(da));
            asm volatile("ds_read_b32 %0, %1 offset:64" : "=v"(dr[1]) : "v"(da));
            asm volatile("ds_read_b32 %0, %1 offset:128" : "=v"(dr[2]) : "v"(da));
            asm volatile("ds_read_b32 %0, %1 offset:192" : "=v"(dr[3]) : "v"(da));
        }
    };
    auto arrived = [&]() {
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(rq[0]), "+v"(rq[1]), "+v"(rq[2]), "+v"(rq[3]), "+v"(sp[0]), "+v"(sp[1]), "+v"(sp[2]), "+v"(sp[3]),
                     "+v"(dd[0]), "+v"(dd[1]), "+v"(dd[2]), "+v"(dd[3]));
    };
    // prepare half step (g, h) of super-block sb; at g = 2 also the tables of sb + 1, whose weights landed at g = 1
    auto prepare = [&](auto KH, auto GG, auto HH, const uint32_t sb) {
        constexpr int khc = decltype(KH)::value, g = decltype(GG)::value, h = decltype(HH)::value;
        constexpr int slot = g % (int)NB;
        const uint32_t par = (sb - sb_begin) & 1u;
#define LARQL_RB(j) if constexpr ((j) < TB) asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(breg[j]) : "v"(b_lane[h]), "n"(slot * (int)B_STAGE + (j) * 2048));
        LARQL_RB(0) LARQL_RB(1) LARQL_RB(2) LARQL_RB(3) LARQL_RB(4) LARQL_RB(5) LARQL_RB(6) LARQL_RB(7)
#undef LARQL_RB
        u32x4 hdr = {};
        if (g == 2) hdr = header_of(par ^ 1u);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const f16x2 e = __builtin_bit_cast(f16x2, sp[i]), dp = __builtin_bit_cast(f16x2, dd[i]);
            const f16x2 sc = {e[h], e[h]}, d = {dp[0], dp[0]}, c = sc * (_Float16)(-7.5f * 0x1p-20f);
            uint32_t o0, o1, o2, o3;
            convert4(rq[i].x, h, sc, c, d, o0, o1);
            convert4(rq[i].y, h, sc, c, d, o2, o3);
            an[i] = (u32x4){o0, o1, o2, o3};
        }
        if (g == 2 && (KS || h == 0)) stage(par ^ 1u, 0, hdr);
        if (g == 2 && (KS || h == 1)) stage(par ^ 1u, 1, hdr);
        // ("memory": the table entries are written before it as well)
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(breg[0]), "+v"(breg[1]), "+v"(breg[2]), "+v"(breg[3]), "+v"(breg[4]), "+v"(breg[5]), "+v"(breg[6]), "+v"(breg[7]) :: "memory");
        if (khc == 1 && g == 1 && (KS || h == 1)) GEMM_WAIT_VMCNT(0);
        __builtin_amdgcn_s_setprio(3);  // (the multiply phase comes next)
    };
    // multiply it; fetch the next step's raw bytes; ask for the activations three steps ahead (KS; else the next step's, whose slot the step
    // before released) or for the weights two super-blocks ahead.  Own copies that may still fly at the end: the activations of the
    // two steps after the next; of the weights everything, until g = 1 prepares
    auto multiply = [&](auto KH, auto GG, auto HH, auto GN, const uint32_t s, const uint32_t sb, const uint32_t sbn) {
        constexpr int khc = decltype(KH)::value, g = decltype(GG)::value, h = decltype(HH)::value;
        constexpr bool offs = g == 0 && (KS || h == 0);  // the super-block's offsets come with its first half step
        if (KS || h == 1) fetch(GN, sbn);
        u32x2 ov[4] = {};
        u32x4 oa[OI];
        if constexpr (offs) {
            asm volatile("ds_read_b64 %0, %1" : "=v"(ov[0]) : "v"(o_lane));
            asm volatile("ds_read_b64 %0, %1 offset:512" : "=v"(ov[1]) : "v"(o_lane));
            if constexpr (!KS) {
                asm volatile("ds_read_b64 %0, %1 offset:1024" : "=v"(ov[2]) : "v"(o_lane));
                asm volatile("ds_read_b64 %0, %1 offset:1536" : "=v"(ov[3]) : "v"(o_lane));
            }
        }
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("s_nop 1");  // (the operand may have been written by the instruction before)
        auto request = [&](const int k) {
            if (khc == 0) {
                // (the sums of the next super-block: their readers' last half step, the offsets' below, is a barrier and more ago)
                if (g == 2 && (KS || h == 0) && k == 0)
#pragma unroll
                    for (int q = 0; q < MP; q++) issue_sx(sb + 1, q);
                if (KS && k % 8 == 3) issue_b(s + 3, (g + 3) & 3, k / 8);
                if (!KS && h == 0 && k % 4 == 3) issue_b(s + 1, (g + 1) & 1, k / 4);
            } else if ((KS || h == 1) && (g == 2 || g == 3)) {
                // three pieces in the second half of g = 2, six in g = 3
                if (g == 2 && k == 2 * TB - 1) arrived();  // (the slot's last readers: this wavefront here, its pair a barrier ago)
                if (g == 2 && k >= 2 * TB && (k - 2 * TB) % (TB / 2) == 0 && (k - 2 * TB) / (TB / 2) < 3) issue_raw(sb + 2, (k - 2 * TB) / (TB / 2));
                if (g == 3 && k % (TB / 2) == 0 && k / (TB / 2) < 6) issue_raw(sb + 2, 3 + k / (TB / 2));
            }
        };
#pragma unroll
        for (int j = 0; j < TB; j++) {
#pragma unroll
            for (int i = 0; i < 4; i++) {
                asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(acc[i][j]) : "v"(an[i]), "v"(breg[j]));
                request(j * 4 + i);
            }
            if constexpr (offs) {
                asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(breg[j]) : "v"(m_lane), "n"(j * 512));
                if (j == 1) {
                    asm volatile("s_waitcnt lgkmcnt(2)" : "+v"(ov[0]), "+v"(ov[1]), "+v"(ov[2]), "+v"(ov[3]));
#pragma unroll
                    for (int i = 0; i < OI; i++)
                        oa[i] = (u32x4){__builtin_amdgcn_perm(0u, ov[i].x, 0x01000100u), __builtin_amdgcn_perm(0u, ov[i].x, 0x03020302u),
                                        __builtin_amdgcn_perm(0u, ov[i].y, 0x01000100u), __builtin_amdgcn_perm(0u, ov[i].y, 0x03020302u)};
                }
            }
        }
        if constexpr (offs) {
            __builtin_amdgcn_sched_barrier(0);
            asm volatile("s_nop 1");
#pragma unroll
            for (int j = 0; j < TB; j++) {
                asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(breg[j]) : "n"(TB - 1 - j));
#pragma unroll
                for (int i = 0; i < OI; i++)
                    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+v"(acc[(KS ? 2 * khc : 0) + i][j]) : "v"(oa[i]), "v"(breg[j]));
            }
        }
        __builtin_amdgcn_s_setprio(0);
        arrived();
        if (khc == 0) {
            // (g = 2: the sums asked for first in this half step may fly as well; they are here a barrier before their first reader)
            if (KS && g == 2) GEMM_WAIT_VMCNT(2 * CP + MP);
            else if (KS) GEMM_WAIT_VMCNT(2 * CP);
            else if (h == 1) GEMM_WAIT_VMCNT(0);
        }
    };
    auto half_end = [&]() {
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" ::: "memory");
    };

    // ---- prologue: exponents and token scales, the first two super-blocks' weights, the first activation steps; tables of the first ----
    if (kh) {
        copy4_to_lds(rexp + row0, (min(row0 + wm + lane, rows - 1) - row0) * 4, lds0 + Q_E_OFF + wm * 4);
#pragma unroll
        for (int p = 0; p < 9; p++) issue_raw(sb_begin, p);
#pragma unroll
        for (int p = 0; p < 9; p++) issue_raw(sb_begin + 1, p);
        GEMM_WAIT_VMCNT(9);
    } else {
        copy4_to_lds(tok_scale + tok0, (min(tok0 + wm + lane, seq - 1) - tok0) * 4, lds0 + Q_S_OFF + wm * 4);
#pragma unroll
        for (int q = 0; q < MP; q++) issue_sx(sb_begin, q);
#pragma unroll
        for (int st = 0; st < (KS ? 3 : 1); st++)
#pragma unroll
            for (int q = 0; q < CP; q++) issue_b(st, st, q);
        GEMM_WAIT_VMCNT(KS ? 2 * CP : 0);
    }
    half_end();
    row_f = ldexpf(1.f, reinterpret_cast<const int *>(glds + Q_E_OFF)[srow] + 5);
    {
        const u32x4 hdr = header_of(0);
        stage(0, 0, hdr);
        stage(0, 1, hdr);
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    half_end();
    //   kh = 0:  P(0) | M(0) | P(1) M(1) | P(2) M(2) | ...
    //   kh = 1:       | P(0) | M(0) P(1) | M(1) P(2) | ...          (| = barrier)
    // What half step n reads of LDS was read before the barrier behind P(n): its slots are asked for again after it.
    auto run = [&](auto KH) {
        constexpr int khc = decltype(KH)::value;
        constexpr std::integral_constant<int, 0> I0;
        constexpr std::integral_constant<int, KS ? khc : 0> H0;
        fetch(I0, sb_begin);
        arrived();
        if (khc == 0) prepare(KH, I0, H0, sb_begin);
        half_end();
        uint32_t s = 0;
        for (uint32_t sb = sb_begin; sb < sb_end; sb++) {
            auto turn = [&](auto GG, auto HH, auto GN, auto HN) {  // this half step, and the one after
                constexpr int g = decltype(GG)::value, gn = decltype(GN)::value;
                const uint32_t sbn = gn == 0 && g == 3 ? sb + 1 : sb;
                if (khc == 0) {
                    multiply(KH, GG, HH, GN, s, sb, sbn);
                    half_end();
                    prepare(KH, GN, HN, sbn);
                } else {
                    prepare(KH, GG, HH, sb);
                    half_end();
                    multiply(KH, GG, HH, GN, s, sb, sbn);
                }
            };
            constexpr std::integral_constant<int, 1> I1;
            constexpr std::integral_constant<int, 2> I2;
            constexpr std::integral_constant<int, 3> I3;
            if constexpr (KS) {
                turn(I0, H0, I1, H0); s++; turn(I1, H0, I2, H0); s++; turn(I2, H0, I3, H0); s++; turn(I3, H0, I0, H0); s++;
            } else {
                turn(I0, I0, I0, I1); turn(I0, I1, I1, I0); s++; turn(I1, I0, I1, I1); turn(I1, I1, I2, I0); s++;
                turn(I2, I0, I2, I1); turn(I2, I1, I3, I0); s++; turn(I3, I0, I3, I1); turn(I3, I1, I0, I0); s++;
            }
        }
    };
    if (!kh) run(std::integral_constant<int, 0>{});
    else run(std::integral_constant<int, 1>{});
    GEMM_WAIT_VMCNT(0);  // the clamped requests past the end

    asm volatile("s_nop 15\n\ts_nop 15");  // (results of the last multiplications are not read for 18 cycles)
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < TB; j++) asm volatile("" : "+v"(acc[i][j]));
    // ---- results: lane (token r16, kq) holds rows 4 kq .. 4 kq + 3 of every block of 16 x 16 ----
    constexpr int I = OI;
    f32x4 back[I];
#pragma unroll
    for (int i = 0; i < I; i++) {
        const i32x4 e = *reinterpret_cast<const i32x4 *>(glds + Q_E_OFF + (wm + (i0 + i) * 16 + kq * 4) * 4);
        back[i] = (f32x4){ldexpf(1.f, -e[0]), ldexpf(1.f, -e[1]), ldexpf(1.f, -e[2]), ldexpf(1.f, -e[3])};
    }
    if (KS) {
        __builtin_amdgcn_s_barrier();  // nobody's copies are still landing in what becomes somebody's block
        asm volatile("" ::: "memory");
        f32x4 *blk = reinterpret_cast<f32x4 *>(glds) + wave * (2 * TB * 64);
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < TB; j++) blk[(i * TB + j) * 64 + lane] = kh ? acc[i][j] : acc[2 + i][j];
        __syncthreads();
        const f32x4 *other = reinterpret_cast<const f32x4 *>(glds) + (wave ^ 4u) * (2 * TB * 64);
#pragma unroll
        for (int i = 0; i < 2; i++)
#pragma unroll
            for (int j = 0; j < TB; j++) acc[i][j] = (kh ? acc[2 + i][j] : acc[i][j]) + other[(i * TB + j) * 64 + lane];
    }
#pragma unroll
    for (int j = 0; j < TB; j++) {
        const uint32_t tok = tok0 + (KS ? 0u : kh * 128) + j * 16 + r16;
        if (tok >= seq) continue;
        // (partial sums stay without the token's scale; q4k_gemm_reduce_kernel adds the slabs in order and applies it)
        const float ts = partial ? 1.f : reinterpret_cast<const float *>(glds + Q_S_OFF)[tok - tok0];
        const uint32_t r = row0 + wm + i0 * 16 + kq * 4;
        float *o = (partial ? partial + ((size_t)range * seq + tok) * rows : out + (size_t)tok * rows) + r;
#pragma unroll
        for (int i = 0; i < I; i++) {
            f32x4 v = acc[i][j];
#pragma unroll
            for (int e = 0; e < 4; e++) v[e] *= ts * back[i][e];
            store4(o + i * 16, v, rows - min(rows, r + i * 16));
        }
    }
}

// activations -> f16 terms, sub-block sums and token scales; with `rexp`, the weight rows' exponents as well
hipError_t q4k_gemm_prep_launch(hipStream_t s, const void *x, int x_is_bf16, uint32_t hidden, uint32_t seq, uint16_t *xh, uint16_t *xl,
                                uint16_t *sx, float *tok_scale, int *any_lo, const uint8_t *w, uint32_t rows, int *rexp) {
    if (seq == 0 && !(rexp && rows)) return hipSuccess;  // (no tokens: only the rows' exponents, if they are asked for)
    // a token per block; wide activations take more threads per token (two vectors of a thread stay in registers: 4096
    // elements for 256 threads, 8192 for 512, 16384 for 1024; 1024 threads on a row of 4352 leave half of themselves idle: 1024 rows
    // x 4352 with 2048 tokens 52.2 us a call, with 512 threads 47.5, and no less with 16)
    const uint32_t threads = hidden > 8192 ? 1024u : hidden > 4096 ? 512u : 256u;
    const uint32_t row_blocks = rexp ? (rows + threads / 16 - 1) / (threads / 16) : 0;
    hipLaunchKernelGGL(q4k_gemm_prep_kernel, dim3(seq + row_blocks), dim3(threads), 0, s, x, hidden, seq, x_is_bf16, 1, xh, sx, tok_scale, xl,
                       any_lo, w, rows, rexp);
    return hipGetLastError();
}


// K-ranges per output tile (1 = no split), where one 256x128 workgroup runs per CU and the unsplit tiles leave CUs idle.
// In tenths of a microsecond: a super-block of a tile takes 45, a split's
// reduction 50 for the launch and 8 bytes per slab element at 4 TB/s.  The range count with the smallest sum is taken, any
// number up to 32 whose workgroups all run at once (so the slabs stay below 256 tiles, 34 MB).
// The ranges group a result's additions, so they must not change with the number of tokens inside a tile (a token's bits would
// depend on how many others came with it): the last tile counts as five eighths full.
// Fitted on the exact kernel with 170 shapes.  The pair kernel's calls of 324 shapes (300 to 15360 rows, 1024 to 13568 elements, 4 to 440 tokens, every
// range count timed) are 0.4 % above each shape's best on average with the same costs, at the worst 18 % (15360 x 1024 with 4 tokens 14.8 unsplit, 12.6 with
// 4 ranges; 1581 x 6656 with 61 21.7 with 26, 19.6 with 13); with 30, 30 and 3 TB/s, a fit to long prompts, 1.4 %, at the worst 22 % (7412 x 3840 with 440
// 62.6 unsplit, 51.2 with 2).  112 more of 520 to 1300 tokens: 0.4 % (2.1 %), at the worst 7 %.
uint32_t q4k_gemm_splits(uint32_t rows, uint32_t hidden, uint32_t seq, uint32_t cu_count) {
    const uint64_t nsb = hidden / 256, cols = (seq + GN - 1) / GN, tiles = (uint64_t)((rows + GM - 1) / GM) * cols, tokens = cols * GN - GN * 3 / 8;
    uint64_t best = nsb * 45, splits = 1;
    for (uint64_t z = 2; z <= 32 && z <= nsb && tiles * z <= cu_count; z++) {
        const uint64_t per = (nsb + z - 1) / z;
        if ((nsb + per - 1) / per != z) continue;  // (the same ranges as a smaller count)
        const uint64_t cost = per * 45 + 50 + z * rows * tokens * 8 / 400000;
        if (cost < best) { best = cost; splits = z; }
    }
    return (uint32_t)splits;
}

// `rexp` (from q4k_gemm_prep_launch): the rows' scales ride in the f16 weight operand (`with_mins` and `accumulate` are not used);
// without it the weight operand is the exact integer and the rows' f32 scales are applied per super-block
hipError_t q4k_gemm_f16_launch(hipStream_t s, const uint8_t *w, const uint16_t *xh, const uint16_t *sx, const int *rexp, const float *tok_scale,
                               float *out, uint32_t rows, uint32_t hidden, uint32_t seq, int with_mins, int accumulate, uint32_t splits,
                               float *partial, uint32_t cu_count) {
    if (rows == 0 || seq == 0) return hipSuccess;
    const uint32_t nsb = hidden / 256;
    const bool split = splits > 1 && partial;
    const uint32_t per = split ? (nsb + splits - 1) / splits : nsb, z = split ? (nsb + per - 1) / per : 1;
    static std::atomic<bool> attr_set{false};  // dynamic LDS above 64 KB has to be allowed once per process
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void *)q4k_gemm_exact_kernel, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        for (const void *k : {(const void *)q4k_gemm_pair_kernel<2, true>, (const void *)q4k_gemm_pair_kernel<4, true>, (const void *)q4k_gemm_pair_kernel<6, true>,
                              (const void *)q4k_gemm_pair_kernel<8, true>, (const void *)q4k_gemm_pair_kernel<8, false>})
            if (e == hipSuccess) e = hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
        if (e != hipSuccess) return e;
        attr_set = true;
    }
    const dim3 grid((rows + GM - 1) / GM, (seq + GN - 1) / GN, z);
    float *slab = split ? partial : (float *)nullptr;
    // a prompt of one token tile copies, reads and multiplies only its blocks of 32 tokens (3840 x 15360, us per call: 16 tokens 21.9,
    // 77 33.9, 128 40.2)
#define LARQL_PAIR(TB, KS) hipLaunchKernelGGL((q4k_gemm_pair_kernel<TB, KS>), dim3(grid.x * tok_tiles * z), dim3(QTHREADS), Q_LDS_BYTES, s, w, xh, sx, rexp, tok_scale, out, rows, \
                                              hidden, seq, grid.x, tok_tiles, per, slab)
    if (rexp) {
        // 256 tokens per workgroup, a call of full rounds over the chip 1.5 to 1.8 times as long as 128: taken where that saves rounds (us per call, 128 / 256:
        // 15360 x 3840 with 2048 tokens, 4 rounds against 2, 277 / 248; 6790 x 3072 with 1199, 2 against 1, 111 / 88; 13270 x 3840 with 1783, 3 against 2,
        // 212 / 226; 15360 x 3840 with 512, 1 against 1, 75 / 104).  The rule sees a prompt's length in whole tiles of 128 only: a token's bits do not depend on its companions
        const uint32_t tiles_n = grid.x * grid.y, tiles_w = grid.x * ((grid.y + 1) / 2);
        const bool wide = z == 1 && grid.y > 1 && ((uint64_t)((tiles_w + cu_count - 1) / cu_count) * 9 < (uint64_t)((tiles_n + cu_count - 1) / cu_count) * 5);
        const uint32_t tok_tiles = wide ? (grid.y + 1) / 2 : grid.y;
        if (wide) LARQL_PAIR(8, false);
        else if (seq <= 32) LARQL_PAIR(2, true);
        else if (seq <= 64) LARQL_PAIR(4, true);
        else if (seq <= 96) LARQL_PAIR(6, true);
        else LARQL_PAIR(8, true);
    }
#undef LARQL_PAIR
    else
        hipLaunchKernelGGL(q4k_gemm_exact_kernel, grid, dim3(GTHREADS), G_LDS_BYTES, s, w, xh, sx, tok_scale, out, rows, hidden, seq, with_mins,
                           accumulate, per, slab);
    if (split) {
        const size_t n = (size_t)rows * seq;
        // odd rows: with four elements per thread every load crosses lines and there are a quarter of the blocks, one element per thread is
        // four times the instructions (us, one / four: 1581 x 7 of 27 slabs 4.0 / 9.9, 3001 x 200 of 4 4.2 / 5.0, 5001 x 256 of 4 (1.3 M elements) 5.4 / 5.4,
        // 13001 x 120 of 4 (1.6 M) 6.8 / 6.3, 5001 x 400 of 2 (2.0 M) 7.2 / 5.8, 15347 x 256 of 2 (3.9 M) 11.9 / 9.3)
        if ((rows % 4 == 0 && (((uintptr_t)partial | (uintptr_t)out) & 15u) == 0) || n >= 1500000)
            hipLaunchKernelGGL(q4k_gemm_reduce_kernel<4>, dim3((uint32_t)((n + 1023) / 1024)), dim3(256), 0, s, partial, z, tok_scale, out, rows, seq, accumulate);
        else
            hipLaunchKernelGGL(q4k_gemm_reduce_kernel<1>, dim3((uint32_t)((n + 255) / 256)), dim3(256), 0, s, partial, z, tok_scale, out, rows, seq, accumulate);
    }
    return hipGetLastError();
}

}  // namespace larql
