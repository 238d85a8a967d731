// topk.hip — top-K selection over rows of a score matrix on gfx950.
//
// Two orderings, both restating the reference's selectors:
//   by |score|  — top_k_by_abs, larql-vindex/src/index/compute/gate_knn/mod.rs:50-108
//                 (NaN is an error there: it panics)
//   by value    — top_k_sorted, larql-vindex/src/index/storage/lm_head/knn.rs:315-386
//                 (non-finite scores are skipped)
// Output is sorted best-first.  Where the reference leaves the order of equal
// keys to its heap and an unstable sort, this kernel fixes it: the lower index
// wins.
//
// Each score becomes a 64-bit key (ordered score bits, then ~index), so one
// unsigned compare decides everything and index recovery needs no side array.
// One workgroup serves one row, each thread a contiguous run of indices.
// The K-th largest ordered-score value T is found exactly by a 4-pass radix
// select (8 bits per pass, a 256-bin histogram in LDS per pass, one wavefront
// scanning the bins from the top); scores above T are taken, and of the scores
// equal to T the lowest indices fill the remaining places (ranked by a prefix
// count in index order).  The <= 64 winners are gathered in LDS and one
// wavefront orders them best-first with a bitonic sort done by cross-lane
// shuffles.  Cost is a handful of passes over the row, whatever its order.
// Rows of up to 16384 scores (every gate matrix) are read once: a thread keeps
// its up to 16 ordered scores in registers, and for K up to 256 a bound with at
// least K scores at or above it (the K-th largest maximum of 128 slices of the
// row, of 512 for K above 64) leaves little more than K candidates, which are
// ranked directly; the radix passes remain for rows with more than 1024 of them.
// Longer rows (a vocabulary) are selected in two launches: every chunk of a row
// leaves its own K best keys, sorted, in a workspace, and one workgroup per row
// selects among those.  One workgroup cannot keep enough loads in flight for a
// 262144-score row (405 us on one CU, six passes over 1 MB).
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <atomic>

#include "kernels.h"
#include "wave.h"

namespace larql {

constexpr int kTopkThreads = 1024;
constexpr int kTopkWaves = kTopkThreads / 64;

__device__ __forceinline__ uint64_t shfl_xor_u64(uint64_t v, int mask) {
    uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
    lo = (uint32_t)__shfl_xor((int)lo, mask, 64);
    hi = (uint32_t)__shfl_xor((int)hi, mask, 64);
    return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ uint64_t shfl_u64(uint64_t v, int src) {
    uint32_t lo = (uint32_t)v, hi = (uint32_t)(v >> 32);
    lo = (uint32_t)__shfl((int)lo, src, 64);
    hi = (uint32_t)__shfl((int)hi, src, 64);
    return ((uint64_t)hi << 32) | lo;
}

// bitonic merge of a bitonic 64-sequence into descending order
__device__ __forceinline__ uint64_t merge_desc(uint64_t key, uint32_t lane) {
#pragma unroll
    for (int j = 32; j > 0; j >>= 1) {
        const uint64_t other = shfl_xor_u64(key, j);
        const bool lower = (lane & j) == 0;
        key = lower ? (key > other ? key : other) : (key < other ? key : other);
    }
    return key;
}

// full bitonic sort of 64 keys, descending by lane
__device__ __forceinline__ uint64_t sort_desc(uint64_t key, uint32_t lane) {
#pragma unroll
    for (int size = 2; size <= 64; size <<= 1) {
        const bool desc_block = (size == 64) || ((lane & size) == 0);
#pragma unroll
        for (int j = size >> 1; j > 0; j >>= 1) {
            const uint64_t other = shfl_xor_u64(key, j);
            const bool lower = (lane & j) == 0;
            const bool take_max = (lower == desc_block);
            key = take_max ? (key > other ? key : other) : (key < other ? key : other);
        }
    }
    return key;
}

template <bool BY_ABS>
__device__ __forceinline__ uint64_t make_key(float s, uint32_t idx, int *nan_flag) {
    const uint32_t bits = __builtin_bit_cast(uint32_t, s);
    uint32_t ord;
    if (BY_ABS) {
        ord = bits & 0x7FFFFFFFu;
        if (ord > 0x7F800000u) { if (nan_flag) atomicOr(nan_flag, 1); ord = 0; }
        ord += 1;  // keep every real score above the padding key 0
    } else {
        if ((bits & 0x7F800000u) == 0x7F800000u) return 0;  // inf / NaN are skipped
        ord = (bits & 0x80000000u) ? ~bits : (bits | 0x80000000u);
    }
    return ((uint64_t)ord << 32) | (uint32_t)(~idx);
}

constexpr int kTopkCached = 16;  // rounds of 64 scores per wavefront held in registers
constexpr int kTopkCandidates = 1024;  // of the short way
// Winners that the short way bounds.  Radix passes / short way, us per gate-KNN call over 10240 features of 256: K = 65 22.7 / 11.7,
// 200 24.9 / 12.9, 256 24.8 / 13.8, 257 27.5 / 14.3, 300 27.5 / 16.0, 400 27.6 / 23.3, 512 27.7 / 32.7; over 4096: 300 20.4 / 13.8, 400 20.5 /
// 20.8.  With K near the 512 slices the bound falls to the smallest maximum and the candidates overflow, so the gain ends between
// 300 and 400; 256 lies on its safe side.  A row of equal scores pays for the attempt: K = 200 52.6 / 54.6.
constexpr uint32_t kTopkShortK = 256;

// What a workgroup selects from: `n` scores of a row, cut into chunks of `chunk` (chunk == n: the whole row), or — KEYS_IN —
// the row's `n` keys that the chunks' workgroups left.  A chunk's workgroup leaves keys (KEYS_OUT): its K best, best
// first, zeros behind them where it has fewer.
struct TopkArgs {
    const float *scores;       // [batch, scores_n]
    const uint64_t *keys_in;   // KEYS_IN: [batch, n]
    uint64_t *keys_out;        // KEYS_OUT: [batch, chunks, k]
    uint32_t *idx_out;
    float *val_out;
    uint32_t *count_out;
    int *nan_flag;
    uint32_t scores_n, n, chunk, k, cap;
    uint32_t by_value;         // (a score then comes out of its key)
};

// ROUNDS: scores per thread held in registers (0: streamed on every pass).
// LARGE (K above 64, up to kTopkMaxK): the selection is the same radix select; the winners are gathered into a
// power-of-two array in dynamic LDS (`cap` keys, zero-padded) and ordered by a bitonic sort of the whole workgroup.
// KEYS_IN: equal scores stand in index order in the workspace (chunks in index order, a chunk's keys best first, the
// lower index before the higher), so the ranking of ties by position serves there too.
// (80 scalar registers: with the 96 the compiler would take, a second 16-wavefront workgroup was not placed on a CU
// until half of the first one's wavefronts had left — more rows than CUs then ran in two rounds)
// The arguments on the way to the first score are plain scalars, so that they are in registers when a wavefront starts; read from
// the block they were one more trip to memory (a gate-KNN over 10240 x 2560 f16 features 16.4 -> 15.85 us).
template <bool BY_ABS, int ROUNDS, bool LARGE, bool KEYS_IN, bool KEYS_OUT>
__global__ void __launch_bounds__(kTopkThreads) __attribute__((amdgpu_num_sgpr(80))) topk_kernel(
    const void *src, int *const nan_flag, uint32_t scores_n, uint32_t row_n, uint32_t chunk, uint32_t k,
    uint32_t cap,  // (in registers when the wavefront starts; src: the scores, or the keys)
    const TopkArgs A) {
    constexpr bool CACHED = ROUNDS > 0, SHORT_WAY = CACHED;
    constexpr int GROUPS = LARGE ? 512 : 128, PL = GROUPS / 64;  // slices of the row that bound the K-th score; maxima per lane
    extern __shared__ __attribute__((aligned(16))) uint64_t big[];  // LARGE: cap keys
    __shared__ uint32_t hist[256];
    __shared__ uint32_t wave_ties[kTopkWaves];
    __shared__ uint64_t winners[64];
    __shared__ uint32_t sh_prefix, sh_need, sh_nwin, sh_ncand;
    __shared__ uint32_t group_max[SHORT_WAY ? GROUPS : 1];
    __shared__ __attribute__((aligned(16))) uint64_t cand[SHORT_WAY ? kTopkCandidates : 1];
    __shared__ float cand_score[SHORT_WAY && BY_ABS && !KEYS_OUT ? kTopkCandidates : 1];  // (by |score| a key has lost the sign)
    const uint32_t row = blockIdx.y, tid = threadIdx.x, lane = tid & 63u, wave = tid >> 6;
    const uint32_t first = blockIdx.x * chunk, n = min(chunk, row_n - first);
    const float *const srow = (KEYS_IN ? A.scores : (const float *)src) + (size_t)row * scores_n;
    const float *const s = srow + first;
    const uint64_t *const keys = KEYS_IN ? (const uint64_t *)src + (size_t)row * row_n + first : nullptr;
    uint64_t *const kout = KEYS_OUT ? A.keys_out + ((size_t)row * gridDim.x + blockIdx.x) * k : nullptr;
    // wavefront w owns the contiguous indices [w0, w1), 64 at a time (lane = index within the 64)
    const uint32_t perw = ((n + kTopkWaves * 64 - 1) / (kTopkWaves * 64)) * 64;
    const uint32_t w0 = min(n, wave * perw), w1 = min(n, w0 + perw);

    // winner number `rank` of the row (or of the chunk)
    auto put = [&](uint32_t rank, uint64_t key, float score) {
        if (KEYS_OUT) {
            kout[rank] = key;
        } else {
            A.idx_out[(size_t)row * k + rank] = ~(uint32_t)key;
            A.val_out[(size_t)row * k + rank] = score;
        }
    };
    auto emit = [&](uint32_t rank, uint64_t key) {
        const uint32_t ord = (uint32_t)(key >> 32);
        if (KEYS_OUT) put(rank, key, 0.f);
        else if (A.by_value) put(rank, key, __builtin_bit_cast(float, (ord & 0x80000000u) ? ord & 0x7FFFFFFFu : ~ord));
        else put(rank, key, srow[~(uint32_t)key]);
    };
    // index i as a key: its ordered score (0: nothing there) and the low word, from the register copy or from memory
    uint32_t cache[CACHED ? ROUNDS : 1], low[KEYS_IN && CACHED ? ROUNDS : 1];
    float raw[CACHED ? ROUNDS : 1];
    if (CACHED && KEYS_IN) {
        uint64_t raw[CACHED ? ROUNDS : 1];
#pragma unroll
        for (int it = 0; it < ROUNDS; it++) raw[it] = keys[min(w0 + it * 64 + lane, n - 1)];
#pragma unroll
        for (int it = 0; it < ROUNDS; it++) {
            cache[it] = w0 + it * 64 + lane < w1 ? (uint32_t)(raw[it] >> 32) : 0u;
            low[it] = (uint32_t)raw[it];
        }
    } else if (CACHED) {
        // every load leaves before the first score is looked at (a load inside a condition is waited for where it
        // stands: sixteen round trips instead of one); an index past the wavefront's range reads the row's last score
#pragma unroll
        for (int it = 0; it < ROUNDS; it++) raw[it] = s[min(w0 + it * 64 + lane, n - 1)];
#pragma unroll
        for (int it = 0; it < ROUNDS; it++) {
            const uint32_t i = w0 + it * 64 + lane;
            cache[it] = i < w1 ? (uint32_t)(make_key<BY_ABS>(raw[it], i, nan_flag) >> 32) : 0u;
        }
    }
    auto low_word = [&](int it) -> uint32_t { return KEYS_IN ? low[KEYS_IN && CACHED ? it : 0] : ~(first + w0 + it * 64 + lane); };
    // f(ord, low) for every index of this wavefront, 64 at a time, all lanes taking part in every round
    auto for_each = [&](auto &&f, int *flag) {
        if (CACHED) {
#pragma unroll
            for (int it = 0; it < ROUNDS; it++) f(cache[it], low_word(it));
        } else {
            for (uint32_t base = w0; base < w1; base += 64) {
                const uint32_t i = base + lane;
                if (KEYS_IN) {
                    const uint64_t key = i < w1 ? keys[i] : 0ull;
                    f((uint32_t)(key >> 32), (uint32_t)key);
                } else {
                    f(i < w1 ? (uint32_t)(make_key<BY_ABS>(s[i], i, flag) >> 32) : 0u, ~(first + i));
                }
            }
        }
    };

    if (tid < 64) winners[tid] = 0;
    if (tid == 0) { sh_prefix = 0; sh_need = k; sh_nwin = 0; sh_ncand = 0; }
    if (SHORT_WAY && k <= kTopkShortK) {
        // ---- short way for a row held in registers.  Every group of neighbouring lanes owns a slice of the row; at least k
        //      scores lie at or above L, the k-th largest of the group maxima (one per group): little more than k of a typical
        //      row (128 groups, k = 64: ~90; the smallest of 64 maxima, the bound before, left ~300-500, and ranking them was a
        //      third of the kernel).  Those are collected, and each one's place in the output is the number of candidates
        //      above it.  A row whose candidates do not fit (many equal scores, too few valid ones) takes the radix passes below.
        //      gate-KNN calls over 10240 features, before / now: K = 64 13.9 / 9.9 us, K = 8 13.8 / 9.5, K = 256 (radix passes
        //      before) 25.2 / 13.8 ----
        uint32_t gmax = 0;
#pragma unroll
        for (int it = 0; it < ROUNDS; it++) gmax = max(gmax, cache[it]);
        for (uint32_t i = tid; i < (uint32_t)kTopkCandidates; i += kTopkThreads) cand[i] = 0;
        if (KEYS_IN) {
            // a chunk's keys stand best first: slices of every eighth (32nd) lane each hold one of the best of every chunk
            // (slices of neighbours would leave the worst of a chunk to themselves and bound nothing)
#pragma unroll
            for (int o = 64 / (1024 / GROUPS); o < 64; o <<= 1) gmax = max(gmax, (uint32_t)__shfl_xor((int)gmax, o, 64));
            if (lane < GROUPS / kTopkWaves) group_max[wave * (GROUPS / kTopkWaves) + lane] = gmax;
        } else {
            // (reductions by DPP row operations: a few cycles each, where a cross-lane shuffle costs an LDS round trip)
            gmax = max(gmax, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)gmax, 0xB1, 0xF, 0xF, true));       // quad_perm [1,0,3,2]
            if (!LARGE) {
                gmax = max(gmax, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)gmax, 0x4E, 0xF, 0xF, true));   // quad_perm [2,3,0,1]
                gmax = max(gmax, (uint32_t)__builtin_amdgcn_update_dpp(0, (int)gmax, 0x141, 0xF, 0xF, true));  // row_half_mirror
            }
            if ((lane & (1024 / GROUPS - 1)) == 0) group_max[tid / (1024 / GROUPS)] = gmax;
        }
        __syncthreads();
        // The k-th largest maximum, every wavefront for itself: from the highest bit in which the largest and the smallest differ,
        // a bit of L is set where k maxima still lie at or above it.  Fourteen bits: a bound may lie lower than the exact one.
        uint32_t gm[PL], top = 0, bottom = ~0u;
#pragma unroll
        for (int q = 0; q < PL; q++) {
            gm[q] = group_max[q * 64 + lane];
            top = max(top, gm[q]);
            bottom = min(bottom, gm[q]);
        }
        top = wave_max_u32(top);
        bottom = ~wave_max_u32(~bottom);
        uint32_t L = bottom;
        if (top != bottom) {
            const int high = 31 - __builtin_clz(top ^ bottom);
            L = top & ~((2u << high) - 1u);  // (bits that all maxima share; high = 31: none)
            for (int b = high; b >= 0 && b > high - 14; b--) {
                const uint32_t trial = L | (1u << b);
                uint32_t have = 0;
#pragma unroll
                for (int q = 0; q < PL; q++) have += (uint32_t)__popcll(__ballot(gm[q] >= trial));
                if (have >= k) L = trial;
            }
        }
        // (L = 0: fewer than k groups hold a score)
        if (L != 0) {
            // a wavefront reserves room for all its candidates at once, then places them round by round
            uint32_t mine = 0;
#pragma unroll
            for (int it = 0; it < ROUNDS; it++) mine += (uint32_t)__popcll(__ballot(cache[it] >= L));
            uint32_t base = 0;
            if (lane == 0 && mine) base = atomicAdd(&sh_ncand, mine);
            base = (uint32_t)__builtin_amdgcn_readfirstlane((int)base);
#pragma unroll
            for (int it = 0; it < ROUNDS; it++) {
                const bool c = cache[it] >= L;
                const uint64_t m = __ballot(c);
                const uint32_t pos = base + (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
                if (c && pos < (uint32_t)kTopkCandidates) {
                    cand[pos] = ((uint64_t)cache[it] << 32) | low_word(it);
                    if (BY_ABS && !KEYS_OUT && !KEYS_IN) cand_score[pos] = raw[it];
                }
                base += (uint32_t)__popcll(m);
            }
            __syncthreads();
            const uint32_t nc = sh_ncand;
            if (nc <= (uint32_t)kTopkCandidates) {  // (uniform over the workgroup)
                // A candidate's rank = the candidates above it: eight neighbouring lanes each count an eighth of the list, read two
                // keys at a time (zero keys, below every real one, stand behind it).
                typedef uint64_t u64x2 __attribute__((ext_vector_type(2)));
                const u64x2 *c2 = reinterpret_cast<const u64x2 *>(cand);
                const uint32_t pairs = (nc + 15) / 16;  // of an eighth
                for (uint32_t c0 = 0; c0 < nc; c0 += kTopkThreads / 8) {
                    const uint32_t ci = c0 + (tid >> 3);
                    const uint64_t key = cand[min(ci, nc - 1)];
                    uint32_t rank = 0;
#pragma unroll 2
                    for (uint32_t j = 0; j < pairs; j++) {
                        const u64x2 a = c2[j * 8 + (tid & 7u)];
                        rank += (a.x > key ? 1u : 0u) + (a.y > key ? 1u : 0u);
                    }
                    rank += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)rank, 0xB1, 0xF, 0xF, true);   // quad_perm [1,0,3,2]
                    rank += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)rank, 0x4E, 0xF, 0xF, true);   // quad_perm [2,3,0,1]
                    rank += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)rank, 0x141, 0xF, 0xF, true);  // row_half_mirror
                    if ((tid & 7u) == 0 && ci < nc && rank < k) {
                        if (BY_ABS && !KEYS_OUT && !KEYS_IN) put(rank, key, cand_score[ci]);
                        else emit(rank, key);
                    }
                }
                if (!KEYS_OUT && tid == 0) A.count_out[row] = min(k, nc);  // (nc >= k: a chunk leaves k keys)
                return;
            }
        }
        __syncthreads();
    }
    if (LARGE)
        for (uint32_t i = tid; i < cap; i += kTopkThreads) big[i] = 0;
    // ---- radix select of the k-th largest ordered score: 8 bits per pass, top byte first ----
    for (int pass = 0; pass < 4; pass++) {
        const int sh = 24 - 8 * pass;
        if (tid < 256) hist[tid] = 0;
        __syncthreads();
        const uint32_t prefix = sh_prefix;
        for_each([&](uint32_t ord, uint32_t) {
            // 64-bit shift: the first pass compares nothing (shift by 32)
            if (ord != 0 && ((uint64_t)ord >> (sh + 8)) == ((uint64_t)prefix >> (sh + 8))) atomicAdd(&hist[(ord >> sh) & 255u], 1u);
        }, pass == 0 ? nan_flag : nullptr);
        __syncthreads();
        if (wave == 0) {
            // lane l holds bins 255-4l .. 252-4l (descending); find the bin where the running count reaches `need`
            const uint32_t need = sh_need;
            const uint32_t b0 = 255u - 4u * lane;
            const uint32_t c0 = hist[b0], c1 = hist[b0 - 1], c2 = hist[b0 - 2], c3 = hist[b0 - 3];
            const uint32_t mine = c0 + c1 + c2 + c3;
            uint32_t incl = mine;  // inclusive scan over lanes (bins in descending order)
#pragma unroll
            for (int o = 1; o < 64; o <<= 1) {
                const uint32_t t = (uint32_t)__shfl_up((int)incl, o, 64);
                if (lane >= (uint32_t)o) incl += t;
            }
            const uint32_t before = incl - mine;
            const bool here = before < need && incl >= need;
            if (here) {
                uint32_t acc = before, bin = b0, above = before;
                const uint32_t c[4] = {c0, c1, c2, c3};
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    if (acc < need && acc + c[q] >= need) { bin = b0 - q; above = acc; }
                    acc += c[q];
                }
                sh_prefix = prefix | (bin << sh);
                sh_need = need - above;  // still to find inside the chosen bin
            }
            // fewer than `need` valid scores in total: nobody is `here`; prefix stays and everything valid is taken
            const uint32_t total = (uint32_t)__shfl((int)incl, 63, 64);
            if (lane == 0 && total < need) { sh_need = 0xFFFFFFFFu; }
        }
        __syncthreads();
        if (sh_need == 0xFFFFFFFFu) break;
    }
    const bool take_all = sh_need == 0xFFFFFFFFu;
    const uint32_t T = take_all ? 0u : sh_prefix;     // scores with ord > T are in
    const uint32_t r = take_all ? 0xFFFFFFFFu : sh_need;  // this many of the scores with ord == T, lowest indices first
    // ---- rank the ties in index order: per-wavefront counts, then ballots inside the wavefront ----
    uint32_t my_ties = 0;
    if (!take_all)
        for_each([&](uint32_t ord, uint32_t) { my_ties += (uint32_t)__popcll(__ballot(ord != 0 && ord == T)); }, nullptr);
    if (lane == 0) wave_ties[wave] = my_ties;
    __syncthreads();
    uint32_t tie_rank = 0;  // ties at lower indices than this wavefront's current 64
    for (uint32_t w = 0; w < wave; w++) tie_rank += wave_ties[w];
    // ---- gather the winners ----
    for_each([&](uint32_t ord, uint32_t lo) {
        const uint64_t key = ((uint64_t)ord << 32) | lo;
        bool in = ord != 0 && ord > T;
        if (!take_all) {
            const bool tie = ord != 0 && ord == T;
            const uint64_t m = __ballot(tie);
            const uint32_t before = (uint32_t)__popcll(m & ((1ull << lane) - 1ull));
            if (tie) in = tie_rank + before < r;
            tie_rank += (uint32_t)__popcll(m);
        }
        if (in) {
            const uint32_t pos = atomicAdd(&sh_nwin, 1u);
            if (LARGE) { if (pos < cap) big[pos] = key; }
            else if (pos < 64) winners[pos] = key;
        }
    }, nullptr);
    __syncthreads();
    if (LARGE) {
        // bitonic sort of the cap keys, descending (the padding keys 0 sink to the end): log2(cap)*(log2(cap)+1)/2 rounds of
        // cap/2 compare-exchanges; thread t's pair in a round with distance j is (i, i+j), i = t with a 0 inserted at bit log2(j)
        for (uint32_t size = 2; size <= cap; size <<= 1) {
            for (uint32_t jd = size >> 1; jd > 0; jd >>= 1) {
                for (uint32_t t = tid; t < (cap >> 1); t += kTopkThreads) {
                    const uint32_t lo = 2 * t - (t & (jd - 1)), hi = lo + jd;
                    const bool desc = (lo & size) == 0;
                    const uint64_t a = big[lo], b = big[hi];
                    if ((a < b) == desc) { big[lo] = b; big[hi] = a; }
                }
                __syncthreads();
            }
        }
        const uint32_t nw = min(min(sh_nwin, cap), k);
        for (uint32_t i = tid; i < nw; i += kTopkThreads) emit(i, big[i]);
        if (KEYS_OUT) for (uint32_t i = nw + tid; i < k; i += kTopkThreads) kout[i] = 0ull;
        else if (tid == 0) A.count_out[row] = nw;
        return;
    }
    if (wave == 0) {
        const uint64_t top = sort_desc(winners[lane], lane);
        const bool valid = top != 0 && lane < k;
        if (KEYS_OUT ? lane < k : valid) emit(lane, top);
        const uint64_t mask = __ballot(valid);
        if (!KEYS_OUT && lane == 0) A.count_out[row] = (uint32_t)__popcll(mask);
    }
}

// How a row of a batch is cut.  A row that one workgroup can hold in registers is not: two launches cost 4 us more than one.
// Above that, K <= 256 (the short way) takes chunks of 4096 (four scores a thread; of 16384 where the chunks' winners would not fit
// the merging workgroup's registers): streamed or cut at 16384 / cut at 4096, us per lm_head call, K = 200:
// 16400 scores 105 / 60, 32768 103 / 56, 262144 116 / 68; 18000 scores, 1 / 100 / 1000 rows 45 / 21, 63 / 42, 246 / 216.
// A larger K takes chunks of 16384 where that is faster than streaming the row: a second launch and a second ordering of K
// winners against ~1.7 us per thousand scores beyond the first 16384 that one workgroup would walk again and again.  The two
// meet at 17408 + 5 K scores (one row, streamed / cut, us: 20000, 500 51.0 / 51.6; 20000, 1000 55.4 / 60.8; 24000, 1000 61.7 / 61.0;
// 24000, 2000 68.2 / 75.9; 32768, 2000 84.4 / 76.8; the same within 5 % for 100 or 1000 rows).
// Above K = 2048 the two orderings (a bitonic sort of 4096 keys is 35 us) take four chunks to pay for (32768, 4096 101.6 / 115.7;
// 65536, 4096 157.1 / 127.9), and do not once the rows fill the chip by themselves (65536, 4096: 100 rows 315 / 300, 300 rows 722 / 731,
// 1000 rows 2044 / 2242).
static uint32_t topk_chunk(uint32_t batch, uint32_t n, uint32_t k) {
    constexpr uint32_t held = kTopkThreads * kTopkCached, small = held / 4;
    if (n <= held) return n;
    if (k <= kTopkShortK) {
        for (uint32_t chunk : {small, held})
            if ((uint64_t)((n + chunk - 1) / chunk) * k <= held) return chunk;
        if (k <= 64) return n;
    }
    if (n > 0x7FFFFFFFu || k > held / 4) return n;
    const bool cut = k <= held / 8 ? n >= held + 1024 + 5 * k : n > 3 * held && batch <= 128;
    return cut ? held : n;
}

// Bytes of workspace that one row's chunks leave their keys in (0: the row is not cut).
static size_t topk_row_bytes(uint32_t n, uint32_t k, uint32_t chunk) {
    return chunk == n ? 0 : (size_t)((n + chunk - 1) / chunk) * k * sizeof(uint64_t);
}

// The workspace is bounded: a batch that needs more is selected in slices of rows (512 at least where K <= 64, and a multiple
// of 256 where it holds so many: the merging launch of a slice is a workgroup per row), and a row that alone needs more is
// streamed.
constexpr size_t kTopkWorkspaceMax = 64u << 20;
size_t topk_workspace_bytes(uint32_t batch, uint32_t n, uint32_t k) {
    const size_t row = topk_row_bytes(n, k, topk_chunk(batch, n, k));
    if (row == 0 || row > kTopkWorkspaceMax) return 0;
    size_t rows = kTopkWorkspaceMax / row;
    if (rows >= batch) rows = batch;
    else if (rows > 256) rows -= rows % 256;
    return row * rows;
}

// one launch over `batch` rows of `chunks` chunks each
template <bool BY_ABS, int ROUNDS, bool LARGE, bool KEYS_IN, bool KEYS_OUT>
static hipError_t topk_stage(hipStream_t stream, TopkArgs A, uint32_t chunks, uint32_t batch) {
    size_t lds = 0;
    if (LARGE) {
        // more than 64 winners: ordered in LDS (room for the next power of two above min(k, n) keys)
        A.cap = 128;
        while (A.cap < A.k && A.cap < A.n) A.cap <<= 1;
        lds = (size_t)A.cap * sizeof(uint64_t);
        static std::atomic<bool> allowed{false};
        if (!allowed) {  // dynamic LDS above 64 KB has to be allowed once per process
            hipError_t e = hipFuncSetAttribute((const void *)topk_kernel<BY_ABS, ROUNDS, LARGE, KEYS_IN, KEYS_OUT>,
                                               hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kTopkMaxK * sizeof(uint64_t)));
            if (e != hipSuccess) return e;
            allowed = true;
        }
    }
    hipLaunchKernelGGL((topk_kernel<BY_ABS, ROUNDS, LARGE, KEYS_IN, KEYS_OUT>), dim3(chunks, batch), dim3(kTopkThreads), lds, stream,
                       KEYS_IN ? (const void *)A.keys_in : (const void *)A.scores, A.nan_flag, A.scores_n, A.n, A.chunk, A.k, A.cap, A);
    return hipGetLastError();
}

// (workspace: room for the keys of all `batch` rows' chunks, or null: the rows are not cut)
template <bool BY_ABS>
static hipError_t topk_rows(hipStream_t stream, TopkArgs A, uint32_t batch, uint32_t chunk, void *workspace) {
    const bool large = A.k > 64 && A.n > 64;
    A.chunk = A.n;
    if (workspace) {
        const uint32_t chunks = (A.n + chunk - 1) / chunk;
        A.chunk = chunk;
        A.keys_out = (uint64_t *)workspace;
        hipError_t e = large ? (chunk <= kTopkThreads * kTopkCached / 4 ? topk_stage<BY_ABS, kTopkCached / 4, true, false, true>(stream, A, chunks, batch)
                                                                         : topk_stage<BY_ABS, kTopkCached, true, false, true>(stream, A, chunks, batch))
                       : chunk <= kTopkThreads * kTopkCached / 4 ? topk_stage<BY_ABS, kTopkCached / 4, false, false, true>(stream, A, chunks, batch)
                                                                 : topk_stage<BY_ABS, kTopkCached, false, false, true>(stream, A, chunks, batch);
        if (e != hipSuccess) return e;
        A.keys_in = A.keys_out;
        A.n = A.chunk = chunks * A.k;
        if (A.n > kTopkThreads * kTopkCached) return topk_stage<false, 0, true, true, false>(stream, A, 1, batch);
        if (A.n <= kTopkThreads * kTopkCached / 4)
            return large ? topk_stage<false, kTopkCached / 4, true, true, false>(stream, A, 1, batch)
                         : topk_stage<false, kTopkCached / 4, false, true, false>(stream, A, 1, batch);
        return large ? topk_stage<false, kTopkCached, true, true, false>(stream, A, 1, batch)
                     : topk_stage<false, kTopkCached, false, true, false>(stream, A, 1, batch);
    }
    const bool cached = A.n <= (uint32_t)(kTopkThreads * kTopkCached);
    if (large) {
        // (the radix passes walk every round of the registers, empty or not: rows of up to 4096 take four instead of sixteen —
        // a KNN call over 1254 features, K = 256: 20.8 us with sixteen, 17.9 with four, 19.3 streamed from memory)
        if (A.n <= (uint32_t)(kTopkThreads * kTopkCached / 4)) return topk_stage<BY_ABS, kTopkCached / 4, true, false, false>(stream, A, 1, batch);
        return cached ? topk_stage<BY_ABS, kTopkCached, true, false, false>(stream, A, 1, batch) : topk_stage<BY_ABS, 0, true, false, false>(stream, A, 1, batch);
    }
    return cached ? topk_stage<BY_ABS, kTopkCached, false, false, false>(stream, A, 1, batch) : topk_stage<BY_ABS, 0, false, false, false>(stream, A, 1, batch);
}

hipError_t topk_launch(hipStream_t stream, const float *scores, uint32_t batch, uint32_t n, uint32_t k, bool by_abs,
                       uint32_t *idx_out, float *val_out, uint32_t *count_out, int *nan_flag, void *workspace, size_t workspace_bytes) {
    if (k > kTopkMaxK) return hipErrorInvalidValue;
    TopkArgs A = {};
    A.scores_n = A.n = n; A.k = k; A.nan_flag = nan_flag; A.by_value = by_abs ? 0u : 1u;
    const size_t need = topk_workspace_bytes(batch, n, k);
    if (need == 0 || workspace_bytes < need) workspace = nullptr;
    const uint32_t chunk = topk_chunk(batch, n, k);
    const uint32_t slice = workspace ? std::min<uint32_t>(65535u, (uint32_t)(need / topk_row_bytes(n, k, chunk))) : 65535u;  // (rows are the grid's y)
    for (uint32_t b0 = 0; b0 < batch; b0 += slice) {
        const uint32_t rows = std::min(slice, batch - b0);
        A.scores = scores + (size_t)b0 * n;
        A.idx_out = idx_out + (size_t)b0 * k; A.val_out = val_out + (size_t)b0 * k; A.count_out = count_out + b0;
        const hipError_t e = by_abs ? topk_rows<true>(stream, A, rows, chunk, workspace) : topk_rows<false>(stream, A, rows, chunk, workspace);
        if (e != hipSuccess) return e;
        if (rows == batch - b0) break;  // (b0 + slice may pass 2^32)
    }
    return hipSuccess;
}

}  // namespace larql
