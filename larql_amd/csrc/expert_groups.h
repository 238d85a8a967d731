// expert_groups.h — the slots (token, rank) of a call grouped by the expert they chose, worked out by every workgroup for itself
// from the router's choice: no job table, no planning launch.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "mx4.h"
#include "wave.h"

namespace larql {

// LDS of a workgroup: slots per expert, groups of the experts before each ([n_experts]: all groups), the slots' experts
struct ExpertGroups {
    uint32_t *cnt, *before;
    uint16_t *ex;
};

// Counts the slots per expert and the groups of up to TG slots before each expert; an id outside the bank belongs to nobody.
// The whole workgroup calls it; it ends with a barrier.
template <int TG>
__device__ __forceinline__ void expert_groups_count(const ExpertGroups &G, const uint32_t *experts, uint32_t slots, uint32_t nE, uint32_t tid, uint32_t lane, uint32_t wv) {
    uint32_t e0 = tid < slots ? ((const GLOBAL_AS uint32_t *)experts)[tid] : 0u;  // (on its way while the counters are cleared)
    for (uint32_t e = tid; e < nE; e += blockDim.x) G.cnt[e] = 0;
    __syncthreads();
    for (uint32_t s = tid; s < slots; s += blockDim.x) {
        const uint32_t e = s == tid ? e0 : ((const GLOBAL_AS uint32_t *)experts)[s];
        G.ex[s] = e < nE ? (uint16_t)e : (uint16_t)0xFFFFu;
        if (e < nE) atomicAdd(&G.cnt[e], 1u);
    }
    __syncthreads();
    if (wv == 0) {
        uint32_t run = 0;
        for (uint32_t base = 0; base < nE; base += 64) {
            const uint32_t e = base + lane, g = e < nE ? (G.cnt[e] + TG - 1) / TG : 0u, incl = wave_inclusive_sum(g);
            if (e < nE) G.before[e] = run + incl - g;
            run += (uint32_t)__builtin_amdgcn_readlane((int)incl, 63);
        }
        if (lane == 0) G.before[nE] = run;
    }
    __syncthreads();
}

// Share `share` of `grid` even ones of `units`: [v, v_end).  One 32-bit division, and what leads to the experts' ids in preloaded
// arguments: two 64-bit divisions and the argument block lay before a launch's first tile (MXFP4 block of 128 tokens 160.5 -> 158.6 us,
// two launches; a k-quant layer of 16 tokens 88.3 -> 87.2).
__device__ __forceinline__ void expert_group_share(uint32_t units, uint32_t share, uint32_t grid, uint32_t &v, uint32_t &v_end) {
    const uint32_t each = units / grid, rest = units - each * grid;
    v = each * share + min(share, rest);
    v_end = v + each + (share < rest ? 1u : 0u);
}

// the expert of group gi
__device__ __forceinline__ uint32_t expert_of_group(const ExpertGroups &G, uint32_t nE, uint32_t gi, uint32_t lane) {
    uint32_t e = 0;
    for (uint32_t base = 0; base < nE; base += 64) {
        const uint32_t q = base + lane;
        const uint64_t m = __ballot(q < nE && G.before[min(q, nE)] <= gi && gi < G.before[min(q + 1, nE)]);
        if (m) { e = base + (uint32_t)__builtin_ctzll(m); break; }
    }
    return __builtin_amdgcn_readfirstlane(e);
}

// The slots of rank lo .. lo + TG - 1 among expert e's, in slot order, to `list`; every wavefront may find them for itself and
// write the same list
template <int TG>
__device__ __forceinline__ void expert_group_slots(const ExpertGroups &G, uint32_t slots, uint32_t e, uint32_t lo, uint16_t *list, uint32_t lane) {
    uint32_t run = 0;
    for (uint32_t base = 0; base < slots; base += 64) {
        const bool is = base + lane < slots && G.ex[min(base + lane, slots - 1)] == e;
        const uint64_t m = __ballot(is);
        const uint32_t rank = run + (uint32_t)__popcll(m & ((1ull << lane) - 1ull)) - lo;
        if (is && rank < (uint32_t)TG) list[rank] = (uint16_t)(base + lane);
        run += (uint32_t)__popcll(m);
        if (run >= lo + TG) break;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

}  // namespace larql
