// pm355_route.h — routing of one token to its experts by one wave (moe.hip, and the prologue of the few-token expert products in dense_small.hip).
#pragma once
#include "pm355_dense.h"

#ifdef __HIPCC__
// LDS of one routing wave: s [E] scores, gs [groups]. ids / w receive `top` entries, largest score first (equal scores: lower index first). E <= 1024, groups <= 1024. z(e): the logits.
// Up to 64 experts: a lane keeps its expert's score, the largest one is taken `top` times (a maximum over lanes and a ballot each). More: ranks - every lane counts, for its own experts,
// how many stand in front of them, a trip to LDS for each of the others.
__device__ __forceinline__ void wave_fence() { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); }
// scores of groups that are not among the `keep` best become -1 (s: in LDS, written and fenced)
__device__ __forceinline__ void route_groups(int E, int groups, int keep, float * s, float * gs) {
    const int lane = threadIdx.x & 63, per = E / groups;
    for (int g = lane; g < groups; g += 64) {
        float m = s[g * per];
        for (int i = 1; i < per; ++i) m = fmaxf(m, s[g * per + i]);
        gs[g] = m;
    }
    wave_fence();
    for (int e = lane; e < E; e += 64) {
        const int g = e / per;
        const float m = gs[g];
        int front = 0;
        for (int i = 0; i < groups; ++i) { const float o = gs[i]; front += o > m || (o == m && i < g); }
        if (front >= keep) s[e] = -1.0f;                   // (only this lane reads s[e] before the fence)
    }
    wave_fence();
}
template <typename Z> __device__ __forceinline__ void route_token(Z z, int E, int top, int groups, int keep, float * s, float * gs, int * ids, float * w) {
    const int lane = threadIdx.x & 63;
    float mx = -INFINITY, sum = 0.0f;
    if (E <= 64) {
        const float v = lane < E ? z(lane) : -INFINITY;
        mx = wave_max(v);
        const float e = lane < E ? expf(v - mx) : 0.0f;
        sum = wave_sum(e);
        float m = lane < E ? e / sum : -2.0f;
        if (keep < groups) {
            if (lane < E) s[lane] = m;
            wave_fence();
            route_groups(E, groups, keep, s, gs);
            if (lane < E) m = s[lane];
        }
        int id = 0;
        float wt = 0.0f;                                   // (a row of NaNs has no largest score)
        for (int k = 0; k < top; ++k) {
            const float best = wave_max(m);
            const uint64_t at = __builtin_amdgcn_ballot_w64(lane < E && m == best);      // (lanes without an expert are the largest where no score compares)
            const int first = at ? __builtin_ctzll(at) : 0;
            if (lane == k && at) { id = first; wt = fmaxf(best, 0.0f); }
            if (lane == first) m = -2.0f;
        }
        if (lane < top) { ids[lane] = id; w[lane] = wt; }
        wave_fence();
        return;
    }
    for (int k = lane; k < top; k += 64) { ids[k] = 0; w[k] = 0.0f; }        // (a row of NaNs has no ranks)
    for (int e = lane; e < E; e += 64) { const float v = z(e); s[e] = v; mx = fmaxf(mx, v); }
    mx = wave_max(mx);
    for (int e = lane; e < E; e += 64) { const float v = expf(s[e] - mx); s[e] = v; sum += v; }
    sum = wave_sum(sum);
    for (int e = lane; e < E; e += 64) s[e] /= sum;
    wave_fence();
    if (keep < groups) route_groups(E, groups, keep, s, gs);
    for (int e = lane; e < E; e += 64) {
        const float m = s[e];
        int front = 0;
        for (int i = 0; i < E; ++i) { const float o = s[i]; front += o > m || (o == m && i < e); }
        if (front < top) { ids[front] = e; w[front] = fmaxf(m, 0.0f); }
    }
    wave_fence();
}
#endif
