// What the kernels of routed experts share: the gated unit, and the walk over units of weight rows and pairs.
#pragma once
#include "common.h"

__device__ __forceinline__ float rx_glu(float g, float u, float limit, float alpha) {
    if (alpha > 0.f) {
        g = fminf(g, limit);
        u = fminf(fmaxf(u, -limit), limit);
        return g / (1.0f + expf(-alpha * g)) * (u + 1.0f);
    }
    return g / (1.0f + expf(-g)) * u;
}

// By one wave: put(e, the sum of of(..) over the experts before e) for e < E; returns the sum over all.
template <typename Of, typename Put>
__device__ __forceinline__ int rx_sums_before(int E, int lane, Of of, Put put) {
    int run = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
        const int e = e0 + lane, mine = e < E ? of(e) : 0;
        int sum = mine;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1)
            if (o < E) {                                      // uniform
                const int v = __shfl_up(sum, o, 64);
                if (lane >= o) sum += v;
            }
        if (e < E) put(e, run + sum - mine);
        run += __shfl(sum, min(63, E - 1 - e0), 64);
    }
    return run;
}

// A unit is a run of output rows of one expert against up to XR of its pairs; the units are numbered expert by expert (experts
// without pairs have none), rows by rows, and for the same rows group by group of pairs.  In LDS: firstL[e] the first pair of expert
// e in the experts' order (firstL[E + 1] = firstL[E]), cum[e] the units before expert e; `tiles` runs of rows an expert.
struct RxUnit { int e, t, j, p0, np; };       // expert, unit of its rows, group of its pairs: the group's first pair and size

template <int XR>
__device__ __forceinline__ RxUnit rx_unit_at(int u, const int* cum, const int* firstL, int E, int tiles) {
    int lo = 0, hi = E;                                       // the expert with cum[e] <= u < cum[e + 1]
    while (hi - lo > 1) {
        const int mid = (lo + hi) >> 1;
        if (cum[mid] <= u) lo = mid; else hi = mid;
    }
    RxUnit r;
    r.e = lo;
    const int n = firstL[lo + 1] - firstL[lo], groups = (n + XR - 1) / XR, at = u - cum[lo];
    r.t = at / groups;
    r.j = at - r.t * groups;
    r.p0 = firstL[lo] + r.j * XR;
    r.np = min(XR, firstL[lo + 1] - r.p0);
    r.e = __builtin_amdgcn_readfirstlane(r.e);
    r.t = __builtin_amdgcn_readfirstlane(r.t);
    r.j = __builtin_amdgcn_readfirstlane(r.j);
    r.p0 = __builtin_amdgcn_readfirstlane(r.p0);
    r.np = __builtin_amdgcn_readfirstlane(r.np);
    return r;
}

template <int XR>
__device__ __forceinline__ void rx_next_unit(RxUnit& r, const int* firstL, int E, int tiles) {
    int end = __builtin_amdgcn_readfirstlane(firstL[r.e + 1]);
    if (r.p0 + XR < end) {
        ++r.j;
        r.p0 += XR;
    } else {
        r.j = 0;
        if (++r.t == tiles) {
            r.t = 0;
            do {
                ++r.e;
                r.p0 = end;
                end = __builtin_amdgcn_readfirstlane(firstL[r.e + 1]);
            } while (r.e < E && end == r.p0);                 // firstL[E + 1] = firstL[E]: ends behind the last expert
        } else r.p0 = __builtin_amdgcn_readfirstlane(firstL[r.e]);
    }
    r.np = min(XR, end - r.p0);
}
