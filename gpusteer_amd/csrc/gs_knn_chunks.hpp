// Exact KNN of a team's query by an exhaustive scan of a small group, chunk by
// chunk: the snapshot is in cell order, so 64 consecutive slots are close to
// each other, and a chunk whose bounding box lies beyond the query's bound is
// skipped.  The box distance is formed with the per-axis subtractions and the
// summation order of a candidate's d2 and every step is monotone, so it is
// never above a member's d2: the skip drops only points the list would reject.
#pragma once
#include "gs_knn_team.hpp"

namespace gs {

// A lower bound on the d2 of chunk c's points (0 for a query that is no number).
__device__ __forceinline__ float chunk_gap2(const float* __restrict__ boxes, uint32_t chunks, uint32_t c,
                                            const float (&q)[3]) {
    float g2[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        const float gap = fmaxf(fmaxf(boxes[a * chunks + c] - q[a], q[a] - boxes[(3 + a) * chunks + c]), 0.f);
        g2[a] = gap * gap;
    }
    return (g2[0] + g2[1]) + g2[2];
}

// boxes: [6][chunks] (launch_chunk_boxes).  Q as for knn_search_team (thr: the
// cap, a seed's bound or that of a search that gave up).  bound_first: two
// passes that keep nothing but each lane's nearest points, over the nearest
// chunk and then over the others within the k-th of those, bound the search
// before it starts; without it a wide bound lets most points of a group into
// the buffer (131,072 queries of 1,254 mixed points, k = 7, unseeded: 332 us,
// with the nearest chunk's bound alone 58, here 54, k = 16 556 / 153 / 91; 5,000 of
// 5,000 about one cluster 96 / 68 / 55).
template <int G, int KM, int RF>
__device__ __forceinline__ void knn_chunks_team(TeamList<G, KM, RF>& L, const FlatQuery& Q, bool bound_first, uint32_t nB,
                                                const float4* __restrict__ bpos, const float* __restrict__ boxes) {
    const __amdgpu_buffer_rsrc_t rb = pos_rsrc(bpos, nB);
    const uint32_t chunks = (nB + 63u) / 64u;
    const float q[3] = {Q.x, Q.y, Q.z};
    L.cnt = 0;
    L.lim = Q.thr;
    if (!Q.active || Q.thr < 0.f) return;  // the whole team
    if (bound_first && chunks > 1u) {
        float best = INFINITY;
        uint32_t at = UINT32_MAX;
        for (uint32_t c = L.lane; c < chunks; c += G) {
            const float d2 = chunk_gap2(boxes, chunks, c, q);
            if (d2 < best) {
                best = d2;
                at = c;
            }
        }
        const float near2 = -L.max_of(-best);
        if (near2 > L.lim) return;  // no chunk in reach
        if (near2 < INFINITY) {
            const auto who = L.votes(best == near2);
            at = (uint32_t)__shfl((int)at, (int)L.first + __ffsll((unsigned long long)who) - 1, 64);
            typename TeamList<G, KM, RF>::Two two;
            int M = 0;
            L.push_run(at * 64u, L.lane == 0 ? min(64u, nB - at * 64u) : 0u, M);
            L.nearest(two, M, Q.x, Q.y, Q.z, Q.self, rb);
            L.lim = fminf(L.lim, L.kth(two));
            for (uint32_t c0 = 0; c0 < chunks; c0 += G) {
                const uint32_t c = c0 + L.lane;
                const float d2 = c < chunks && c != at ? chunk_gap2(boxes, chunks, c, q) : INFINITY;
                M = 0;
                L.push_run(c * 64u, (c < chunks && c != at && d2 <= L.lim) ? min(64u, nB - c * 64u) : 0u, M);
                if (M != 0) L.nearest(two, M, Q.x, Q.y, Q.z, Q.self, rb);
            }
            L.lim = fminf(L.lim, L.kth(two));
        }
    }
    for (uint32_t c0 = 0; c0 < chunks; c0 += G) {
        const uint32_t c = c0 + L.lane;
        const float d2 = c < chunks ? chunk_gap2(boxes, chunks, c, q) : INFINITY;
        int M = 0;
        L.push_run(c * 64u, (c < chunks && d2 <= L.lim) ? min(64u, nB - c * 64u) : 0u, M);
        if (M != 0) L.scan(M, Q.x, Q.y, Q.z, Q.self, rb);
    }
    L.reduce();
}

}  // namespace gs
