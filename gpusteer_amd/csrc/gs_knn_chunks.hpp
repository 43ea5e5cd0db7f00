// Exact KNN of a team's query by an exhaustive scan of a small group, chunk by
// chunk: the snapshot is in cell order, so 64 consecutive slots are close to
// each other, and a chunk whose bounding box lies beyond the query's bound is
// skipped.  The box distance is formed with the per-axis subtractions and the
// summation order of a candidate's d2 and every step is monotone, so it is
// never above a member's d2: the skip drops only points the list would reject.
#pragma once
#include "gs_knn_team.hpp"

namespace gs {

// boxes: [7][chunks] (launch_chunk_boxes).  Q as for knn_search_team (thr: the
// cap or the seed's bound).  Without a bound the nearest chunk that holds
// enough points gives one: its farthest corner.
template <int G, int KM, int RF>
__device__ __forceinline__ void knn_chunks_team(TeamList<G, KM, RF>& L, const FlatQuery& Q, uint32_t nB,
                                                const float4* __restrict__ bpos, const float* __restrict__ boxes) {
    const __amdgpu_buffer_rsrc_t rb = pos_rsrc(bpos, nB);
    const uint32_t chunks = (nB + 63u) / 64u;
    const float q[3] = {Q.x, Q.y, Q.z};
    L.cnt = 0;
    L.lim = Q.thr;
    if (!Q.active || Q.thr < 0.f) return;  // the whole team
    if (L.lim == INFINITY) {
        float far2 = INFINITY;
        for (uint32_t c = L.lane; c < chunks; c += G) {
            float d2 = 0.f;
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const float lo = q[a] - boxes[a * chunks + c], hi = boxes[(3 + a) * chunks + c] - q[a];
                const float e = fmaxf(fabsf(lo), fabsf(hi));
                d2 += e * e;
            }
            // more than k points: the query may be one of them
            if (boxes[6 * chunks + c] > (float)L.k) far2 = fminf(far2, d2 * (1.f + 2e-5f) + 0x1p-100f);
        }
        // (a NaN distance leaves the bound infinite)
        L.lim = -L.max_of(-far2);
    }
    for (uint32_t c0 = 0; c0 < chunks; c0 += G) {
        const uint32_t c = c0 + L.lane;
        float d2 = INFINITY;
        if (c < chunks) {
            float g2[3];
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                const float gap =
                    fmaxf(fmaxf(boxes[a * chunks + c] - q[a], q[a] - boxes[(3 + a) * chunks + c]), 0.f);
                g2[a] = gap * gap;
            }
            d2 = (g2[0] + g2[1]) + g2[2];
        }
        int M = 0;
        L.push_run(c * 64u, (c < chunks && d2 <= L.lim) ? min(64u, nB - c * 64u) : 0u, M);
        if (M != 0) L.scan(M, Q.x, Q.y, Q.z, Q.self, rb);
    }
    L.reduce();
}

}  // namespace gs
