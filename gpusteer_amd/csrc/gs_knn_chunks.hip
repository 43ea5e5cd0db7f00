// Exhaustive exact search of small or sparse target groups (walls, obstacles,
// a small group's search of another far away) by teams of lanes over the
// target's 64-slot chunks (gs_knn_chunks.hpp).
#include "gs_knn_chunks.hpp"

namespace gs {

// One wavefront per chunk.
__global__ __launch_bounds__(kBlock) void k_chunk_boxes(uint32_t n, uint32_t chunks, const float4* __restrict__ pos,
                                                        float* __restrict__ boxes) {
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x, c = s >> 6;
    if (c >= chunks) return;  // the whole wavefront
    const float nan = __builtin_nanf("");
    const float4 p = s < n ? pos[s] : make_float4(nan, nan, nan, 0.f);
    // fminf / fmaxf ignore NaN; a chunk without numbers keeps the empty box.
    float lo[3] = {fminf(p.x, INFINITY), fminf(p.y, INFINITY), fminf(p.z, INFINITY)};
    float hi[3] = {fmaxf(p.x, -INFINITY), fmaxf(p.y, -INFINITY), fmaxf(p.z, -INFINITY)};
    const uint64_t numbers = __ballot(p.x == p.x && p.y == p.y && p.z == p.z);
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) {
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            lo[a] = fminf(lo[a], __shfl_xor(lo[a], off, 64));
            hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], off, 64));
        }
    }
    if ((threadIdx.x & 63u) != 0) return;
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        boxes[a * chunks + c] = lo[a];
        boxes[(3 + a) * chunks + c] = hi[a];
    }
    boxes[6 * chunks + c] = (float)__popcll(numbers);
}

void launch_chunk_boxes(gs_group_s* B) {
    if (B->n == 0 || (B->cbox_fresh && !recording_frame())) return;
    const uint32_t chunks = (B->n + 63u) / 64u;
    k_chunk_boxes<<<blocks_for(B->n), kBlock, 0, B->ctx->stream>>>(B->n, chunks, B->spos.p, B->cbox.p);
    GS_LAUNCHED("k_chunk_boxes");
    B->cbox_fresh = !recording_frame();
}

template <int G, int KM>
__global__ __launch_bounds__(kBlock) void k_knn_chunks(uint32_t nA, const float4* __restrict__ apos, uint32_t nB,
                                                       const float4* __restrict__ bpos,
                                                       const float* __restrict__ boxes, int self, uint32_t k, float cap2,
                                                       const uint32_t* __restrict__ seed,
                                                       const uint32_t* __restrict__ row_map,
                                                       const uint32_t* __restrict__ val_map,
                                                       uint32_t* __restrict__ out_idx, float* __restrict__ out_dist) {
    __shared__ TeamLds<G, KM, 1> lds;
    TeamList<G, KM, 1> L(lds, k);
    const uint32_t s = blockIdx.x * team_queries<G>() + threadIdx.x / G;
    const bool active = s < nA;
    const float4 q = active ? apos[s] : make_float4(0.f, 0.f, 0.f, 0.f);
    if (nB > 0) {
        float thr = cap2;
        if (seed)
            thr = fminf(cap2, team_seed_bound(L, active, seed, nA, (active && row_map) ? row_map[s] : s, nB, val_map, q.x,
                                              q.y, q.z, bpos));
        const FlatQuery Q{q.x, q.y, q.z, thr, self ? s : UINT32_MAX, active};
        knn_chunks_team(L, Q, nB, bpos, boxes);
    }
    if (active) L.store(nA, s, out_idx, out_dist);
}

void launch_knn_chunks(gs_group_s* A, gs_knn_s* out, gs_group_s* B, float cap2, const uint32_t* seed,
                       const uint32_t* row_map, const uint32_t* val_map) {
    const uint32_t nA = A->n;
    if (nA == 0) return;
    launch_chunk_boxes(B);
    const bool wide = team_lanes(nA, out->k) == 16;
#define GS_CHUNKS(G, KM)                                                                                       \
    k_knn_chunks<G, KM><<<blocks_for(nA, team_queries<G>()), kBlock, 0, A->ctx->stream>>>(                     \
        nA, A->spos.p, B->n, B->spos.p, B->cbox.p, A == B ? 1 : 0, out->k, cap2, seed, row_map, val_map,       \
        out->idx_alt(), out->dist_alt())
    if (wide && out->k <= 8) GS_CHUNKS(16, 8);
    else if (wide) GS_CHUNKS(16, 16);
    else if (out->k <= 8) GS_CHUNKS(8, 8);
    else GS_CHUNKS(8, 16);
#undef GS_CHUNKS
    GS_LAUNCHED("k_knn_chunks");
}

}  // namespace gs
