// Exact search of small or sparse target groups (walls, obstacles) and of small
// groups by small groups, by teams of lanes over the target's 64-slot chunks
// (gs_knn_chunks.hpp).
#include <cmath>

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
}

void launch_chunk_boxes(gs_group_s* B) {
    if (B->n == 0 || (B->cbox_fresh && !recording_frame())) return;
    const uint32_t chunks = (B->n + 63u) / 64u;
    k_chunk_boxes<<<blocks_for(B->n), kBlock, 0, B->ctx->stream>>>(B->n, chunks, B->spos.p, B->cbox.p);
    GS_LAUNCHED("k_chunk_boxes");
    B->cbox_fresh = !recording_frame();
}

// Local: the cells around the query first (bstart, g: B's lattice), as far as
// that takes no more columns than there are chunks; then the chunks.
template <int G, int KM, int RF, bool Local>
__global__ __launch_bounds__(kBlock) void k_knn_chunks(uint32_t nA, const float4* __restrict__ apos, uint32_t nB,
                                                       const float4* __restrict__ bpos,
                                                       const float* __restrict__ boxes,
                                                       const uint32_t* __restrict__ bstart, GridDev g,
                                                       const uint32_t* __restrict__ box, int self, uint32_t k,
                                                       float cap2, int wide_cap, const uint32_t* __restrict__ seed,
                                                       const uint32_t* __restrict__ row_map,
                                                       const uint32_t* __restrict__ val_map,
                                                       uint32_t* __restrict__ out_idx, float* __restrict__ out_dist) {
    __shared__ TeamLds<G, KM, RF> lds;
    TeamList<G, KM, RF> L(lds, k);
    const uint32_t s = blockIdx.x * team_queries<G>() + threadIdx.x / G;
    const bool active = s < nA;
    const float4 q = active ? apos[s] : make_float4(0.f, 0.f, 0.f, 0.f);
    if (nB > 0) {
        float thr = cap2;
        if (seed)
            thr = fminf(cap2, team_seed_bound(L, active, seed, nA, (active && row_map) ? row_map[s] : s, nB, val_map, q.x,
                                              q.y, q.z, bpos));
        // A list that the cap left short last time needs no other bound.
        const bool bound_first = (!seed && wide_cap) || thr == INFINITY;
        // As k_knn_binned: no candidate within the cap of B's bounding box.
        if (box && active && box_beyond(box, q.x, q.y, q.z, cap2)) thr = -1.f;
        FlatQuery Q{q.x, q.y, q.z, thr, self ? s : UINT32_MAX, active};
        bool found = false;
        if (Local) {
            found = knn_search_team<true>(L, Q, g, nB, bpos, bstart, bound_first, (int)((nB + 63u) / 64u));
            Q.thr = L.lim;
        }
        if (!found) knn_chunks_team(L, Q, bound_first, nB, bpos, boxes);
    }
    if (active) L.store(nA, s, out_idx, out_dist);
}

// Bound by latency at a few thousand queries, by VALU issue beyond.  131,072
// agents x 1,254 walls (k = 3, cap 140): 46.5 -> 14.8 us (one lane per query,
// no seed, before).  Two groups of 5,000 (k = 7, cap of ten cells, 100 x 1 x
// 100 cells): 47 us by ranges per block and a merge, 50 over the chunks alone (a
// chunk is a strip across the lattice, and one query without a seed under a
// wide cap holds its block up), 16 + 3 with the cells around the query first
// and rings without an end, 13 + 3 here.  The rings end at as many columns as
// chunks, at more cells than points, and at a ring full of points: with 5,000
// queries of 5,000 points (k = 7, 32^3 cells) mixed / apart / about one cluster,
// seeded: chunks alone 15 / 5 / 15 us, no end 20 / 59 / 125, here 17 / 14 / 15;
// unseeded, no cap 71 / 4 / 205, 28 / 58 / 230, here 26 / 25 / 36 (100 x 1 x 100
// cells 16 / 41 / 69; by ranges and a merge 100 / 117 / 98).
//
// A whole wavefront per query where there are few queries and many points; wider
// lattices than one cell high have more columns to share.  16 / 64 lanes, us, k
// = 7, seeded: 500 queries of 16,000 points mixed 14 / 11, apart 26 / 14, about
// one cluster 65 / 16; 2,048 of 16,384 14 / 12, 27 / 15, 69 / 19; 5,000 of 5,000
// 28 / 17, 17 / 15, 26 / 15, but 13 / 15, 20 / 23, 27 / 23 on 100 x 1 x 100 cells;
// 16,384 of 4,096 33 / 39, 19 / 31, 28 / 31 and 15 / 36, 25 / 49, 30 / 50.
constexpr uint32_t kTeam64Max = 4096, kTeam64MaxColumns = 8192, kTeam64MinPoints = 257;
void launch_knn_chunks(gs_group_s* A, gs_knn_s* out, gs_group_s* B, float cap2, const uint32_t* seed,
                       const uint32_t* row_map, const uint32_t* val_map, uint32_t local, bool wide_cap) {
    const uint32_t nA = A->n;
    if (nA == 0) return;
    launch_chunk_boxes(B);
    const bool wide = team_lanes(nA, out->k) == 16;
    const uint32_t* box = (local && std::isfinite(cap2) && B->bbox_fresh) ? B->bbox[B->bbox_cur].p : nullptr;
#define GS_CHUNKS(G, KM, RF, Local)                                                                            \
    k_knn_chunks<G, KM, RF, Local><<<blocks_for(nA, team_queries<G>()), kBlock, 0, A->ctx->stream>>>(          \
        nA, A->spos.p, B->n, B->spos.p, B->cbox.p, B->start.p, B->bin_grid, box, A == B ? 1 : 0, out->k, cap2, \
        wide_cap ? 1 : 0, seed, row_map, val_map, out->idx_alt(), out->dist_alt())
    static_assert(kSplitMaxA <= kTeam16Max, "a local search has 16 lanes per query");
    const bool columns = local && B->bin_grid.dx > 1 && B->bin_grid.dy > 1;
    if (nA <= (columns ? kTeam64MaxColumns : kTeam64Max) && B->n >= kTeam64MinPoints) {
        if (local >= 2 && out->k <= 8) GS_CHUNKS(64, 8, 2, true);
        else if (local >= 2) GS_CHUNKS(64, 16, 2, true);
        else if (local && out->k <= 8) GS_CHUNKS(64, 8, 1, true);
        else if (local) GS_CHUNKS(64, 16, 1, true);
        else if (out->k <= 8) GS_CHUNKS(64, 8, 1, false);
        else GS_CHUNKS(64, 16, 1, false);
    } else if (local >= 2 && out->k <= 8) GS_CHUNKS(16, 8, 2, true);
    else if (local >= 2) GS_CHUNKS(16, 16, 2, true);
    else if (local && out->k <= 8) GS_CHUNKS(16, 8, 1, true);
    else if (local) GS_CHUNKS(16, 16, 1, true);
    else if (wide && out->k <= 8) GS_CHUNKS(16, 8, 1, false);
    else if (wide) GS_CHUNKS(16, 16, 1, false);
    else if (out->k <= 8) GS_CHUNKS(8, 8, 1, false);
    else GS_CHUNKS(8, 16, 1, false);
#undef GS_CHUNKS
    GS_LAUNCHED("k_knn_chunks");
}

// The same search with one lane per query, for few targets and many queries
// and for lists longer than a team's.  B's snapshot is scanned from LDS.
//
// The snapshot is in cell order, so each wave's 64 entries of a tile are
// spatially coherent: the wave takes their bounding box, and a wave skips a
// chunk when no lane's query can reach the box within its current bound
// (its k-th key's d2, or the cap).  The box distance is formed with the
// same per-axis subtractions and the same summation order as a candidate's
// d2, and every step is monotone, so a member's d2 is never below it: the
// skip drops only candidates the heap would reject.
template <int KMAX>
__global__ __launch_bounds__(kBlock) void k_knn_snap_brute(uint32_t nA, const float4* __restrict__ apos, uint32_t nB,
                                                           const float4* __restrict__ bpos, int self, uint32_t k,
                                                           float cap2, uint32_t* __restrict__ out_idx,
                                                           float* __restrict__ out_dist) {
    __shared__ float4 tile[kBlock];
    __shared__ float box[kBlock / 64][6];
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = s < nA;
    const float4 q = active ? apos[s] : make_float4(0.f, 0.f, 0.f, 0.f);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    TopK<KMAX> h;
    h.init(k);
    for (uint32_t base = 0; base < nB; base += kBlock) {
        const uint32_t t = base + threadIdx.x;
        float lo[3] = {INFINITY, INFINITY, INFINITY}, hi[3] = {-INFINITY, -INFINITY, -INFINITY};
        if (t < nB) {
            const float4 p = bpos[t];
            tile[threadIdx.x] = p;
            lo[0] = hi[0] = p.x;
            lo[1] = hi[1] = p.y;
            lo[2] = hi[2] = p.z;
        }
#pragma unroll
        for (int off = 32; off >= 1; off >>= 1) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                lo[a] = fminf(lo[a], __shfl_xor(lo[a], off, 64));
                hi[a] = fmaxf(hi[a], __shfl_xor(hi[a], off, 64));
            }
        }
        if (lane == 0) {
#pragma unroll
            for (int a = 0; a < 3; ++a) {
                box[wave][a] = lo[a];
                box[wave][3 + a] = hi[a];
            }
        }
        __syncthreads();
        const uint32_t m = min((uint32_t)kBlock, nB - base);
        for (uint32_t c0 = 0; c0 < m; c0 += 64) {
            const int c = c0 >> 6;
            const float gx = fmaxf(fmaxf(box[c][0] - q.x, q.x - box[c][3]), 0.f);
            const float gy = fmaxf(fmaxf(box[c][1] - q.y, q.y - box[c][4]), 0.f);
            const float gz = fmaxf(fmaxf(box[c][2] - q.z, q.z - box[c][5]), 0.f);
            const float d2box = ((gx * gx) + (gy * gy)) + (gz * gz);
            const bool need = active && d2box <= fminf(cap2, h.worst());
            if (__ballot(need) == 0) continue;
            const uint32_t c1 = min(c0 + 64, m);
            if (need) {
                for (uint32_t j = c0; j < c1; ++j) {
                    const uint32_t b = base + j;
                    if (self && b == s) continue;
                    const float4 p = tile[j];
                    const float d2 = sqdist4(q.x, q.y, q.z, p);
                    const uint64_t kk = make_key(d2, id_of(p));
                    if (d2 <= cap2 && h.accepts(kk)) h.push(kk, b);
                }
            }
        }
        __syncthreads();
    }
    if (active) h.store(k, nA, s, out_idx, out_dist);
}

void launch_knn_snap_brute(gs_group_s* A, gs_knn_s* out, gs_group_s* B, float cap2) {
    const uint32_t nA = A->n;
    if (nA == 0) return;
    hipStream_t st = A->ctx->stream;
    const int self = A == B ? 1 : 0;
#define GS_SB(KM)                                                                                             \
    k_knn_snap_brute<KM><<<blocks_for(nA), kBlock, 0, st>>>(nA, A->spos.p, B->n, B->spos.p, self, out->k, cap2, \
                                                            out->idx_alt(), out->dist_alt())
    if (out->k <= 8) GS_SB(8);
    else if (out->k <= 16) GS_SB(16);
    else GS_SB(32);
#undef GS_SB
    GS_LAUNCHED("k_knn_snap_brute");
}

}  // namespace gs
