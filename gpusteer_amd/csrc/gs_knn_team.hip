// Launches of the team search (gs_knn_team.hpp): the binned search of small
// and middle query groups.
#include <cmath>

#include "gs_knn_team.hpp"

namespace gs {

// G lanes per query (knn_search_team), kBlock / G queries per block.
template <int G, int KM, int RF>
__global__ __launch_bounds__(kBlock) void k_knn_team(uint32_t nA, const float4* __restrict__ apos, uint32_t nB,
                                                     const float4* __restrict__ bpos,
                                                     const uint32_t* __restrict__ bstart, GridDev g, int self,
                                                     uint32_t k, float cap2, int wide_cap,
                                                     const uint32_t* __restrict__ seed,
                                                     const uint32_t* __restrict__ row_map,
                                                     const uint32_t* __restrict__ val_map,
                                                     uint32_t* __restrict__ out_idx, float* __restrict__ out_dist,
                                                     const uint32_t* __restrict__ box) {
    __shared__ TeamLds<G, KM, RF> lds;
    TeamList<G, KM, RF> L(lds, k);
    const uint32_t s = xcd_block(blockIdx.x, gridDim.x) * team_queries<G>() + threadIdx.x / G;
    const bool active = s < nA;
    const float4 q = active ? apos[s] : make_float4(0.f, 0.f, 0.f, 0.f);
    if (nB > 0) {
        float thr = cap2;
        if (seed)
            thr = fminf(cap2, team_seed_bound(L, active, seed, nA, (active && row_map) ? row_map[s] : s, nB, val_map,
                                                 q.x, q.y, q.z, bpos));
        const bool bound_first = thr == INFINITY || (!seed && wide_cap);
        // As k_knn_binned: no candidate within the cap of B's bounding box.
        if (box && active && box_beyond(box, q.x, q.y, q.z, cap2)) thr = -1.f;
        const FlatQuery Q{q.x, q.y, q.z, thr, self ? s : UINT32_MAX, active};
        knn_search_team<false>(L, Q, g, nB, bpos, bstart, bound_first);
    }
    if (active) L.store(nA, s, out_idx, out_dist);
}

// Bound by the serial chain of one team (seven dependent loads: query, seed,
// maps, neighbours, cell starts, candidates) while the chip is not full, by
// VALU issue (about 1,000 instructions per wavefront of 64 / G queries)
// beyond.  4,096 agents, k = 7: 44.5 -> 13 us (16 lanes); 100,003: 50.9 -> 32
// us (8 lanes); 65,536 points unseeded, half of them in clumps: 161 -> 52 us.
template <int G>
static void run_team(gs_group_s* A, gs_knn_s* out, gs_group_s* B, uint32_t R0, float cap2, const uint32_t* seed,
                     const uint32_t* row_map, const uint32_t* val_map, bool dist, bool wide_cap) {
    const uint32_t nA = A->n;
    const uint32_t* box = (std::isfinite(cap2) && B->bbox_fresh) ? B->bbox[B->bbox_cur].p : nullptr;
    const unsigned nb = blocks_for(nA, team_queries<G>());
#define GS_TEAM(KM, RF)                                                                                          \
    k_knn_team<G, KM, RF><<<nb, kBlock, 0, A->ctx->stream>>>(                                                   \
        nA, A->spos.p, B->n, B->spos.p, B->start.p, B->bin_grid, A == B ? 1 : 0, out->k, cap2, wide_cap ? 1 : 0, \
        seed, row_map, val_map, out->idx_alt(), dist ? out->dist_alt() : nullptr, box)
    if (out->k <= 8 && R0 >= 2) GS_TEAM(8, 2);
    else if (out->k <= 8) GS_TEAM(8, 1);
    else if (R0 >= 2) GS_TEAM(16, 2);
    else GS_TEAM(16, 1);
#undef GS_TEAM
    GS_LAUNCHED("k_knn_team");
}

bool launch_knn_team(gs_group_s* A, gs_knn_s* out, gs_group_s* B, uint32_t search_radius, float cap2,
                     const uint32_t* seed, const uint32_t* row_map, const uint32_t* val_map, bool dist,
                     bool wide_cap) {
    if (out->k > kTeamMaxK || B->n >= kFlatMaxPoints) return false;
    // A launch shape set by the caller (gs_context_set_shape) is the
    // one-lane search's.
    const LaunchShape sh = A->ctx->shape[GS_SHAPE_KNN];
    if (out->k == 7 && (sh.block != kBlock || sh.apl != 1)) return false;
    const int lanes = team_lanes(A->n, out->k);
    if (lanes == 16) run_team<16>(A, out, B, search_radius, cap2, seed, row_map, val_map, dist, wide_cap);
    else if (lanes == 8) run_team<8>(A, out, B, search_radius, cap2, seed, row_map, val_map, dist, wide_cap);
    return lanes != 1;
}

}  // namespace gs
