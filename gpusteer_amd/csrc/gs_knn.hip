// Exact k-nearest-neighbour search through the bins (brute force:
// gs_knn_brute.hip).
//
// Semantics (both): for each query a of group A, the k points b of
// group B with the smallest key (d2, b), d2 = ((ax-bx)^2 + (ay-by)^2) + (az-bz)^2
// in fp32, excluding a itself when A and B are the same group.  This is the
// order KNNBruteForceCUDAKernelV2 produces (strict '<' over an ascending scan:
// the lower index wins ties, include/OpenSteer/CUDA/KNNBruteForceCudaKernel.cu:245-270).
// Output is slot-major [k][nA] indexed by the query's own index
// (KNNBinningV2Kernel.cu:520-526), padded with UINT32_MAX / FLT_MAX (:451-457),
// distance = sqrtf(d2).
//
// Top-k selection: a register-resident sorted list of KMAX (d2, index) pairs
// with a branch-free compare-exchange ripple.  For k < KMAX the first KMAX-k
// entries hold a sentinel below every real key, so the list's last entry is
// always the k-th best and no register is ever indexed dynamically.
//
// Binned search replaces KNNBinningV2Kernel (KNNBinningV2Kernel.cu:417-528),
// which scans a fixed cell radius and is therefore approximate.  Here each
// query (one lane, queries in sorted/cell order so a wavefront's lanes share
// cells) scans the box of ring 1 around its cell (3 x 3 columns, or 5 x 5 for
// fine lattices, each column's z-run trimmed to the bound's sphere), then
// rings of growing radius while the k-th best d2 is not below the squared
// distance to every unscanned cell.  The bound starts at +inf or, when the
// container holds the exact result of the previous call for the same groups,
// at the largest current d2 of those k previous neighbours (a valid upper
// bound on the k-th distance: they are k distinct candidates).  Either way
// the result is the exact k nearest.
#include "gs_knn_core.hpp"

namespace gs {

// One lane per query slot s of A (storage = cell order, so a wavefront's lanes
// share cells and their candidate runs overlap in cache).  The flat path
// (RF == 1) takes its launch shape as template arguments: BS threads per
// block and APL queries per lane (a block covers APL consecutive runs of BS
// slots), both picked by the autotuner (gs_context_set_shape).
template <int KMAX, int RF, int BS = kBlock, int APL = 1>
__global__ __launch_bounds__(BS, RF == 1 ? (KMAX <= 8 ? 5 : (KMAX <= 16 ? 4 : 1)) : 1) void k_knn_binned(uint32_t nA, const float4* __restrict__ apos, uint32_t nB,
                                                       const float4* __restrict__ bpos,
                                                       const uint32_t* __restrict__ bstart, GridDev g, int self,
                                                       uint32_t k, int R0, float cap2, const uint32_t* __restrict__ seed,
                                                       const uint32_t* __restrict__ row_map,
                                                       const uint32_t* __restrict__ val_map,
                                                       uint32_t* __restrict__ out_idx, float* __restrict__ out_dist,
                                                       const uint32_t* __restrict__ box) {
    if constexpr (RF == 1) {
        // Slot a of the lane's APL slots (a block covers APL runs of BS slots).
        auto one = [&](uint32_t s) {
            TopK<KMAX> h;
            h.init(k);
            // Every lane stays to the end: the wavefront completes its lanes'
            // inexact queries together (lanes past nA only help).
            const bool active = s < nA;
            const float4 q = active ? apos[s] : make_float4(0.f, 0.f, 0.f, 0.f);
            FlatQuery Q{q.x, q.y, q.z, INFINITY, self ? s : UINT32_MAX, active};
            if (nB > 0) {
                Q.thr = fminf(cap2, (seed && active) ? seed_bound<KMAX>(seed, k, nA, row_map ? row_map[s] : s, nB,
                                                                        val_map, q.x, q.y, q.z, bpos)
                                                     : INFINITY);
                // A capped query that cannot reach B's bounding box has no
                // candidate (box: NULL for an uncapped search).
                if (box && active && box_beyond(box, q.x, q.y, q.z, cap2)) Q.thr = -1.f;
                GS_FLAT_LDS_NK(BS, KMAX)
                knn_search_flat<KMAX, BS>(h, Q, g, nB, bpos, bstart, flds);
            }
            if (active) h.store(k, nA, s, out_idx, out_dist);
        };
        if constexpr (APL == 1) {
            one(xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x);
        } else {
            for (int a = 0; a < APL; ++a) one((xcd_block(blockIdx.x, gridDim.x) * APL + a) * BS + threadIdx.x);
        }
    } else {
        static_assert(BS == kBlock && APL == 1, "the box walk has the default shape");
        const uint32_t s = xcd_block(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
        TopK<KMAX> h;
        h.init(k);
        if (s >= nA) return;
        const float4 q = apos[s];
        if (nB > 0) {
            const float thr = fminf(cap2, seed ? seed_bound<KMAX>(seed, k, nA, row_map ? row_map[s] : s, nB,
                                                                  val_map, q.x, q.y, q.z, bpos)
                                               : INFINITY);
            GS_DEFER_LDS
            knn_search<KMAX, RF>(h, thr, q.x, q.y, q.z, self ? s : UINT32_MAX, g, R0, bpos, bstart, lbuf);
        }
        h.store(k, nA, s, out_idx, out_dist);
    }
}

// Moves a [k][nA] result from the previous storage order of A and/or B to the
// current one: row s_old -> row_map[s_old], value v_old -> val_map[v_old].
__global__ __launch_bounds__(kBlock) void k_knn_remap(uint32_t nA, uint32_t k, const uint32_t* __restrict__ in_idx,
                                                      const float* __restrict__ in_dist,
                                                      const uint32_t* __restrict__ row_map,
                                                      const uint32_t* __restrict__ val_map,
                                                      uint32_t* __restrict__ out_idx, float* __restrict__ out_dist) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= nA) return;
    const uint32_t r = row_map ? row_map[s] : s;
    for (uint32_t j = 0; j < k; ++j) {
        uint32_t v = in_idx[(size_t)j * nA + s];
        if (v != UINT32_MAX && val_map) v = val_map[v];
        out_idx[(size_t)j * nA + r] = v;
        out_dist[(size_t)j * nA + r] = in_dist[(size_t)j * nA + s];
    }
}

template <int KMAX, int RF, int BS = kBlock, int APL = 1>
static void run_binned_shape(gs_group_s* A, gs_knn_s* out, gs_group_s* B, uint32_t R0, float cap2,
                             const uint32_t* seed, const uint32_t* row_map, const uint32_t* val_map, bool dist) {
    const uint32_t nA = A->n;
    k_knn_binned<KMAX, RF, BS, APL><<<blocks_for(nA, BS * APL), BS, 0, A->ctx->stream>>>(
        nA, A->spos.p, B->n, B->spos.p, B->start.p, B->bin_grid, A == B ? 1 : 0, out->k, (int)R0, cap2, seed,
        row_map, val_map, out->idx_alt(), dist ? out->dist_alt() : nullptr,
        (std::isfinite(cap2) && B->bbox_fresh) ? B->bbox[B->bbox_cur].p : nullptr);
    GS_LAUNCHED("k_knn_binned");
}

template <int KMAX, int RF>
static void run_binned(gs_group_s* A, gs_knn_s* out, gs_group_s* B, uint32_t R0, float cap2, const uint32_t* seed,
                       const uint32_t* row_map, const uint32_t* val_map, bool d) {
    // The k = 7 flat search runs in the context's launch shape.
    if constexpr (KMAX == 7 && RF == 1) {
        const LaunchShape sh = A->ctx->shape[GS_SHAPE_KNN];
        if (sh.block == 128 && sh.apl == 1) return run_binned_shape<7, 1, 128, 1>(A, out, B, R0, cap2, seed, row_map, val_map, d);
        if (sh.block == 128 && sh.apl == 2) return run_binned_shape<7, 1, 128, 2>(A, out, B, R0, cap2, seed, row_map, val_map, d);
        if (sh.block == 256 && sh.apl == 2) return run_binned_shape<7, 1, 256, 2>(A, out, B, R0, cap2, seed, row_map, val_map, d);
        if (sh.block == 512 && sh.apl == 1) return run_binned_shape<7, 1, 512, 1>(A, out, B, R0, cap2, seed, row_map, val_map, d);
        if (sh.block == 512 && sh.apl == 2) return run_binned_shape<7, 1, 512, 2>(A, out, B, R0, cap2, seed, row_map, val_map, d);
    }
    run_binned_shape<KMAX, RF>(A, out, B, R0, cap2, seed, row_map, val_map, d);
}

template <int KMAX>
static void run_binned_rf(gs_group_s* A, gs_knn_s* out, gs_group_s* B, uint32_t R0, float cap2,
                          const uint32_t* seed, const uint32_t* row_map, const uint32_t* val_map, bool d) {
    // search_radius selects the fast path's column radius: 3 x 3 columns for
    // lattices whose cell is about the k-th neighbour distance, 5 x 5 for
    // finer lattices.
    // The 3 x 3 path addresses B with 32-bit byte offsets (fewer than 2^27
    // points); larger groups take the 5 x 5 walk, which is exact as well.
    // Lists longer than 8 keep the 3 x 3 path on every lattice: the 5 x 5
    // walk holding 16 keys exceeds the register file and spills.
    if ((R0 >= 2 && KMAX <= 8) || B->n >= kFlatMaxPoints)
        run_binned<KMAX, 2>(A, out, B, R0, cap2, seed, row_map, val_map, d);
    else run_binned<KMAX, 1>(A, out, B, R0, cap2, seed, row_map, val_map, d);
}

void launch_knn_binned(gs_group_s* A, gs_knn_s* out, gs_group_s* B, uint32_t search_radius, float cap2,
                       const uint32_t* seed, const uint32_t* row_map, const uint32_t* val_map, bool dist,
                       bool wide_cap) {
    if (A->n == 0) return;
    if (launch_knn_team(A, out, B, search_radius, cap2, seed, row_map, val_map, dist, wide_cap)) return;
    // k = 7 (the parameter files' default) gets lists of exactly 7 entries:
    // one compare-exchange fewer per insertion than the 8-entry lists.
    if (out->k == 7) run_binned_rf<7>(A, out, B, search_radius, cap2, seed, row_map, val_map, dist);
    else if (out->k <= 8) run_binned_rf<8>(A, out, B, search_radius, cap2, seed, row_map, val_map, dist);
    else if (out->k <= 16) run_binned_rf<16>(A, out, B, search_radius, cap2, seed, row_map, val_map, dist);
    else run_binned_rf<32>(A, out, B, search_radius, cap2, seed, row_map, val_map, dist);
}

void launch_knn_remap(gs_knn_s* out, uint32_t nA, const uint32_t* row_map, const uint32_t* val_map) {
    if (nA == 0) return;
    k_knn_remap<<<blocks_for(nA), kBlock, 0, out->ctx->stream>>>(nA, out->k, out->idx(), out->dist(), row_map,
                                                                 val_map, out->idx_alt(), out->dist_alt());
    GS_LAUNCHED("k_knn_remap");
}

}  // namespace gs
