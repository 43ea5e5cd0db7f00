// Crowd frames of two small groups, phase by phase for both groups at once.
//
// The call sequence of a crowd frame (plugins/ChokePointGroup.cpp:683-728) is
// some thirty launches of 2 - 10 us over a few thousand agents each: what they
// cost is launches and latency, on a chip that is nearly empty.  Here a frame
// is six: the builds' three passes (gs_bins.hip), the eight searches, walls and
// obstacles, separation with seek and the integrate, each over both groups.
// 10,000 agents: 159 -> 54 us a frame (search 14.2, reorder 9.5, integrate 8.0,
// walls and obstacles 6.9, scan 6.6, keys 3.8 us).
//
// Same results, bit for bit.  Between the calls of the sequence the groups see
// each other's state: group 0's separation from group 1 reads group 1's
// positions before group 1's walls move them, which are the snapshot's, and
// everything else reads the positions that the walls have left, which the
// second phase only reads.  Both phases write positions and forward vectors to
// the alternate buffers: a frame then leaves every field in the buffer in which
// the separate calls would, which recorded frames are compared by.
#include "gs_knn_chunks.hpp"
#include "gs_ops.hpp"

namespace gs {

constexpr int kPairLanes = 16;
struct PairList {
    const float4* bpos;
    const uint32_t* start;  // cell starts, or NULL: exhaustive over the chunk boxes
    const float* boxes;
    const uint32_t* box;  // B's bounding box (capped searches), or NULL
    const uint32_t *seed, *row_map, *val_map;
    uint32_t* idx;
    float* dist;
    uint32_t nB, k;
    int self;
    float cap2;
};
struct PairSearch {
    const float4* apos[2];
    uint32_t n[2];
    PairList l[8];
    GridDev g;
};

// blockIdx.y: the list.
__global__ __launch_bounds__(kBlock) void k_pair_search(PairSearch P) {
    __shared__ TeamLds<kPairLanes, 8, 1> lds;
    const PairList& l = P.l[blockIdx.y];
    const uint32_t g = blockIdx.y >> 2, nA = P.n[g];
    TeamList<kPairLanes, 8, 1> L(lds, l.k);
    const uint32_t s = blockIdx.x * team_queries<kPairLanes>() + threadIdx.x / kPairLanes;
    const bool active = s < nA;
    const float4 q = active ? P.apos[g][s] : make_float4(0.f, 0.f, 0.f, 0.f);
    if (l.nB > 0) {
        float thr = l.cap2;
        if (l.seed)
            thr = fminf(thr, team_seed_bound(L, active, l.seed, nA, (active && l.row_map) ? l.row_map[s] : s, l.nB,
                                             l.val_map, q.x, q.y, q.z, l.bpos));
        const bool bound_first = thr == INFINITY;
        if (l.box && active && box_beyond(l.box, q.x, q.y, q.z, l.cap2)) thr = -1.f;
        const FlatQuery Q{q.x, q.y, q.z, thr, l.self ? s : UINT32_MAX, active};
        if (l.start) knn_search_team<false>(L, Q, P.g, l.nB, l.bpos, l.start, bound_first);
        else knn_chunks_team(L, Q, bound_first, l.nB, l.bpos, l.boxes);
    }
    if (active) L.store(nA, s, l.idx, l.dist);
}

void launch_pair_search(gs_group_s* const g[2], gs_group_s* W, gs_group_s* O, gs_knn_s* const knn[8],
                        const ListSeed seeds[4], float cap2) {
    launch_chunk_boxes(W);
    launch_chunk_boxes(O);
    PairSearch P{};
    P.g = g[0]->bin_grid;
    uint32_t n = 0;
    for (int i = 0; i < 2; ++i) {
        P.apos[i] = g[i]->spos.p;
        P.n[i] = g[i]->n;
        n = std::max(n, g[i]->n);
    }
    for (int j = 0; j < 8; ++j) {
        PairList& l = P.l[j];
        const int a = j / 4, w = j % 4;
        gs_group_s* const B = w == 0 ? g[a] : w == 1 ? g[1 - a] : w == 2 ? W : O;
        l.bpos = B->spos.p;
        l.nB = B->n;
        l.k = knn[j]->k;
        l.idx = knn[j]->idx_alt();
        l.dist = knn[j]->dist_alt();
        l.self = w == 0;
        l.cap2 = w == 1 ? cap2 : INFINITY;
        if (w < 2) {
            l.start = B->start.p;
            const ListSeed& sd = seeds[2 * a + w];
            l.seed = sd.seed;
            l.row_map = sd.row_map;
            l.val_map = sd.val_map;
            if (w == 1 && cap2 < INFINITY && B->bbox_fresh) l.box = B->bbox[B->bbox_cur].p;
        } else {
            l.boxes = B->cbox.p;
        }
    }
    k_pair_search<<<dim3(blocks_for(n, team_queries<kPairLanes>()), 8), kBlock, 0, g[0]->ctx->stream>>>(P);
    GS_LAUNCHED("k_pair_search");
}

struct PairAgents {
    uint32_t n;
    Agents A;
    const uint32_t *kown, *kother, *kwalls, *kobs;
    uint32_t k[4];
    float *npx, *npy, *npz, *nfx, *nfy, *nfz;  // A's alternate buffers
    float goal[3];
};
struct PairSteer {
    PairAgents a[2];
    const float4* spos1;  // group 1's snapshot
    uint32_t nW, nO;
    gs_walls W;
    const float *ox, *oy, *oz, *orad;
    float mt_walls, w_walls, mt_obs, w_obs, w_seek, dt;
    uint32_t mask_seek;
    FlockTerm sep;
};

// gs_clear_bits, gs_steer_avoid_walls, gs_steer_avoid_obstacles.
__global__ __launch_bounds__(kBlock) void k_pair_avoid(PairSteer P) {
    const PairAgents& G = P.a[blockIdx.y];
    const Agents& A = G.A;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= G.n) return;
    uint32_t bits = 0u;
    f3 pos = ld3(A.px, A.py, A.pz, i), dir = ld3(A.fx, A.fy, A.fz, i);
    const f3 side = ld3(A.sx, A.sy, A.sz, i);
    f3 steering = ld3(A.gx, A.gy, A.gz, i);
    const float radius = A.radius[i], speed = A.speed[i];
    avoid_walls_one(pos, dir, side, radius, speed, G.kwalls + i, G.n, G.k[2], P.nW, P.W, P.mt_walls, P.w_walls, steering,
                    bits);
    avoid_obstacles_one(pos, dir, side, ld3(A.ux, A.uy, A.uz, i), radius, speed, G.kobs + i, G.n, G.k[3], P.nO, P.ox, P.oy,
                        P.oz, P.orad, P.mt_obs, P.w_obs, steering, bits);
    st3(G.npx, G.npy, G.npz, i, pos);
    st3(G.nfx, G.nfy, G.nfz, i, dir);
    st3(A.gx, A.gy, A.gz, i, steering);
    A.bits[i] = bits;
}

// gs_steer_separation from the own and the other group, gs_steer_seek,
// gs_update_group.
template <int MODE>
__global__ __launch_bounds__(kBlock) void k_pair_finish(PairSteer P) {
    const PairAgents &G = P.a[blockIdx.y], &H = P.a[1 - blockIdx.y];
    const Agents& A = G.A;
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= G.n) return;
    uint32_t bits = A.bits[i];
    f3 steering = ld3(A.gx, A.gy, A.gz, i);
    f3 pos = ld3(A.px, A.py, A.pz, i), fwd = ld3(A.fx, A.fy, A.fz, i);
    const float radius = A.radius[i];
    float speed = A.speed[i];
    const FlockTerm off{0.f, 0.f, 0.f, 0.f, 0u, 0};
    for (int w = 0; w < 2; ++w) {
        if (bits & P.sep.mask) break;  // bits only accumulate
        const Agents& B = w == 0 ? G.A : H.A;
        f3 bp[8], bf[8];
        const int m = gather_neighbours<8>(w == 0 ? G.kown : G.kother, G.k[w], G.n, i, w == 0 ? G.n : H.n,
                                           w == 1 && blockIdx.y == 0 ? P.spos1 : nullptr, B.px, B.py, B.pz, nullptr,
                                           nullptr, nullptr, false, bp, bf);
        flock_core<MODE, 8>(pos, fwd, radius, m, bp, bf, P.sep, off, off, steering, bits);
    }
    if (!(bits & P.mask_seek)) {
        const f3 desired = mk3(G.goal[0], G.goal[1], G.goal[2]) - pos;
        const f3 f = (MODE == GS_MODE_GPUREF) ? normalize3(desired - fwd) : desired - fwd * speed;
        apply(steering, bits, f, P.w_seek, GS_BIT_SEEK);
    }
    f3 side = ld3(A.sx, A.sy, A.sz, i), up = ld3(A.ux, A.uy, A.uz, i);
    f3 sacc = ld3(A.ax, A.ay, A.az, i);
    integrate<MODE>(steering, pos, fwd, speed, sacc, side, up, A.max_force[i], A.max_speed[i], A.mass[i], P.dt);
    st3(G.npx, G.npy, G.npz, i, pos);
    st3(G.nfx, G.nfy, G.nfz, i, fwd);
    st3(A.sx, A.sy, A.sz, i, side);
    st3(A.ux, A.uy, A.uz, i, up);
    if (MODE == GS_MODE_OPENSTEER) st3(A.ax, A.ay, A.az, i, sacc);
    A.speed[i] = speed;
    st3(A.gx, A.gy, A.gz, i, mk3(0.f, 0.f, 0.f));
    A.bits[i] = 0u;
}

void launch_pair_steer(gs_group_s* const g[2], gs_group_s* W, gs_group_s* O, gs_knn_s* const knn[8],
                       const gs_scenario* s) {
    PairSteer P{};
    uint32_t n = 0;
    for (int i = 0; i < 2; ++i) {
        PairAgents& a = P.a[i];
        a.n = g[i]->n;
        n = std::max(n, a.n);
        a.kown = knn[4 * i]->idx();
        a.kother = knn[4 * i + 1]->idx();
        a.kwalls = knn[4 * i + 2]->idx();
        a.kobs = knn[4 * i + 3]->idx();
        for (int j = 0; j < 4; ++j) a.k[j] = knn[4 * i + j]->k;
        for (int j = 0; j < 3; ++j) a.goal[j] = s->goal[i][j];
    }
    // Where the next kernel reads and writes positions and forward vectors.
    auto state = [&] {
        for (int i = 0; i < 2; ++i) {
            PairAgents& a = P.a[i];
            a.A = g[i]->dev_agents();
            float** out[6] = {&a.npx, &a.npy, &a.npz, &a.nfx, &a.nfy, &a.nfz};
            for (int j = 0; j < 6; ++j) *out[j] = g[i]->Falt(j);
        }
    };
    auto written = [&] {
        for (int i = 0; i < 2; ++i)
            for (int j = 0; j < 6; ++j) g[i]->flip(j);
    };
    P.spos1 = g[1]->spos.p;
    P.nW = W->n;
    P.nO = O->n;
    const int f0 = kWallField;
    P.W = gs_walls{W->F(f0),     W->F(f0 + 1), W->F(f0 + 2), W->F(f0 + 3), W->F(f0 + 4),
                   W->F(f0 + 5), W->F(f0 + 6), W->F(f0 + 7), W->F(f0 + 8)};
    P.ox = O->F(0);
    P.oy = O->F(1);
    P.oz = O->F(2);
    P.orad = O->F(19);
    P.mt_walls = s->walls_min_time;
    P.w_walls = s->walls_weight;
    P.mt_obs = s->obstacles_min_time;
    P.w_obs = s->obstacles_weight;
    P.w_seek = s->seek_weight;
    P.mask_seek = s->seek_mask;
    P.dt = s->dt;
    const gs_flock_term& t = s->choke_separation;
    P.sep = FlockTerm{t.min_d, t.max_d, t.cos_max, t.weight, t.mask, 1};
    hipStream_t st = g[0]->ctx->stream;
    const unsigned block = agent_block(n);
    const dim3 grid(agent_blocks(n), 2);
    state();
    k_pair_avoid<<<grid, block, 0, st>>>(P);
    GS_LAUNCHED("k_pair_avoid");
    written();
    state();
    if (s->mode == GS_MODE_GPUREF) k_pair_finish<GS_MODE_GPUREF><<<grid, block, 0, st>>>(P);
    else k_pair_finish<GS_MODE_OPENSTEER><<<grid, block, 0, st>>>(P);
    GS_LAUNCHED("k_pair_finish");
    written();
    for (int i = 0; i < 2; ++i) {
        g[i]->mark_written(kFSteer | 0x3Fu, true);
        g[i]->mark_integrated();
    }
}

}  // namespace gs
