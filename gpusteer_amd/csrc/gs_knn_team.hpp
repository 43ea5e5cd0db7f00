// Exact KNN of one query by a team of G consecutive lanes of a wavefront,
// for query counts that leave the one-lane-per-query search
// (knn_search_flat) a few wavefronts per SIMD or fewer: its time is then the
// serial chain of one lane (about 45 us for 4,096 agents as for 100,000, an
// empty chip either way).  A team shares every stage of that chain: the seed's k
// neighbours and the columns of the search box are dealt to its lanes, runs
// of candidate slots are read G at a time (consecutive lanes, consecutive
// slots), and the candidates within the bound are collected in an unordered
// LDS buffer of the query.  No register list: the buffer is reduced to its k
// smallest keys by counting, for every entry, the entries below it.
//
// The keys (d2 bits, agent index), the candidate set and the exactness test
// are those of the flat search, so the lists are the same.
#pragma once
#include <type_traits>

#include "gs_knn_core.hpp"

namespace gs {

// Longest list a team keeps.
constexpr uint32_t kTeamMaxK = 16;
// Lanes per query for n queries of k neighbours.  Lanes pay while the chip is
// not full: a team costs about twice the instructions of a lane of the flat
// search per query.  Measured (us, uniform flock, seeded; flat / 8 lanes / 16
// lanes): k = 7, 16,384 queries 30.4 / 17.5 / 13.9; 32,768 32.1 / 18.2 /
// 18.6; 131,072 38.1 / 35.3 / 44.7; 262,144 50.7 / 57.5 / 77.6.  k = 16,
// 65,536 64.2 / 48.1 / 39.7; 131,072 75.7 / 63.6 / 61.9; 262,144 110 / 98.4 /
// 103; 524,288 160 / 175 / 201.  Four lanes were slower than eight
// throughout (k = 7: 24.2 us at 16,384, 60.3 at 262,144).  Near the lines a
// lane is ahead where the seed is as good as it gets, in a uniform flock at rest
// (131,072, k = 1 13 / 20, k = 4 18 / 24, k = 7 28 / 27; 262,144, k = 16 57 / 62),
// and far behind in clumps (131,072, k = 7 102 / 59) or apart from its targets
// (100,000 of 20,000, no cap 5,140 / 525, about one cluster 10,900 / 486).
constexpr uint32_t kTeam16Max = 24576, kTeam8Max = 131072;          // k <= 8
constexpr uint32_t kTeam16MaxLong = 131072, kTeam8MaxLong = 262144;  // longer lists
inline int team_lanes(uint32_t n, uint32_t k) {
    const bool wide = k > 8;
    if (n <= (wide ? kTeam16MaxLong : kTeam16Max)) return 16;
    return n <= (wide ? kTeam8MaxLong : kTeam8Max) ? 8 : 1;
}
// LDS of a block of kBlock / G queries with lists of up to KM entries and a
// first box of column radius RF.
template <int G, int KM, int RF> struct TeamLds {
    static constexpr int queries = kBlock / G;
    // The buffer holds a list and the candidates of two more chunks of G.
    static constexpr int cap = KM + 2 * G;
    // Odd strides, so that the teams of a wavefront read different banks;
    // four pad keys fit past the buffer.
    static constexpr int stride = cap + 5, best_stride = KM + 1;
    // Runs: the columns of the first box, two per lane in the rings beyond
    // it; one more is read ahead.
    static constexpr int box_columns = (2 * RF + 1) * (2 * RF + 1);
    static constexpr int runs = (2 * G > box_columns ? 2 * G : box_columns) + 1;
    uint64_t key[queries * stride];
    uint64_t best_key[queries * best_stride];
    uint2 run[queries * runs];  // first slot, length
    uint32_t slot[queries * stride];
    uint32_t best_slot[queries * best_stride];
};
template <int G> constexpr int team_queries() { return kBlock / G; }

// Orders this wavefront's LDS accesses (a team never spans wavefronts).
__device__ __forceinline__ void team_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The query's candidate buffer.  cnt, lim and k are the same in every lane of
// the team; control flow around its calls is team-uniform.
template <int G, int KM, int RF> struct TeamList {
    typedef TeamLds<G, KM, RF> Lds;
    uint64_t *key, *best_key;
    uint32_t *slot, *best_slot;
    uint2* run;
    uint32_t lane;   // within the team
    uint32_t first;  // the team's first lane in the wavefront
    uint32_t k;
    int cnt;
    float lim;  // candidates beyond it are dropped

    __device__ __forceinline__ TeamList(Lds& L, uint32_t k_) {
        const uint32_t q = threadIdx.x / G;
        key = L.key + q * Lds::stride;
        slot = L.slot + q * Lds::stride;
        best_key = L.best_key + q * Lds::best_stride;
        best_slot = L.best_slot + q * Lds::best_stride;
        run = L.run + q * Lds::runs;
        lane = threadIdx.x % G;
        first = (threadIdx.x & 63u) - lane;
        k = k_;
        cnt = 0;
        lim = INFINITY;
    }
    // Which lanes of the team hold p (bit = lane of the team).
    typedef typename std::conditional<(G > 32), uint64_t, uint32_t>::type Mask;
    __device__ __forceinline__ Mask votes(bool p) const {
        return (Mask)(__ballot(p) >> first) & ((Mask)~(Mask)0 >> (8 * sizeof(Mask) - G));
    }
    __device__ __forceinline__ static int count(Mask m) { return G > 32 ? __popcll(m) : __popc((uint32_t)m); }
    // The lanes of the mask below this one.
    __device__ __forceinline__ int rank(Mask m) const { return count(m & (((Mask)1 << lane) - 1)); }
    __device__ __forceinline__ float max_of(float v) const {
#pragma unroll
        for (int off = G / 2; off >= 1; off >>= 1) v = fmaxf(v, __shfl_xor(v, off, 64));
        return v;
    }

    __device__ __forceinline__ uint32_t sum_of(uint32_t v) const {
#pragma unroll
        for (int off = G / 2; off >= 1; off >>= 1) v += (uint32_t)__shfl_xor((int)v, off, 64);
        return v;
    }

    // The buffer's k smallest keys, sorted, in best_key / best_slot and at the
    // buffer's front, and the bound they give.  An entry's place is the number
    // of keys below its own (keys are distinct).
    __device__ __forceinline__ void reduce() {
        if (lane < 4u) key[cnt + lane] = ~0ull;  // the count reads four at a time
        team_fence();
        for (int i = (int)lane; i < cnt; i += G) {
            const uint64_t mk = key[i];
            uint32_t r = 0;
            for (int f = 0; f < cnt; f += 4) {
                uint64_t o[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) o[u] = key[f + u];
#pragma unroll
                for (int u = 0; u < 4; ++u) r += o[u] < mk ? 1u : 0u;
            }
            if (r < k) {
                best_key[r] = mk;
                best_slot[r] = slot[i];
            }
        }
        team_fence();
        cnt = min(cnt, (int)k);
        for (int i = (int)lane; i < cnt; i += G) {
            key[i] = best_key[i];
            slot[i] = best_slot[i];
        }
        if (cnt == (int)k) lim = fminf(lim, __uint_as_float((uint32_t)(best_key[k - 1u] >> 32)));
        team_fence();
    }

    // Appends each lane's run (len 0: none) to the M runs of the team.
    __device__ __forceinline__ void push_run(uint32_t t0, uint32_t len, int& M) {
        const Mask m = votes(len != 0u);
        if (len != 0u) run[M + rank(m)] = make_uint2(t0, len);
        M += count(m);
    }

    // Walks the team's M runs in chunks of G slots, four chunks in flight:
    // each(d2, ok, slot, point) gets the lane's four candidates.
    template <class F>
    __device__ __forceinline__ void walk(int M, float qx, float qy, float qz, uint32_t self,
                                         __amdgpu_buffer_rsrc_t rb, F&& each) {
        team_fence();
        int m = 0;
        uint32_t i = 0;
        uint2 r = run[0];
        while (m < M) {
            uint32_t t[4];
            bool ok[4];
            float4 p[4];
            float d2[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                t[u] = r.x + i + lane;
                ok[u] = m < M && i + lane < r.y && t[u] != self;
                i += G;
                if (m < M && i >= r.y) {
                    ++m;
                    i = 0;
                    r = run[m];  // one past the last is read, never used
                }
            }
            // Lanes past a chunk's end load slot 0; their value is not used.
#pragma unroll
            for (int u = 0; u < 4; ++u) p[u] = ld_pos(rb, ok[u] ? t[u] * 16u : 0u);
#pragma unroll
            for (int u = 0; u < 4; ++u) d2[u] = sqdist4(qx, qy, qz, p[u]);
            each(d2, ok, t, p);
        }
        team_fence();
    }

    // Collects the candidates of the M runs within the bound.
    __device__ __forceinline__ void scan(int M, float qx, float qy, float qz, uint32_t self,
                                         __amdgpu_buffer_rsrc_t rb) {
        walk(M, qx, qy, qz, self, rb, [&](const float* d2, const bool* ok, const uint32_t* t, const float4* p) {
#pragma unroll
            for (int h = 0; h < 4; h += 2) {
                const bool pa = ok[h] && d2[h] <= lim, pb = ok[h + 1] && d2[h + 1] <= lim;
                const Mask va = votes(pa), vb = votes(pb);
                if ((va | vb) == 0) continue;
                const int na = count(va), total = na + count(vb);
                if (cnt + total > Lds::cap) reduce();  // leaves at most k: the two chunks now fit
                if (pa) {
                    const int at = cnt + rank(va);
                    key[at] = make_key(d2[h], id_of(p[h]));
                    slot[at] = t[h];
                }
                if (pb) {
                    const int at = cnt + na + rank(vb);
                    key[at] = make_key(d2[h + 1], id_of(p[h + 1]));
                    slot[at] = t[h + 1];
                }
                cnt += total;
            }
        });
    }

    // Each lane's candidate, when it has one (pass).
    __device__ __forceinline__ void add(bool pass, float d2, uint32_t id, uint32_t t) {
        const Mask v = votes(pass);
        if (v == 0) return;
        if (cnt + count(v) > Lds::cap) reduce();
        if (pass) {
            const int at = cnt + rank(v);
            key[at] = make_key(d2, id);
            slot[at] = t;
        }
        cnt += count(v);
    }

    // The sorted list to column `row` of the slot-major [k][n] output (pads
    // UINT32_MAX / FLT_MAX); no distances when out_dist is NULL.
    __device__ __forceinline__ void store(uint32_t n, uint32_t row, uint32_t* __restrict__ out_idx,
                                          float* __restrict__ out_dist) const {
        for (uint32_t j = lane; j < k; j += G) {
            const size_t o = (size_t)j * n + row;
            const bool pad = (int)j >= cnt;
            out_idx[o] = pad ? UINT32_MAX : best_slot[j];
            if (out_dist) out_dist[o] = pad ? FLT_MAX : sqrtf(__uint_as_float((uint32_t)(best_key[j] >> 32)));
        }
    }

    // A bound on the k-th distance: the lanes' two nearest candidates are
    // distinct points, and the k-th nearest of them lies no nearer than the
    // k-th of all (+inf with fewer than k).  Keeps nothing in LDS, so a
    // pass over the runs costs little more than their loads.
    struct Two {
        float a = INFINITY, b = INFINITY;
    };
    __device__ __forceinline__ void nearest(Two& two, int M, float qx, float qy, float qz, uint32_t self,
                                            __amdgpu_buffer_rsrc_t rb) {
        walk(M, qx, qy, qz, self, rb, [&](const float* d2, const bool* ok, const uint32_t*, const float4*) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float d = ok[u] && d2[u] < INFINITY ? d2[u] : INFINITY;  // a NaN is no candidate
                two.b = fminf(two.b, fmaxf(two.a, d));
                two.a = fminf(two.a, d);
            }
        });
    }
    // The values are made distinct by their place in the low bits and ranked by
    // counting; the bound has those bits set, a relative 2^-16 at most above.
    __device__ __forceinline__ float kth(const Two& two) {
        constexpr uint32_t N = G > 16 ? G : 2 * G;  // wide teams: the nearest of each lane
        static_assert(KM <= (int)N && KM + (int)N / 2 <= Lds::cap, "the bound needs k values, and room for them");
        uint32_t* v = (uint32_t*)(key + cnt);  // past the collected keys (fewer than k)
        const uint32_t ua = (__float_as_uint(two.a) & ~(N - 1u)) | lane;
        const uint32_t ub = (__float_as_uint(two.b) & ~(N - 1u)) | (G + lane);
        v[lane] = ua;
        if (N > G) v[G + lane] = ub;
        team_fence();
        uint32_t ra = 0, rb = 0;
#pragma unroll
        for (uint32_t j = 0; j < N / 2; ++j) {
            const uint2 o = ((const uint2*)v)[j];
            ra += (o.x < ua ? 1u : 0u) + (o.y < ua ? 1u : 0u);
            if (N > G) rb += (o.x < ub ? 1u : 0u) + (o.y < ub ? 1u : 0u);
        }
        team_fence();
        uint32_t u = 0u;
        if (ra == k - 1u) u = ua | (N - 1u);
        if (N > G && rb == k - 1u) u = ub | (N - 1u);
        return max_of(u < 0x7F800000u ? __uint_as_float(u) : INFINITY);
    }
};

// Largest d2 to the k neighbours of the previous exact result (seed_bound's
// value, the neighbours dealt to the team's lanes), +inf when incomplete or
// when one is at no distance (NaN).
template <int G, int KM, int RF>
__device__ __forceinline__ float team_seed_bound(const TeamList<G, KM, RF>& L, bool active,
                                                 const uint32_t* __restrict__ seed, uint32_t nA, uint32_t row,
                                                 uint32_t nB, const uint32_t* __restrict__ val_map, float qx, float qy,
                                                 float qz, const float4* __restrict__ bpos) {
    float m = 0.f;
    bool bad = false;
    for (uint32_t j = L.lane; active && j < L.k; j += G) {
        uint32_t v = seed[(size_t)j * nA + row];
        if (v >= nB) {
            bad = true;
        } else {
            if (val_map) v = val_map[v];
            const float d2 = sqdist4(qx, qy, qz, bpos[v]);
            m = fmaxf(m, d2);
            bad = bad || (d2 != d2 && qx == qx && qy == qy && qz == qz);
        }
    }
    m = L.max_of(m);
    return L.votes(bad) ? INFINITY : m;
}

// Exact top-k of the team's query among B's points (Q, bpos, bstart as for
// knn_search_flat; 1 <= nB < kFlatMaxPoints, k <= KM); RF is the first
// box's column radius (1: 3 x 3, 2: 5 x 5 for lattices finer than the
// neighbour distance).  Leaves the sorted list in L.  Called by every lane of
// the wavefront; teams without a query pass active = false.  bound_first: the
// box is walked twice, for a bound, then for the candidates within it.
//
// Local: false when the next box would have more columns than max_columns or more
// cells than there are points, or when a ring's runs hold more than
// kLocalCandidates; L.lim is then a bound on the k-th d2 (at most Q.thr) and the
// list is to be found another way.
constexpr uint32_t kLocalCandidates = 256;
template <bool Local, int G, int KM, int RF>
__device__ __forceinline__ bool knn_search_team(TeamList<G, KM, RF>& L, const FlatQuery& Q, const GridDev& g,
                                                uint32_t nB, const float4* __restrict__ bpos,
                                                const uint32_t* __restrict__ bstart, bool bound_first,
                                                int max_columns = 0) {
    const __amdgpu_buffer_rsrc_t rb = pos_rsrc(bpos, nB);
    const float grow = 1.0f + 2e-5f;
    const float qx = Q.x, qy = Q.y, qz = Q.z;
    L.cnt = 0;
    L.lim = Q.thr;
    if (!Q.active || Q.thr < 0.f) return true;  // the whole team
    const int cx = axis_cell_bound(qx, g.ox, g.rx, g.dx);
    const int cy = axis_cell_bound(qy, g.oy, g.ry, g.dy);
    const int cz = axis_cell_bound(qz, g.oz, g.rz, g.dz);
    // First the box of ring RF, one run per column; then larger boxes (R cells
    // each way in x and y, R * zr in z), a column per lane and round: a column
    // outside the box before (ring Rin) is one run, the others the two runs
    // above and below it.
    int R = RF, Rin = RF, M = 0;
    for (;; bound_first = false) {
        constexpr int W = 2 * RF + 1, rounds = (W * W + G - 1) / G;
        const float bound = L.lim * grow;
        const int zlo = max(cz - RF * g.zr, 0), zhi = min(cz + RF * g.zr, g.dz - 1);
        uint2 r[rounds];
#pragma unroll
        for (int i = 0; i < rounds; ++i) {
            const int c = i * G + (int)L.lane;
            const int ix = cx + c / W - RF, iy = cy + c % W - RF;
            const bool valid = c < W * W && ix >= 0 && ix < g.dx && iy >= 0 && iy < g.dy;
            const float gx = axis_gap(qx, ix, ix, g.ox, g.hx, g.dx, g.slack);
            const float gy = axis_gap(qy, iy, iy, g.oy, g.hy, g.dy, g.slack);
            r[i] = flat_column_run(valid, gx * gx + gy * gy, bound, grow, qz, zlo, zhi,
                                   (uint32_t)(ix * g.dy * g.dz + iy * g.dz), g, bstart);
        }
        M = 0;
#pragma unroll
        for (int i = 0; i < rounds; ++i) L.push_run(r[i].x, r[i].y - r[i].x, M);
        if (!bound_first) break;
        typename TeamList<G, KM, RF>::Two two;
        L.nearest(two, M, qx, qy, qz, Q.self, rb);
        L.lim = fminf(L.lim, L.kth(two));
    }
    int c0 = 0, columns = 0;
    bool last = false;  // nothing is left to scan after the runs at hand
    for (;;) {
        L.scan(M, qx, qy, qz, Q.self, rb);
        M = 0;
        if (c0 >= columns) {
            L.reduce();
            bool all;
            const float dmin = outside_gap(g, cx, cy, cz, R, qx, qy, qz, all);
            if (last || all || exact_after(L.lim, dmin)) return true;
            // One ring more, then boxes of twice the extent, as far as the
            // bound reaches: a target far away or a cap without k points
            // under it is reached in a few rounds.  Ring by ring every step
            // was a test, a reduction and two dependent loads (a step of 24
            // scenarios, 220,000 agents: 0.32 -> 0.23 ms).
            Rin = R;
            R = R == RF ? R + 1 : 2 * R;
            if (Rin != RF && L.lim < INFINITY) {
                float h = INFINITY;
                if (g.dx > 1) h = fminf(h, g.hx);
                if (g.dy > 1) h = fminf(h, g.hy);
                if (g.dz > 1) h = fminf(h, g.hz * (float)g.zr);
                const float need = (__builtin_amdgcn_sqrtf(L.lim) * grow + g.slack) * __builtin_amdgcn_rcpf(h);
                if (need < (float)R) R = max(Rin + 1, (int)need + 1);
            }
            const uint32_t tlo = bstart[0], thi = bstart[(uint32_t)g.dx * (uint32_t)g.dy * (uint32_t)g.dz];
            if (box_beyond_points(g, R, thi - tlo)) {
                if (Local) return false;
                // More cells than points: every point again, the list's own
                // among them (they lie within the bound).
                L.cnt = 0;
                last = true;
                L.push_run(tlo, L.lane == 0 ? thi - tlo : 0u, M);
                continue;
            }
            columns = (min(cx + R, g.dx - 1) - max(cx - R, 0) + 1) * (min(cy + R, g.dy - 1) - max(cy - R, 0) + 1);
            if (Local && columns > max_columns) return false;
            c0 = 0;
        }
        const int Z = R * g.zr, Zin = Rin * g.zr;
        const int x0 = max(cx - R, 0), y0 = max(cy - R, 0), ny = min(cy + R, g.dy - 1) - y0 + 1;
        for (; M == 0 && c0 < columns; c0 += G) {
            const int c = c0 + (int)L.lane;
            const int ix = x0 + c / ny, iy = y0 + c % ny;
            const bool valid = c < columns;
            const bool edge = abs(ix - cx) > Rin || abs(iy - cy) > Rin;
            const float gx = axis_gap(qx, ix, ix, g.ox, g.hx, g.dx, g.slack);
            const float gy = axis_gap(qy, iy, iy, g.oy, g.hy, g.dy, g.slack);
            const float gxy = gx * gx + gy * gy;
            const float bound = L.lim * grow;
            const uint32_t base = (uint32_t)(ix * g.dy * g.dz + iy * g.dz);
            const uint2 lo = flat_column_run(valid, gxy, bound, grow, qz, max(cz - Z, 0),
                                             min(edge ? cz + Z : cz - Zin - 1, g.dz - 1), base, g, bstart);
            const uint2 hi = flat_column_run(valid && !edge, gxy, bound, grow, qz, max(cz + Zin + 1, 0),
                                             min(cz + Z, g.dz - 1), base, g, bstart);
            if (Local && L.sum_of((lo.y - lo.x) + (hi.y - hi.x)) > kLocalCandidates) return false;
            L.push_run(lo.x, lo.y - lo.x, M);
            L.push_run(hi.x, hi.y - hi.x, M);
        }
    }
}

}  // namespace gs
