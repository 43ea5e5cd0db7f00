// Brute-force exact KNN: every point of B against every query of A, on the
// matrix cores.
//
// The squared distance of query q and point p, less |q|^2, is the dot product
// of (-2 qx, -2 qy, -2 qz, 1) and (px, py, pz, |p|^2): a K = 4 product, one
// v_mfma_f32_16x16x4f32 for 16 points x 16 queries.  Its rounding is not that
// of the key's d2, so the matrix only decides which pairs are worth a key:
//
//   bound   one pass keeps, per query, the smallest product of each of 64
//           disjoint groups of points; the (k + 1)-th smallest of those (one
//           may be the query itself) bounds the k-th distance from above
//   filter  a second pass collects the slots of the points within the bound
//   select  a wavefront per query forms the exact keys (d2 bits, agent
//           index) of the few collected points and ranks them
//
// Error bounds.  Positions are taken relative to a point of B (c), u = 2^-24.
// A product errs by at most 2^-20 (|q|^2 + |p|^2) (its eight roundings and
// those of |p|^2, and of the subtraction of c).  |p|^2 is scaled by 1 - e,
// e = 2^-18, which makes every product an under-estimate by more than that in
// |p|^2; with |p|^2 <= 2 |q|^2 + 2 d2 a group's smallest product t gives
//   d2 <= (t + |q|^2 + 2^-16 |q|^2 + 2^-100) (1 + 2^-15) =: lim
// (2^-100: the matrix cores may take subnormal numbers as 0),
// and every point with d2 <= lim has a product of at most
//   lim (1 + 2^-16) - |q|^2 (1 - e) + 2^-100.
// Points and queries that are not finite, or so far from c that a square could
// overflow, pass the filter against everything.  A query with more
// collected points than its buffer holds (ties, such points, a bound that the
// distance from c makes loose) is searched again by its wavefront, exactly.
//
// Layout: a block of 16 wavefronts takes 16 T queries; wavefront w reads the
// 64-point chunks w, w + 16, ... once per pass, puts (p, |p|^2) into the
// operand's layout through LDS, and reuses it for the T query tiles.
//
// 16,384 queries x 16,384 points are 2 x 2^20 matrix instructions of 32 cycles
// on 1,024 SIMDs, 27 us; measured 103 us, the rest being the minima and
// compares of the products (four per instruction and lane) and the staging,
// which four wavefronts per SIMD overlap only in part.  One lane per query with
// a serial insertion per pair takes 2,148 us (64 blocks on 256 CUs); few points
// for many queries are still searched that way (brute_by_lanes).
#include <algorithm>

#include "gs_knn_core.hpp"

namespace gs {

constexpr int kBruteWaves = 16;
constexpr int kBruteThreads = 64 * kBruteWaves;
constexpr int kBruteCap = 128;     // collected slots per query (two per lane)
constexpr int kBruteGroups = 64;   // groups of the bound: 4 lanes x 16 wavefronts
static_assert(GS_MAX_K + 1 <= kBruteGroups, "the bound needs k + 1 groups");
static_assert(kBruteCap >= kBruteGroups && kBruteCap >= 64 + (int)GS_MAX_K, "buffer sizes");

typedef float v4f __attribute__((ext_vector_type(4)));

// Orders a wavefront's LDS accesses.
__device__ __forceinline__ void wave_fence() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The k smallest of cnt <= kBruteCap entries to the front, sorted (by the
// whole wavefront; keys are distinct).
__device__ __forceinline__ int brute_reduce(uint64_t* key, uint32_t* slot, int cnt, uint32_t k) {
    const int lane = (int)(threadIdx.x & 63u);
    wave_fence();
    uint64_t mk[2];
    uint32_t ms[2], r[2] = {0u, 0u};
#pragma unroll
    for (int e = 0; e < 2; ++e) {
        const int i = lane + 64 * e;
        mk[e] = i < cnt ? key[i] : ~0ull;
        ms[e] = i < cnt ? slot[i] : 0u;
    }
#pragma unroll 4
    for (int f = 0; f < cnt; ++f) {
        const uint64_t o = key[f];
        r[0] += o < mk[0] ? 1u : 0u;
        r[1] += o < mk[1] ? 1u : 0u;
    }
    wave_fence();
#pragma unroll
    for (int e = 0; e < 2; ++e)
        if (lane + 64 * e < cnt && r[e] < k) {
            key[r[e]] = mk[e];
            slot[r[e]] = ms[e];
        }
    wave_fence();
    return min(cnt, (int)k);
}

template <int T>
__global__ __launch_bounds__(kBruteThreads) void k_knn_brute(
    uint32_t nA, const float* __restrict__ ax, const float* __restrict__ ay, const float* __restrict__ az, uint32_t nB,
    const float* __restrict__ bx, const float* __restrict__ by, const float* __restrict__ bz,
    const uint32_t* __restrict__ bids, int self, uint32_t k, float cap2, uint32_t* __restrict__ out_idx,
    float* __restrict__ out_dist) {
    constexpr int Q = 16 * T;
    constexpr float huge = 0x1p120f;  // squared distances from c beyond this are special
    // The group minima of the bound, then the collected slots.
    __shared__ uint32_t lds_slot[Q * kBruteCap];
    __shared__ v4f lds_point[kBruteThreads];  // per wavefront 64 points, later 128 keys
    __shared__ float lds_thr[Q], lds_lim[Q];
    __shared__ uint32_t lds_cnt[Q];
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint32_t col = lane & 15u, comp = lane >> 4;
    const uint32_t q0 = blockIdx.x * Q;
    float cx = 0.f, cy = 0.f, cz = 0.f;
    if (nB > 0) {
        const uint32_t m = nB / 2;
        const float x = bx[m], y = by[m], z = bz[m];
        if (fabsf(x) < 0x1p60f && fabsf(y) < 0x1p60f && fabsf(z) < 0x1p60f) cx = x, cy = y, cz = z;
    }
    // |q|^2 relative to c; not below huge (or NaN): special.
    auto q2_of = [&](uint32_t q, float& x, float& y, float& z) {
        const bool in = q < nA;
        x = in ? ax[q] - cx : 0.f;
        y = in ? ay[q] - cy : 0.f;
        z = in ? az[q] - cz : 0.f;
        return __builtin_fmaf(x, x, __builtin_fmaf(y, y, z * z));
    };
    float qop[T];  // the query operand of each tile
#pragma unroll
    for (int t = 0; t < T; ++t) {
        float x, y, z;
        const float q2 = q2_of(q0 + t * 16 + col, x, y, z);
        const float v = comp == 0 ? -2.f * x : (comp == 1 ? -2.f * y : (comp == 2 ? -2.f * z : 1.f));
        qop[t] = (q2 < huge || comp == 3) ? v : 0.f;
    }
    v4f* const pts = lds_point + wave * 64;
    const float* const ptf = (const float*)pts;
    const uint32_t chunks = (nB + 63u) / 64u;
    // This lane's point of the chunk to come, loaded one chunk ahead.
    float nx, ny, nz;
    auto fetch = [&](uint32_t c) {
        const uint32_t b = min(c * 64u + lane, nB - 1u);
        nx = bx[b];
        ny = by[b];
        nz = bz[b];
    };
    // Point operands of the fetched chunk c: `special` is the |p|^2 entry of
    // special points (0 coordinates, so the product is that entry for every
    // query).
    float pop[4];
    auto stage_chunk = [&](uint32_t c, float special) {
        const float x = nx - cx, y = ny - cy, z = nz - cz;
        if (c + kBruteWaves < chunks) fetch(c + kBruteWaves);
        const float p2 = __builtin_fmaf(x, x, __builtin_fmaf(y, y, z * z));
        v4f p = {0.f, 0.f, 0.f, special};
        if (p2 < huge) p = v4f{x, y, z, p2 * (1.f - 0x1p-18f)};
        if (c * 64u + lane >= nB) p = v4f{0.f, 0.f, 0.f, INFINITY};  // past the end: beyond every bound
        wave_fence();
        pts[lane] = p;
        wave_fence();
#pragma unroll
        for (int m = 0; m < 4; ++m) pop[m] = ptf[(m * 16 + col) * 4 + comp];
    };
    // ---- bound
    {
        float least[T];
#pragma unroll
        for (int t = 0; t < T; ++t) least[t] = INFINITY;
        if (wave < chunks) fetch(wave);
        for (uint32_t c = wave; c < chunks; c += kBruteWaves) {
            stage_chunk(c, INFINITY);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                v4f d[4];
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    d[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(pop[m], qop[t], v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    least[t] = fminf(least[t], fminf(fminf(d[m].x, d[m].y), fminf(d[m].z, d[m].w)));
            }
        }
        float* group = (float*)lds_slot;
#pragma unroll
        for (int t = 0; t < T; ++t) group[(t * 16 + col) * kBruteGroups + wave * 4 + comp] = least[t];
        __syncthreads();
        const uint32_t need = self ? k : k - 1u;  // rank of the bounding group
        float lim[T], thr[T];
#pragma unroll
        for (int t = 0; t < T; ++t) {
            const uint32_t q = wave * T + t;
            const float v = group[q * kBruteGroups + lane];
            uint32_t r = 0;
#pragma unroll 4
            for (uint32_t j = 0; j < (uint32_t)kBruteGroups; j += 4) {
                const v4f o = *(const v4f*)(group + q * kBruteGroups + j);
#pragma unroll
                for (uint32_t i = 0; i < 4; ++i) r += (o[i] < v || (o[i] == v && j + i < lane)) ? 1u : 0u;
            }
            const float tk = __shfl(v, __ffsll((unsigned long long)__ballot(r == need)) - 1, 64);
            float x, y, z;
            const float q2 = q2_of(q0 + q, x, y, z);
            lim[t] = thr[t] = INFINITY;
            if (q2 < huge && tk < INFINITY) {
                lim[t] = fminf(cap2, (fmaxf((tk + q2) + q2 * 0x1p-16f, 0.f) + 0x1p-100f) * (1.f + 0x1p-15f));
                thr[t] = (lim[t] * (1.f + 0x1p-16f) - q2 * (1.f - 0x1p-18f)) + 0x1p-100f;
            } else {
                lim[t] = cap2;
            }
        }
        __syncthreads();  // the minima are read; their space becomes the slots
        if (lane == 0) {
#pragma unroll
            for (int t = 0; t < T; ++t) {
                lds_lim[wave * T + t] = lim[t];
                lds_thr[wave * T + t] = thr[t];
                lds_cnt[wave * T + t] = 0u;
            }
        }
        __syncthreads();
    }
    // ---- filter
    {
        float thr[T];
#pragma unroll
        for (int t = 0; t < T; ++t) thr[t] = lds_thr[t * 16 + col];
        if (wave < chunks) fetch(wave);
        for (uint32_t c = wave; c < chunks; c += kBruteWaves) {
            stage_chunk(c, -INFINITY);
#pragma unroll
            for (int t = 0; t < T; ++t) {
                v4f d[4];
#pragma unroll
                for (int m = 0; m < 4; ++m)
                    d[m] = __builtin_amdgcn_mfma_f32_16x16x4f32(pop[m], qop[t], v4f{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
                float least[4];
#pragma unroll
                for (int m = 0; m < 4; ++m) least[m] = fminf(fminf(d[m].x, d[m].y), fminf(d[m].z, d[m].w));
                if (!__any(!(fminf(fminf(least[0], least[1]), fminf(least[2], least[3])) > thr[t]))) continue;
                const uint32_t q = t * 16 + col;
#pragma unroll
                for (int m = 0; m < 4; ++m) {
                    if (least[m] > thr[t]) continue;
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        const uint32_t b = c * 64u + m * 16u + comp * 4u + i;
                        if (!(d[m][i] > thr[t]) && b < nB && !(self && b == q0 + q)) {
                            const uint32_t at = atomicAdd(&lds_cnt[q], 1u);
                            if (at < (uint32_t)kBruteCap) lds_slot[q * kBruteCap + at] = b;
                        }
                    }
                }
            }
        }
        __syncthreads();
    }
    // ---- select: a wavefront's T queries one after another, their collected
    // points' loads all in flight first
    uint64_t* const key = (uint64_t*)pts;  // this wavefront's own points: 128 keys
    uint32_t first[T], got[T];
    float fx[T], fy[T], fz[T];
    uint32_t fid[T];
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const uint32_t ql = wave * T + t;
        got[t] = q0 + ql < nA ? lds_cnt[ql] : 0u;
        first[t] = lane < min(got[t], (uint32_t)kBruteCap) ? lds_slot[ql * kBruteCap + lane] : 0u;
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        if (nB == 0) continue;
        fx[t] = bx[first[t]];
        fy[t] = by[first[t]];
        fz[t] = bz[first[t]];
        fid[t] = bids[first[t]];
    }
#pragma unroll
    for (int t = 0; t < T; ++t) {
        const uint32_t ql = wave * T + t, q = q0 + ql;
        if (q >= nA) break;
        uint32_t* const slot = lds_slot + ql * kBruteCap;
        const float qx = ax[q], qy = ay[q], qz = az[q];
        float lim = lds_lim[ql];
        int cnt = 0;
        // Adds each lane's point (when it has one) with d2 <= lim.
        uint64_t worst = ~0ull;  // the k-th key once k are known: most ties lie beyond it
        auto add = [&](bool has, uint32_t b, float x, float y, float z, uint32_t id) {
            const float d2 = sqdist(qx, qy, qz, x, y, z);
            const uint64_t mk = make_key(d2, id);
            const bool pass = has && d2 <= lim && mk <= worst;
            const uint64_t v = __ballot(pass);
            if (pass) {
                const int at = cnt + __popcll(v & ((1ull << lane) - 1ull));
                key[at] = mk;
                slot[at] = b;
            }
            cnt += __popcll(v);
        };
        if (got[t] <= (uint32_t)kBruteCap) {
            const bool more = got[t] > 64u;
            const bool has = more && lane + 64u < got[t];
            const uint32_t b = has ? slot[lane + 64u] : 0u;
            wave_fence();
            add(lane < got[t], first[t], fx[t], fy[t], fz[t], fid[t]);
            if (more) add(has, b, bx[b], by[b], bz[b], bids[b]);
        } else {
            for (uint32_t b0 = 0; b0 < nB; b0 += 64u) {
                const uint32_t b = min(b0 + lane, nB - 1u);
                add(b0 + lane < nB && !(self && b == q), b, bx[b], by[b], bz[b], bids[b]);
                if (cnt + 64 > kBruteCap) {
                    cnt = brute_reduce(key, slot, cnt, k);
                    if (cnt == (int)k) worst = key[k - 1u];
                }
            }
        }
        cnt = brute_reduce(key, slot, cnt, k);
        if (lane < k) {
            const size_t o = (size_t)lane * nA + q;
            const bool pad = (int)lane >= cnt;
            out_idx[o] = pad ? UINT32_MAX : slot[lane];
            out_dist[o] = pad ? FLT_MAX : sqrtf(__uint_as_float((uint32_t)(key[lane] >> 32)));
        }
        wave_fence();
    }
}

// One lane per query, B staged through LDS in tiles of one block (positions and
// agent indices).  Bound by the serial insertions of a lane, about 0.2 (k = 1)
// to 0.6 us (k = 32) per point while the chip is not full.
template <int KMAX>
__global__ __launch_bounds__(kBlock) void k_knn_brute_lanes(
    uint32_t nA, const float* __restrict__ ax, const float* __restrict__ ay, const float* __restrict__ az, uint32_t nB,
    const float* __restrict__ bx, const float* __restrict__ by, const float* __restrict__ bz,
    const uint32_t* __restrict__ bids, int self, uint32_t k, float cap2, uint32_t* __restrict__ out_idx,
    float* __restrict__ out_dist) {
    __shared__ float tx[kBlock], ty[kBlock], tz[kBlock];
    __shared__ uint32_t tid[kBlock];
    const uint32_t q = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = q < nA;
    const float qx = active ? ax[q] : 0.f, qy = active ? ay[q] : 0.f, qz = active ? az[q] : 0.f;
    TopK<KMAX> h;
    h.init(k);
    for (uint32_t base = 0; base < nB; base += kBlock) {
        const uint32_t t = base + threadIdx.x;
        if (t < nB) {
            tx[threadIdx.x] = bx[t];
            ty[threadIdx.x] = by[t];
            tz[threadIdx.x] = bz[t];
            tid[threadIdx.x] = bids[t];
        }
        __syncthreads();
        const uint32_t m = min((uint32_t)kBlock, nB - base);
        if (active) {
            for (uint32_t j = 0; j < m; ++j) {
                const uint32_t b = base + j;
                if (self && b == q) continue;
                const float d2 = sqdist(qx, qy, qz, tx[j], ty[j], tz[j]);
                const uint64_t kk = make_key(d2, tid[j]);
                if (d2 <= cap2 && h.accepts(kk)) h.push(kk, b);
            }
        }
        __syncthreads();
    }
    if (active) h.store(k, nA, q, out_idx, out_dist);
}

// Whether few points meet many queries, where a lane per query is faster: the
// matrix form spends about 1.6 us per 1,000 queries beyond 4,096 on its blocks'
// set-up and selection whatever nB, the lanes a time per point that grows with
// the list and, once the chip is full, with the queries (short lists fill it
// later).  Lanes / matrix, us, k = 7: 4,096 queries 7 / 10 at 16 points, 16 / 12
// at 50; 16,384 29 / 33 at 100, 52 / 32 at 200; 65,536 99 / 117 at 400, 178 / 120
// at 800; 131,072 38 / 235 at 100, 222 / 236 at 800; 500,000 940 / 1,038 at
// 1,600.  k = 16: 16,384 42 / 48 at 100, 78 / 60 at 200; 131,072 227 / 255 at 400,
// 422 / 256 at 800.  k = 32: 16,384 36 / 39 at 50, 65 / 48 at 100; 131,072 441 /
// 537 at 400, 880 / 294 at 800.
static bool brute_by_lanes(uint32_t nA, uint32_t nB, uint32_t k) {
    const double point = k <= 8 ? 18.0 : (k <= 16 ? 24.0 : 30.0);
    const double full = std::max(1.0, nA / 98304.0 * std::min(k + 2u, 12u) / 12.0);
    return nB * point * full <= 336.0 + (std::max(nA, 4096u) - 4096u) / 7.5;
}

void launch_knn_brute(gs_group_s* A, gs_knn_s* out, gs_group_s* B, float cap2) {
    const uint32_t nA = A->n;
    if (nA == 0) return;
    hipStream_t st = A->ctx->stream;
    const int self = A == B ? 1 : 0;
    if (brute_by_lanes(nA, B->n, out->k)) {
#define GS_BRUTE_LANES(KM)                                                                                           \
    k_knn_brute_lanes<KM><<<blocks_for(nA), kBlock, 0, st>>>(nA, A->F(0), A->F(1), A->F(2), B->n, B->F(0), B->F(1), \
                                                             B->F(2), B->ids(), self, out->k, cap2, out->idx_alt(), \
                                                             out->dist_alt())
        if (out->k <= 8) GS_BRUTE_LANES(8);
        else if (out->k <= 16) GS_BRUTE_LANES(16);
        else GS_BRUTE_LANES(32);
#undef GS_BRUTE_LANES
        GS_LAUNCHED("k_knn_brute_lanes");
        return;
    }
#define GS_BRUTE(T)                                                                                                 \
    k_knn_brute<T><<<blocks_for(nA, 16 * T), kBruteThreads, 0, st>>>(nA, A->F(0), A->F(1), A->F(2), B->n, B->F(0),   \
                                                                     B->F(1), B->F(2), B->ids(), self, out->k, cap2, \
                                                                     out->idx_alt(), out->dist_alt())
    // Four query tiles per point operand once that still gives every CU a
    // block; fewer queries take more, smaller blocks.
    if (nA <= 16u * 256u) GS_BRUTE(1);
    else if (nA <= 32u * 256u) GS_BRUTE(2);
    else GS_BRUTE(4);
#undef GS_BRUTE
    GS_LAUNCHED("k_knn_brute");
}

}  // namespace gs
