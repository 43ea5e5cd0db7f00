// Bin database build: counting sort of a group's points by lattice cell, and
// the physical reorder of the group's state into that order.
//
// Replaces KNNBinningV2UpdateDBCUDA::run (include/OpenSteer/CUDA/KNNBinningV2.cu:87-162):
// BuildDB (cell key per agent, KNNBinningV2Kernel.cu:269-296), thrust::sort_by_key
// (:127-129), the cellStart memset (:132) and ReorderDB (KNNBinningV2Kernel.cu:314-379).
//
// Passes (all over storage slots, coalesced):
//   1. key      cell per point + atomic arrival rank within the cell (+ optional wrap)
//   2. scan     exclusive scan of the per-cell counts -> start[C+1]; clears counts
//   3. scatter  id_tmp[start[cell] + rank] = agent index (the arrival order);
//               with pass 2 in one block for small groups and lattices, left
//               out where the order inside a cell is free (k_reorder_free)
//   4. reorder  per old slot: its final slot puts the members of each cell in
//               ascending agent index (a stable sort by cell, as thrust's);
//               every live field, the bits and the agent index are written
//               there in the alternate buffers, with the old <-> new maps.
// Because the previous build left the state in cell order and agents move
// little between builds, the reorder's writes land nearly sequentially.  The
// counts array is all-zero between builds (pass 2 clears it), so no memset is
// recorded in the stream.
#include <algorithm>

#include "gs_internal.hpp"

namespace gs {

// Members of a cell are put in ascending agent index (the stable sort's
// order) by counting, for each member, the members with a smaller index: m
// reads per member of an m-member cell, issued by all members at once.
// Cells with more members than this keep the atomic arrival order instead
// (KNN results never depend on the order inside a cell; the per-cell
// velocity sum of such a cell does).
constexpr uint32_t kCanonCap = 65536;
constexpr int kScanItems = 8;
constexpr int kScanTile = kBlock * kScanItems;  // 2048 cells per scan block

__global__ __launch_bounds__(kBlock) void k_fill_u32(uint32_t* __restrict__ p, uint32_t n, uint32_t v) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = v;
}

__global__ __launch_bounds__(kBlock) void k_iota(uint32_t* __restrict__ p, uint32_t n) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = i;
}

__global__ __launch_bounds__(kBlock) void k_invert(uint32_t n, const uint32_t* __restrict__ ids,
                                                   uint32_t* __restrict__ slot_of_id) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < n) slot_of_id[ids[s]] = s;
}

void launch_invert_ids(gs_group_s* g) {
    if (g->n == 0) return;
    k_invert<<<blocks_for(g->n), kBlock, 0, g->ctx->stream>>>(g->n, g->ids(), g->slot_of_id.p);
    GS_LAUNCHED("k_invert");
}

void launch_fill_u32(uint32_t* p, uint32_t n, uint32_t v, hipStream_t st) {
    if (n == 0) return;
    k_fill_u32<<<blocks_for(n), kBlock, 0, st>>>(p, n, v);
    GS_LAUNCHED("k_fill_u32");
}

void launch_iota(uint32_t* p, uint32_t n, hipStream_t st) {
    if (n == 0) return;
    k_iota<<<blocks_for(n), kBlock, 0, st>>>(p, n);
    GS_LAUNCHED("k_iota");
}

__device__ __forceinline__ void bin_key(uint32_t n, float* __restrict__ px, float* __restrict__ py,
                                        float* __restrict__ pz, const GridDev& g, uint32_t* __restrict__ key,
                                        uint32_t* __restrict__ rank, uint32_t* __restrict__ count, int wrap_shape,
                                        float wcx, float wcy, float wcz, float wsx, float wsy, float wsz,
                                        uint32_t* __restrict__ box_acc, uint32_t* __restrict__ box_clear) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    const bool active = i < n;
    const int lane = threadIdx.x & 63;
    // Inactive lanes get a key no cell has, so they form segments of their own.
    uint32_t c = 0xFFFFFFC0u | (uint32_t)lane;
    float x = 0.f, y = 0.f, z = 0.f;
    if (active) {
        x = px[i], y = py[i], z = pz[i];
        const float x0 = x, y0 = y, z0 = z;
        wrap_point(wrap_shape, wcx, wcy, wcz, wsx, wsy, wsz, x, y, z);
        // Only wrapped coordinates are written back.
        if (__float_as_uint(x) != __float_as_uint(x0)) px[i] = x;
        if (__float_as_uint(y) != __float_as_uint(y0)) py[i] = y;
        if (__float_as_uint(z) != __float_as_uint(z0)) pz[i] = z;
        c = cell_index(g, axis_cell(x, g.ox, g.sx, g.dx), axis_cell(y, g.oy, g.sy, g.dy),
                       axis_cell(z, g.oz, g.sz, g.dz));
        key[i] = c;
    }
    count_and_rank(active, c, i, count, rank);
    if (box_acc) {
        // The bounding box of the positions this build snapshots (after the
        // wrap); the other buffer is cleared for the next build.
        if (blockIdx.x == 0 && threadIdx.x < 6) box_clear[threadIdx.x] = threadIdx.x < 3 ? kBoxEmptyMin : kBoxEmptyMax;
        box_accumulate(active, x, y, z, box_acc);
    }
}

__global__ __launch_bounds__(kBlock) void k_bin_key(uint32_t n, float* px, float* py, float* pz, GridDev g,
                                                    uint32_t* key, uint32_t* rank, uint32_t* count, int wrap_shape,
                                                    float wcx, float wcy, float wcz, float wsx, float wsy, float wsz,
                                                    uint32_t* box_acc, uint32_t* box_clear) {
    bin_key(n, px, py, pz, g, key, rank, count, wrap_shape, wcx, wcy, wcz, wsx, wsy, wsz, box_acc, box_clear);
}

// Wavefront-then-block exclusive scan of one value per thread.
__device__ __forceinline__ uint32_t block_exclusive_scan(uint32_t v, uint32_t* lds_wave, uint32_t& total) {
    const int lane = threadIdx.x & 63;
    const int wave = threadIdx.x >> 6;
    uint32_t inc = v;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(inc, d, 64);
        if (lane >= d) inc += t;
    }
    if (lane == 63) lds_wave[wave] = inc;
    __syncthreads();
    uint32_t wave_off = 0, sum = 0;
#pragma unroll
    for (int w = 0; w < kBlock / 64; ++w) {
        const uint32_t s = lds_wave[w];
        if (w < wave) wave_off += s;
        sum += s;
    }
    total = sum;
    return wave_off + inc - v;
}

// Pass 2a: each block scans kScanTile counts locally, writes local offsets
// into start and its tile sum into partial[block].
__global__ __launch_bounds__(kBlock) void k_scan_tiles(uint32_t C, const uint32_t* __restrict__ count,
                                                       uint32_t* __restrict__ start, uint32_t* __restrict__ partial) {
    __shared__ uint32_t lds[kBlock / 64];
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile + (uint64_t)threadIdx.x * kScanItems;
    uint32_t v[kScanItems];
    uint32_t sum = 0;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        v[j] = (base + j < C) ? count[base + j] : 0u;
        sum += v[j];
    }
    uint32_t total;
    uint32_t off = block_exclusive_scan(sum, lds, total);
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        if (base + j < C) start[base + j] = off;
        off += v[j];
    }
    if (threadIdx.x == 0) partial[blockIdx.x] = total;
}

// Pass 2b (many tiles): one block scans the tile sums in place (exclusive)
// and writes the grand total to start[C].
__global__ __launch_bounds__(kBlock) void k_scan_partials(uint32_t nparts, uint32_t* __restrict__ partial,
                                                          uint32_t* __restrict__ start, uint32_t C) {
    __shared__ uint32_t lds[kBlock / 64];
    uint32_t carry = 0;
    for (uint32_t base = 0; base < nparts; base += kBlock) {
        const uint32_t i = base + threadIdx.x;
        const uint32_t v = i < nparts ? partial[i] : 0u;
        uint32_t total;
        const uint32_t ex = block_exclusive_scan(v, lds, total);
        if (i < nparts) partial[i] = carry + ex;
        carry += total;
        __syncthreads();
    }
    if (threadIdx.x == 0) start[C] = carry;
}

// Pass 2c: add the tile offsets and clear the counts for the next build.
// With few tiles (fused = 1) each block sums the tile totals before its own
// tile itself, which saves the launch of pass 2b; the last block then writes
// the grand total to start[C].
constexpr uint32_t kScanFusedTiles = 1024;
__global__ __launch_bounds__(kBlock) void k_scan_add(uint32_t C, const uint32_t* __restrict__ partial,
                                                     uint32_t* __restrict__ start, uint32_t* __restrict__ count,
                                                     int fused) {
    __shared__ uint32_t lds[kBlock / 64];
    uint32_t add;
    if (fused) {
        uint32_t part = 0;
        for (uint32_t i = threadIdx.x; i < blockIdx.x; i += kBlock) part += partial[i];
        (void)block_exclusive_scan(part, lds, add);
    } else {
        add = partial[blockIdx.x];
    }
    const uint64_t base = (uint64_t)blockIdx.x * kScanTile;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        const uint64_t c = base + (uint64_t)j * kBlock + threadIdx.x;
        if (c < C) {
            start[c] += add;
            count[c] = 0u;
        }
    }
    if (fused && blockIdx.x == gridDim.x - 1 && threadIdx.x == 0) start[C] = add + partial[blockIdx.x];
}

// Passes 2 (and 3) of a small lattice in one block: each thread scans a run of
// consecutive counts, clears them, and with n > 0 the block then scatters the
// agent indices as k_scatter does.  Bound by latency: 4,096 cells and agents
// 7.7 us, for launches of 4.7 (tiles), 4.6 (add) and 4.6 us (scatter); with
// counts read and starts written 16 bytes at a time 5.6 us, and 12,167 cells
// with 5,000 agents 13.5 -> 8.7 us.
constexpr int kScanOneThreads = 1024;
constexpr uint32_t kScanOneCells = 16 * kScanOneThreads;
constexpr uint32_t kScanOneAgents = 16 * kScanOneThreads;
// Where one block pays.  The scan alone replaces two launches by one whose time
// grows with the lattice; the scatter in it replaces a third one and adds 0.75
// us per 1,024 agents.  Whole build, us, passes in launches of their own / in
// one block: 500 agents on 12,167 cells 15.2 / 13.5, on 15,625 15.3 / 15.4;
// 4,096 on 4,096 cells 15.8 / 13.1, on 12,167 15.8 / 15.6; 6,000 on 1,728 15.2 /
// 15.3, on 8,000 16.0 / 16.1; 8,192 on 4,096 16.0 / 16.2, 16,384 on 4,096 19.3 /
// 23.0 (with the scan alone 17).
constexpr uint32_t kScanAloneCells = 12 * kScanOneThreads;
constexpr uint32_t kScatterOneAgents = 5 * kScanOneThreads, kScatterOneSum = 10 * kScanOneThreads;
static bool scatter_in_scan(uint32_t n, uint32_t C) {
    return n > 0 && n <= kScatterOneAgents && C <= kScanOneCells && n + C / 2 <= kScatterOneSum;
}
__device__ __forceinline__ void scan_one(uint32_t C, uint32_t* __restrict__ count, uint32_t* start, uint32_t n,
                                         const uint32_t* __restrict__ key, const uint32_t* __restrict__ rank,
                                         const uint32_t* __restrict__ ids, uint32_t* __restrict__ id_tmp) {
    __shared__ uint32_t lds[kScanOneThreads / 64];
    // Consecutive counts per thread, a multiple of four (16-byte accesses), at
    // most 16.
    const uint32_t per = ((C + kScanOneThreads - 1) / kScanOneThreads + 3u) & ~3u;
    const uint32_t c0 = threadIdx.x * per;
    uint4 v4[4];
    uint32_t* const v = (uint32_t*)v4;
    uint32_t sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < 16; j += 4) {
        v4[j / 4] = make_uint4(0u, 0u, 0u, 0u);
        if (j < per && c0 + j + 4u <= C) {
            v4[j / 4] = *(const uint4*)(count + c0 + j);
        } else if (j < per) {
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u) v[j + u] = c0 + j + u < C ? count[c0 + j + u] : 0u;
        }
#pragma unroll
        for (uint32_t u = 0; u < 4; ++u) sum += v[j + u];
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    uint32_t inc = sum;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
        const uint32_t t = __shfl_up(inc, d, 64);
        if (lane >= d) inc += t;
    }
    if (lane == 63) lds[wave] = inc;
    __syncthreads();
    uint32_t off = inc - sum, total = 0;
#pragma unroll
    for (int w = 0; w < kScanOneThreads / 64; ++w) {
        off += w < wave ? lds[w] : 0u;
        total += lds[w];
    }
#pragma unroll
    for (uint32_t j = 0; j < 16; j += 4) {
        uint4 o;
        o.x = off;
        o.y = o.x + v[j];
        o.z = o.y + v[j + 1];
        o.w = o.z + v[j + 2];
        off = o.w + v[j + 3];
        if (j < per && c0 + j + 4u <= C) {
            *(uint4*)(start + c0 + j) = o;
            *(uint4*)(count + c0 + j) = make_uint4(0u, 0u, 0u, 0u);
        } else if (j < per) {
            const uint32_t w[4] = {o.x, o.y, o.z, o.w};
#pragma unroll
            for (uint32_t u = 0; u < 4; ++u)
                if (c0 + j + u < C) {
                    start[c0 + j + u] = w[u];
                    count[c0 + j + u] = 0u;
                }
        }
    }
    if (threadIdx.x == 0) start[C] = total;
    if (n == 0) return;
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < n; i += kScanOneThreads) {
        const uint32_t t = start[key[i]] + rank[i];
        if (t < n) id_tmp[t] = ids[i];
    }
}

__global__ __launch_bounds__(kScanOneThreads) void k_scan_one(uint32_t C, uint32_t* count, uint32_t* start, uint32_t n,
                                                              const uint32_t* key, const uint32_t* rank,
                                                              const uint32_t* ids, uint32_t* id_tmp) {
    scan_one(C, count, start, n, key, rank, ids, id_tmp);
}

// Pass 3: the agent index of every slot of the arrival order (slot t =
// start[cell] + arrival rank), which the reorder's canonical ranks read.
__global__ __launch_bounds__(kBlock) void k_scatter(uint32_t n, const uint32_t* __restrict__ key,
                                                    const uint32_t* __restrict__ rank,
                                                    const uint32_t* __restrict__ start,
                                                    const uint32_t* __restrict__ ids, uint32_t* __restrict__ id_tmp) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    // start[key]+rank < n whenever the counts were zero before the key pass;
    // the guard keeps a corrupted count array from writing out of bounds.
    const uint32_t t = start[key[i]] + rank[i];
    if (t < n) id_tmp[t] = ids[i];
}

// Pass 4, one lane per old slot s (every read coalesced, the writes land
// near s since agents rarely change cells): the agent's arrival slot is
// t = start[cell] + rank, its final slot the cell start plus the number of
// members of its cell with a smaller agent index (id_tmp NULL: the order
// inside a cell is free, and the arrival slot is final).
__device__ __forceinline__ void reorder(uint32_t n, const uint32_t* __restrict__ rank,
                                        const uint32_t* __restrict__ id_tmp, const uint32_t* __restrict__ key,
                                        const uint32_t* __restrict__ start, const uint32_t* __restrict__ ids,
                                        uint32_t* __restrict__ ids_new, uint32_t* __restrict__ new_to_old,
                                        uint32_t* __restrict__ old_to_new, const uint32_t* __restrict__ bits,
                                        uint32_t* __restrict__ bits_new, const FieldSet& fs,
                                        float4* __restrict__ spos, float4* __restrict__ sfwd) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t c = key[s];
    const uint32_t b = start[c], e = min(start[c + 1], n);
    const uint32_t t = b + rank[s];
    if (t >= n) return;  // only after a corrupted build (see k_scatter)
    const uint32_t id = ids[s];
    uint32_t d = t;
    if (id_tmp && e - b <= kCanonCap) {
        // Eight members at a time, so that a crowded cell's reads overlap.
        uint32_t r = 0;
        for (uint32_t j = b; j < e; j += 8) {
            uint32_t o[8];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) o[u] = id_tmp[min(j + u, e - 1u)];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) r += (j + u < e && o[u] < id) ? 1u : 0u;
        }
        d = b + r;
    }
    new_to_old[d] = s;
    old_to_new[s] = d;
    ids_new[d] = id;
    if (bits) bits_new[d] = bits[s];
#pragma unroll
    for (int f = 0; f < kFields; ++f)
        if (f < fs.nf) fs.dst[f][d] = fs.src[f][s];
    // fields 0..2 (positions) are always first in the set; a lazy build also
    // snapshots forward and speed (fields 3..6, passed after them)
    spos[d] = make_float4(fs.src[0][s], fs.src[1][s], fs.src[2][s], __uint_as_float(id));
    if (sfwd) sfwd[d] = make_float4(fs.src[3][s], fs.src[4][s], fs.src[5][s], fs.src[6][s]);
}

__global__ __launch_bounds__(kBlock) void k_reorder(uint32_t n, const uint32_t* rank, const uint32_t* id_tmp,
                                                    const uint32_t* key, const uint32_t* start, const uint32_t* ids,
                                                    uint32_t* ids_new, uint32_t* new_to_old, uint32_t* old_to_new,
                                                    const uint32_t* bits, uint32_t* bits_new, FieldSet fs,
                                                    float4* spos, float4* sfwd) {
    reorder(n, rank, id_tmp, key, start, ids, ids_new, new_to_old, old_to_new, bits, bits_new, fs, spos, sfwd);
}

// The three passes of two small groups' builds on one lattice at once: group
// blockIdx.y.
struct PairBuild {
    struct One {
        uint32_t n;
        float *px, *py, *pz;
        uint32_t *key, *rank, *count, *start, *id_tmp, *ids, *ids_new, *new_to_old, *old_to_new, *box_acc, *box_clear;
        uint32_t *bits, *bits_new;
        FieldSet fs;
        float4* spos;
    } g[2];
};
__global__ __launch_bounds__(kBlock) void k_pair_key(PairBuild P, GridDev g) {
    const PairBuild::One& b = P.g[blockIdx.y];
    bin_key(b.n, b.px, b.py, b.pz, g, b.key, b.rank, b.count, -1, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, b.box_acc, b.box_clear);
}
__global__ __launch_bounds__(kScanOneThreads) void k_pair_scan(PairBuild P, uint32_t C) {
    const PairBuild::One& b = P.g[blockIdx.y];
    scan_one(C, b.count, b.start, b.n, b.key, b.rank, b.ids, b.id_tmp);
}
__global__ __launch_bounds__(kBlock) void k_pair_reorder(PairBuild P) {
    const PairBuild::One& b = P.g[blockIdx.y];
    reorder(b.n, b.rank, b.id_tmp, b.key, b.start, b.ids, b.ids_new, b.new_to_old, b.old_to_new, b.bits, b.bits_new,
            b.fs, b.spos, nullptr);
}

// Passes 2 and 4 of a lazy build whose order inside a cell is free (a step of
// a call that steps again: results never depend on it, and the call's last
// step restores the canonical order): an agent's slot is its cell's start plus
// its arrival rank, so the scatter pass is not needed, and the tile offsets
// are added here.  Bound by memory (52 bytes read and written per agent) and
// launches: 1,048,576 agents on 524,288 cells, scan_add + scatter + reorder 5.1
// + 5.3 + 21.7 us, here 20.0 us.  `off` holds each cell's offset within its scan tile and
// partial the tile sums; every block scans those itself.  Blocks past the
// agents' write the cells' starts and clear the counts.
__global__ __launch_bounds__(kBlock) void k_reorder_free(uint32_t n, uint32_t C, uint32_t ntiles,
                                                         const uint32_t* __restrict__ rank,
                                                         const uint32_t* __restrict__ key,
                                                         const uint32_t* __restrict__ off,
                                                         const uint32_t* __restrict__ partial,
                                                         const uint32_t* __restrict__ ids,
                                                         uint32_t* __restrict__ ids_new,
                                                         uint32_t* __restrict__ new_to_old,
                                                         uint32_t* __restrict__ old_to_new, FieldSet fs,
                                                         float4* __restrict__ spos, float4* __restrict__ sfwd,
                                                         uint32_t* __restrict__ start, uint32_t* __restrict__ count) {
    __shared__ uint32_t lds[kBlock / 64];
    __shared__ uint32_t tile[kScanFusedTiles];
    const uint32_t agent_blocks = (n + kBlock - 1) / kBlock;
    const uint32_t s = blockIdx.x * kBlock + threadIdx.x;
    // The agent's loads first: they overlap the scan of the tile sums.
    const bool active = blockIdx.x < agent_blocks && s < n;
    uint32_t c = 0, t = 0, id = 0;
    float4 p, f;
    if (active) {
        c = key[s];
        t = off[c] + rank[s];
        id = ids[s];
        p = make_float4(fs.src[0][s], fs.src[1][s], fs.src[2][s], __uint_as_float(id));
        f = make_float4(fs.src[3][s], fs.src[4][s], fs.src[5][s], fs.src[6][s]);
    }
    // Exclusive scan of the tile sums, four per thread.
    constexpr uint32_t kPer = kScanFusedTiles / kBlock;
    uint32_t v[kPer], sum = 0;
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) {
        const uint32_t i = threadIdx.x * kPer + j;
        v[j] = i < ntiles ? partial[i] : 0u;
        sum += v[j];
    }
    uint32_t total;
    uint32_t o = block_exclusive_scan(sum, lds, total);
#pragma unroll
    for (uint32_t j = 0; j < kPer; ++j) {
        tile[threadIdx.x * kPer + j] = o;
        o += v[j];
    }
    __syncthreads();
    if (blockIdx.x < agent_blocks) {
        if (!active) return;
        t += tile[c / kScanTile];
        if (t >= n) return;  // only after a corrupted count array (see k_scatter)
        new_to_old[t] = s;
        old_to_new[s] = t;
        ids_new[t] = id;
        spos[t] = p;
        sfwd[t] = f;
        return;
    }
    const uint32_t b = blockIdx.x - agent_blocks;
    const uint32_t add = tile[b];
    const uint64_t base = (uint64_t)b * kScanTile;
#pragma unroll
    for (int j = 0; j < kScanItems; ++j) {
        const uint64_t i = base + (uint64_t)j * kBlock + threadIdx.x;
        if (i < C) {
            start[i] = off[i] + add;
            count[i] = 0u;
        }
    }
    if (b == 0 && threadIdx.x == 0) start[C] = total;
}

void launch_scan_counts(uint32_t* count, uint32_t* start, uint32_t C, hipStream_t st) {
    if (C <= kScanAloneCells) {
        k_scan_one<<<1, kScanOneThreads, 0, st>>>(C, count, start, 0, nullptr, nullptr, nullptr, nullptr);
        GS_LAUNCHED("k_scan_one");
        return;
    }
    const uint32_t ntiles = (C + kScanTile - 1) / kScanTile;
    uint32_t* partial = start + C + 1;
    k_scan_tiles<<<ntiles, kBlock, 0, st>>>(C, count, start, partial);
    GS_LAUNCHED("k_scan_tiles");
    const int fused = ntiles <= kScanFusedTiles ? 1 : 0;
    if (!fused) {
        k_scan_partials<<<1, kBlock, 0, st>>>(ntiles, partial, start, C);
        GS_LAUNCHED("k_scan_partials");
    }
    k_scan_add<<<ntiles, kBlock, 0, st>>>(C, partial, start, count, fused);
    GS_LAUNCHED("k_scan_add");
}

void launch_scatter_reorder(uint32_t n, const uint32_t* key, const uint32_t* rank, const uint32_t* start,
                            const uint32_t* ids, uint32_t* ids_new, uint32_t* id_tmp,
                            uint32_t* new_to_old, uint32_t* old_to_new, const uint32_t* bits, uint32_t* bits_new,
                            const FieldSet& fs, float4* spos, hipStream_t st, float4* sfwd, bool scattered) {
    if (n == 0) return;
    if (!scattered) {
        k_scatter<<<blocks_for(n), kBlock, 0, st>>>(n, key, rank, start, ids, id_tmp);
        GS_LAUNCHED("k_scatter");
    }
    k_reorder<<<agent_blocks(n), agent_block(n), 0, st>>>(n, rank, id_tmp, key, start, ids, ids_new, new_to_old,
                                                old_to_new, bits, bits_new, fs, spos, sfwd);
    GS_LAUNCHED("k_reorder");
}

// Buffers of a build of g on b (counts zero for a new lattice), and where its
// key pass keeps the positions' bounding box once a capped search targets the
// group (acc NULL: nowhere).
struct BoxPair {
    uint32_t *acc, *clear;
};
static BoxPair begin_build(gs_group_s* g, const gs_bins_s* b) {
    const uint32_t n = g->n, C = b->cells;
    g->key.reserve(n);
    g->rank.reserve(n);
    g->id_tmp.reserve(n);
    g->new_to_old.reserve(n);
    g->old_to_new.reserve(n);
    g->spos.reserve(n);
    g->start.reserve((size_t)C + 1 + (C + kScanTile - 1) / kScanTile);  // partial tile sums live after start[C]
    if (!g->binned || g->bin_cells != C || g->count.cap < C) {
        g->count.reserve(C);
        // A fill kernel rather than hipMemsetAsync, so the build can be
        // captured into a graph.
        launch_fill_u32(g->count.p, C, 0u, g->ctx->stream);
    }
    g->bin_cells = C;
    g->bin_grid = b->g;
    BoxPair box{nullptr, nullptr};
    if (g->bbox_wanted && g->bbox[0].p && g->bbox[1].p && n > 0) {
        g->bbox_cur ^= 1;
        box.acc = g->bbox[g->bbox_cur].p;
        box.clear = g->bbox[g->bbox_cur ^ 1].p;
    }
    g->bbox_fresh = box.acc != nullptr;
    g->cbox_fresh = false;
    return box;
}
// The fields a build moves.  Fields holding one value in every slot are
// unchanged by any permutation and stay where they are (positions always
// move: the snapshot is built from them).
static uint32_t moved_fields(const gs_group_s* g, FieldSet& fs) {
    const uint32_t moved = g->live & ~(g->inv & ~kFPos);
    fs.nf = 0;
    for (int f = 0; f < kFields; ++f)
        if (moved & (1u << f)) {
            fs.src[fs.nf] = g->F(f);
            fs.dst[fs.nf] = g->Falt(f);
            ++fs.nf;
        }
    return moved;
}
static bool moves_bits(const gs_group_s* g) { return g->kind == GS_KIND_AGENTS && !g->bits_zero; }
static void end_build(gs_group_s* g, uint32_t moved, bool bits) {
    for (int f = 0; f < kFields; ++f)
        if (moved & (1u << f)) g->flip(f);
    if (bits) g->bcur ^= 1;
    if (g->n > 0) g->icur ^= 1;
    g->binned = true;
    g->snap_valid = true;
}

bool pair_build_ok(const gs_group_s* g, const gs_bins_s* b) {
    return g->n > 0 && g->n <= kScanOneAgents && b->cells <= kScanOneCells;
}
void launch_pair_build(gs_group_s* const g[2], const gs_bins_s* b) {
    PairBuild P{};
    uint32_t moved[2], n = 0;
    bool bits[2];
    for (int i = 0; i < 2; ++i) {
        const BoxPair box = begin_build(g[i], b);
        PairBuild::One& o = P.g[i];
        o.n = g[i]->n;
        n = std::max(n, o.n);
        o.px = g[i]->F(0);
        o.py = g[i]->F(1);
        o.pz = g[i]->F(2);
        o.key = g[i]->key.p;
        o.rank = g[i]->rank.p;
        o.count = g[i]->count.p;
        o.start = g[i]->start.p;
        o.id_tmp = g[i]->id_tmp.p;
        o.ids = g[i]->ids();
        o.ids_new = g[i]->ids_alt();
        o.new_to_old = g[i]->new_to_old.p;
        o.old_to_new = g[i]->old_to_new.p;
        o.box_acc = box.acc;
        o.box_clear = box.clear;
        moved[i] = moved_fields(g[i], o.fs);
        bits[i] = moves_bits(g[i]);
        o.bits = bits[i] ? g[i]->bits() : nullptr;
        o.bits_new = bits[i] ? g[i]->bitsb[g[i]->bcur ^ 1].p : nullptr;
        o.spos = g[i]->spos.p;
    }
    hipStream_t st = g[0]->ctx->stream;
    k_pair_key<<<dim3(blocks_for(n), 2), kBlock, 0, st>>>(P, b->g);
    GS_LAUNCHED("k_pair_key");
    k_pair_scan<<<dim3(1, 2), kScanOneThreads, 0, st>>>(P, b->cells);
    GS_LAUNCHED("k_pair_scan");
    k_pair_reorder<<<dim3(agent_blocks(n), 2), agent_block(n), 0, st>>>(P);
    GS_LAUNCHED("k_pair_reorder");
    for (int i = 0; i < 2; ++i) end_build(g[i], moved[i], bits[i]);
}

// lazy (fused Boids step only): move nothing but the snapshots (positions,
// and forward + speed into sfwd), the agent indices and the maps; every
// other field stays in the previous order until the flock kernel, which reads
// it through new_to_old and writes the step's results in the new order.
void launch_bins_build(gs_group_s* g, const gs_bins_s* b, int wrap_shape, const float* wc, const float* ws,
                       bool lazy, bool keys_ready, bool free_order) {
    const uint32_t n = g->n;
    const uint32_t C = b->cells;
    hipStream_t st = g->ctx->stream;
    // Keys from the previous step's flock kernel (counts already taken):
    // only for the lattice that step was built on, never with a box to keep.
    if (keys_ready && (!g->binned || g->bin_cells != C || g->count.cap < C || g->bbox_wanted))
        fail(GS_ERR_INVALID_ARGUMENT, "internal: stale fused keys");
    const BoxPair box = begin_build(g, b);
    const uint32_t ntiles = (C + kScanTile - 1) / kScanTile;
    free_order = free_order && lazy && n > 0;
    // With k_reorder_free the offsets within the tiles use the scatter's
    // buffer.
    const bool free_tiles = free_order && C > kScanAloneCells && C <= n && ntiles <= kScanFusedTiles;
    float wcv[3] = {0, 0, 0}, wsv[3] = {0, 0, 0};
    if (wc) memcpy(wcv, wc, sizeof wcv);
    if (ws) memcpy(wsv, ws, sizeof wsv);
    if (n > 0 && !keys_ready) {
        k_bin_key<<<blocks_for(n), kBlock, 0, st>>>(n, g->F(0), g->F(1), g->F(2), b->g, g->key.p, g->rank.p,
                                                    g->count.p, wrap_shape, wcv[0], wcv[1], wcv[2], wsv[0], wsv[1],
                                                    wsv[2], box.acc, box.clear);
        GS_LAUNCHED("k_bin_key");
    }
    // Small groups on small lattices: scan and scatter in one launch.
    const bool one = !free_order && scatter_in_scan(n, C);
    if (one) {
        k_scan_one<<<1, kScanOneThreads, 0, st>>>(C, g->count.p, g->start.p, n, g->key.p, g->rank.p, g->ids(),
                                                  g->id_tmp.p);
        GS_LAUNCHED("k_scan_one");
    } else if (free_tiles) {
        uint32_t *partial = g->start.p + C + 1, *off = g->id_tmp.p;
        k_scan_tiles<<<ntiles, kBlock, 0, st>>>(C, g->count.p, off, partial);
        GS_LAUNCHED("k_scan_tiles");
        FieldSet fs{};
        for (int f = 0; f < 7; ++f) fs.src[f] = g->F(f);
        g->sfwd.reserve(n);
        k_reorder_free<<<blocks_for(n) + ntiles, kBlock, 0, st>>>(n, C, ntiles, g->rank.p, g->key.p, off, partial,
                                                                  g->ids(), g->ids_alt(), g->new_to_old.p,
                                                                  g->old_to_new.p, fs, g->spos.p, g->sfwd.p,
                                                                  g->start.p, g->count.p);
        GS_LAUNCHED("k_reorder_free");
    } else {
        launch_scan_counts(g->count.p, g->start.p, C, st);
    }
    uint32_t moved = 0;
    bool has_bits = false;
    if (n > 0 && !free_tiles) {
        FieldSet fs{};
        if (lazy) {
            for (int f = 0; f < 7; ++f) fs.src[f] = g->F(f);
            g->sfwd.reserve(n);
        } else {
            moved = moved_fields(g, fs);
            has_bits = moves_bits(g);
        }
        launch_scatter_reorder(n, g->key.p, g->rank.p, g->start.p, g->ids(), g->ids_alt(),
                               free_order ? nullptr : g->id_tmp.p, g->new_to_old.p, g->old_to_new.p,
                               has_bits ? g->bits() : nullptr, has_bits ? g->bitsb[g->bcur ^ 1].p : nullptr, fs,
                               g->spos.p, st, lazy ? g->sfwd.p : nullptr, one || free_order);
    }
    end_build(g, moved, has_bits);
}

}  // namespace gs
