// Kernels of the host transfers: state and lists between storage (slot) order
// and agent-index order.  The host then moves one packed block instead of one
// small copy per field, and nothing is permuted on the host.
//
// Bound by the copy over PCIe and, for small groups, by the calls; the kernels
// read coalesced and write each field's words scattered by agent index, which
// stays in L2.
#include "gs_internal.hpp"

namespace gs {

__global__ __launch_bounds__(kBlock) void k_pack_fields(uint32_t n, const uint32_t* __restrict__ ids, FieldWords f,
                                                        uint32_t* __restrict__ out, uint32_t* __restrict__ bad) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t id = ids[s];
    if (id >= n) {  // a corrupted id map
        *bad = 1u;
        return;
    }
#pragma unroll
    for (int j = 0; j < kMaxWords; ++j)
        if (j < f.nf) out[(size_t)j * n + id] = f.p[j][s];
}

__global__ __launch_bounds__(kBlock) void k_unpack_fields(uint32_t n, const uint32_t* __restrict__ in, FieldWords f) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
#pragma unroll
    for (int j = 0; j < kMaxWords; ++j)
        if (j < f.nf) f.p[j][i] = in[(size_t)j * n + i];
}

// Rows j0 .. j0 + rows - 1 of a slot-space list as agent indices: out holds
// the rows' neighbour indices, then their distances.
__global__ __launch_bounds__(kBlock) void k_pack_knn(uint32_t n, uint32_t nb, uint32_t j0, uint32_t rows,
                                                     const uint32_t* __restrict__ idx, const float* __restrict__ dist,
                                                     const uint32_t* __restrict__ ida, const uint32_t* __restrict__ idb,
                                                     uint32_t* __restrict__ out) {
    const uint32_t s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= n) return;
    const uint32_t a = ida[s];
    for (uint32_t j = 0; j < rows; ++j) {
        const uint32_t v = idx[(size_t)(j0 + j) * n + s];
        out[(size_t)j * n + a] = v < nb ? idb[v] : UINT32_MAX;
        out[(size_t)(rows + j) * n + a] = __float_as_uint(dist[(size_t)(j0 + j) * n + s]);
    }
}

void launch_pack_fields(uint32_t n, const uint32_t* ids, const FieldWords& f, uint32_t* out, uint32_t* bad,
                        hipStream_t st) {
    launch_fill_u32(bad, 1, 0u, st);
    k_pack_fields<<<blocks_for(n), kBlock, 0, st>>>(n, ids, f, out, bad);
    GS_LAUNCHED("k_pack_fields");
}

void launch_unpack_fields(uint32_t n, const uint32_t* in, const FieldWords& f, hipStream_t st) {
    k_unpack_fields<<<blocks_for(n), kBlock, 0, st>>>(n, in, f);
    GS_LAUNCHED("k_unpack_fields");
}

void launch_pack_knn(uint32_t n, uint32_t nb, uint32_t j0, uint32_t rows, const uint32_t* idx, const float* dist,
                     const uint32_t* ida, const uint32_t* idb, uint32_t* out, hipStream_t st) {
    k_pack_knn<<<blocks_for(n), kBlock, 0, st>>>(n, nb, j0, rows, idx, dist, ida, idb, out);
    GS_LAUNCHED("k_pack_knn");
}

}  // namespace gs
