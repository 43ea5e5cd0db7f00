"""Host transfers at the sizes where they change their way: packed through
pinned memory, packed in passes, field by field."""
import ctypes as C

import numpy as np
import pytest

from gpusteer_amd import _capi as capi
from gpusteer_amd import scenarios
from gpusteer_amd.state import AGENT_FIELDS

pytestmark = pytest.mark.gpu


def _state(n):
    g = np.random.default_rng(n)
    st = scenarios.make_agents(g.uniform(0, 50, (n, 3)).astype(np.float32), scenarios.unit_vectors(g, n),
                               np.zeros(n), 0.5, 1.0, 1.0)
    for f in AGENT_FIELDS[3:]:
        st.arrays[f] = g.normal(size=n).astype(np.float32)
    st.bits = g.integers(0, 1 << 13, n).astype(np.uint32)
    return st


# 24 words per agent: uploads are packed up to 1,048,576 words (43,690
# agents), read backs one pass up to 2,097,152 (87,381 agents).
@pytest.mark.parametrize("n", [1, 2, 257, 43690, 43691, 87381, 87382, 300001])
def test_state_round_trip(gs, ctx, n):
    st = _state(n)
    A = gs.AgentGroup(ctx, st)
    bins = gs.KNNBinData(ctx, (9, 9, 9), (50.0,) * 3, origin=(0.0,) * 3)
    for _ in range(2):
        out = A.download()
        for f in AGENT_FIELDS + ("bits",):
            np.testing.assert_array_equal(out[f], st[f], err_msg=f)
        gs.updateKNNDatabase(A, bins)  # storage order is cell order from here on
    # only some fields wanted
    s, px, bits = capi.GsAgents(), np.zeros(n, np.float32), np.zeros(n, np.uint32)
    s.px, s.bits = capi.fptr(px), capi.uptr(bits)
    capi.check(capi.lib.gs_group_download_agents(A.h, C.byref(s)), "gs_group_download_agents")
    np.testing.assert_array_equal(px, st["px"])
    np.testing.assert_array_equal(bits, st.bits)
    for h in (A, bins):
        h.close()


# Two words per list entry: one pass up to 1,048,576 entries, then by rows.
@pytest.mark.parametrize("na,nb,k", [(1, 3, 2), (65536, 65536, 16), (65537, 500, 16), (300001, 1000, 3)])
def test_lists_in_agent_order(gs, ctx, orc, na, nb, k):
    a, b = _state(na), _state(nb)
    A, B = gs.AgentGroup(ctx, a), gs.AgentGroup(ctx, b)
    bins = gs.KNNBinData(ctx, (9, 9, 9), (50.0,) * 3, origin=(0.0,) * 3)
    for G in (A, B):
        gs.updateKNNDatabase(G, bins)
    knn = gs.KNNData(ctx, na, k)
    gs.findKNearestNeighbors(A, knn, bins, B, 1)
    idx, dist = knn.download()
    q = np.unique(np.linspace(0, na - 1, 200).astype(np.uint32))
    r_idx, r_dist = orc.knn_brute(a.pos(), b.pos(), k, False, queries=q)
    np.testing.assert_array_equal(idx[:, q], r_idx[:, q])
    np.testing.assert_array_equal(dist[:, q], r_dist[:, q])
    only = np.zeros((k, na), np.float32)
    capi.check(capi.lib.gs_knn_download(knn.h, None, capi.fptr(only)), "gs_knn_download")
    np.testing.assert_array_equal(only, dist)
    for h in (knn, bins, A, B):
        h.close()


def _same(a, b):
    for f in AGENT_FIELDS + ("bits",):
        np.testing.assert_array_equal(a[f], b[f], err_msg=f)


# Without room on the device for the packed block the transfers go field by
# field: an upload, which has changed its handle before, ends whole, and results
# can be read back.
def test_transfers_without_staging_memory(gs, orc):
    c = gs.Context(0)  # no staging yet, and 50,000 agents take none
    a, b = _state(50000), _state(5000)
    A = gs.AgentGroup(c, a)
    bins = gs.KNNBinData(c, (9, 9, 9), (50.0,) * 3, origin=(0.0,) * 3)
    knn = gs.KNNData(c, 50000, 7)
    gs.updateKNNDatabase(A, bins)  # storage order is cell order from here on
    gs.findKNearestNeighbors(A, knn, bins, A, 1)
    try:
        capi.lib.gs_debug_fail_alloc_after(0)
        _same(A.download(), a)
        idx, dist = knn.download()
        A.upload(b)
        _same(A.download(), b)
    finally:
        capi.lib.gs_debug_fail_alloc_after(-1)
    _same(A.download(), b)
    q = np.unique(np.linspace(0, 49999, 200).astype(np.uint32))
    r_idx, r_dist = orc.knn_brute(a.pos(), a.pos(), 7, True, queries=q)
    np.testing.assert_array_equal(idx[:, q], r_idx[:, q])
    np.testing.assert_array_equal(dist[:, q], r_dist[:, q])
    for h in (knn, bins, A):
        h.close()
    c.close()


def test_ensemble_transfers_without_staging_memory(gs):
    c = gs.Context(0)
    st, p = scenarios.boids_sphere(n=5000)
    other, _ = scenarios.boids_sphere(n=5000, workload=2)
    e = gs.Ensemble(c, [("boids", st, p)])
    e.step(3)  # storage order is cell order from here on
    try:
        capi.lib.gs_debug_fail_alloc_after(0)
        out = e.download(0)  # one word more than the upload's staging
        e.upload(0, 0, other)
        _same(e.download(0), other)
    finally:
        capi.lib.gs_debug_fail_alloc_after(-1)
    _same(e.download(0), other)
    e.upload(0, 0, st)
    e.step(3)
    _same(e.download(0), out)
    e.close()
    c.close()
