"""The several-lanes-per-query search at the sizes where its dispatch, its
teams and its buffers have edges (and the one-lane search beyond them), bit-exact against the oracle's brute force
(on a sample of queries) and against the one-lane search (which a launch shape
set on the context selects for k = 7)."""
import numpy as np
import pytest

from gpusteer_amd import _capi as capi
from gpusteer_amd import scenarios

pytestmark = pytest.mark.gpu

SIZE = 40.0


def _points(n, seed, dims=3):
    """Uniform points, a sixth of them in a dense clump inside one cell, some
    exact duplicates, some outside the lattice."""
    g = np.random.default_rng(seed)
    p = g.uniform(0.0, SIZE, size=(n, 3))
    m = n // 6
    p[:m] = 7.0 + 0.3 * g.normal(size=(m, 3))
    if n > 40:
        p[-8:] = p[:8]
        p[m:m + 4] = [[-5.0, 3.0, 3.0], [55.0, 1.0, 2.0], [3.0, 3.0, -60.0], [20.0, 90.0, 20.0]]
    if dims == 2:
        p[:, 1] = 0.0
    return p.astype(np.float32)[g.permutation(n)]


def _group(gs, ctx, pos):
    n = pos.shape[0]
    return gs.AgentGroup(ctx, scenarios.make_agents(pos, np.tile([[0.0, 0.0, 1.0]], (n, 1)), np.zeros(n), 0.5, 1.0, 1.0))


def _search(gs, ctx, a, b, k, cells, radius=1, cap=None, calls=1):
    """One list per call (the second and later calls are seeded)."""
    bins = gs.KNNBinData(ctx, cells, (SIZE,) * 3, origin=(0.0, 0.0, 0.0))
    A = _group(gs, ctx, a)
    B = A if b is None else _group(gs, ctx, b)
    for G in {A, B}:
        gs.updateKNNDatabase(G, bins)
    knn = gs.KNNData(ctx, a.shape[0], k)
    out = []
    for _ in range(calls):
        if cap is None:
            gs.findKNearestNeighbors(A, knn, bins, B, radius, capi.GS_KNN_BINNED)
        else:
            gs.findKNearestNeighborsWithin(A, knn, bins, B, cap, radius, capi.GS_KNN_BINNED)
        out.append(knn.download())
    for h in (knn, bins, A) + (() if b is None else (B,)):
        h.close()
    return out


# Few points; teams and blocks that end inside a wavefront; both sides of the
# dispatch's lines (16 lanes to 24,576 and 8 to 131,072 queries for k <= 8,
# 131,072 and 262,144 for longer lists).
@pytest.mark.parametrize("n,k,cells,radius", [
    (1, 7, (4, 4, 4), 1), (3, 8, (4, 4, 4), 1), (9, 16, (2, 2, 2), 1), (31, 7, (8, 8, 24), 1), (257, 1, (5, 5, 5), 1),
    (1000, 7, (1, 1, 1), 1), (1000, 16, (30, 30, 30), 2), (2049, 9, (9, 7, 21), 1), (5000, 8, (30, 30, 60), 2),
    (5000, 7, (40, 1, 40), 1), (24576, 7, (20, 20, 20), 1), (24577, 7, (20, 20, 20), 1), (24577, 4, (50, 50, 50), 2),
    (131072, 7, (36, 36, 36), 1), (131073, 7, (36, 36, 36), 1), (131072, 16, (30, 30, 60), 1),
    (131073, 16, (30, 30, 60), 1), (262144, 12, (40, 40, 80), 1), (262145, 12, (40, 40, 80), 1),
    (131073, 1, (36, 36, 36), 1), (131073, 4, (36, 36, 36), 1), (131073, 8, (30, 30, 90), 1), (131073, 5, (36, 36, 36), 2),
    (131073, 8, (60, 1, 60), 1), (262145, 16, (40, 40, 80), 1), (262145, 9, (60, 60, 60), 2)])
def test_lists_at_the_edges(gs, ctx, orc, n, k, cells, radius):
    print(f"case n={n} k={k} cells={cells} radius={radius}", flush=True)
    pos = _points(n, n + k, dims=2 if cells[1] == 1 and cells[0] > 1 else 3)
    q = np.unique(np.linspace(0, n - 1, min(n, 300)).astype(np.uint32))
    r_idx, r_dist = orc.knn_brute(pos, pos, k, True, queries=q)
    for idx, dist in _search(gs, ctx, pos, None, k, cells, radius, calls=2):
        np.testing.assert_array_equal(idx[:, q], r_idx[:, q])
        np.testing.assert_array_equal(dist[:, q], r_dist[:, q])


@pytest.mark.parametrize("na,nb,k,cap", [(700, 3000, 7, 1.0), (3000, 700, 16, 2.5), (30000, 5000, 7, 0.5),
                                         (300, 1, 7, 30.0), (5000, 5000, 3, 100.0),
                                         (30000, 20000, 7, 6.0), (9000, 30000, 16, 4.0), (30000, 18000, 7, 1.9), (30000, 18000, 7, 2.1),
                                         (131073, 5000, 4, 1.0), (131073, 5000, 8, 2.5), (131073, 20000, 7, 0.5),
                                         (262145, 5000, 16, 1.0), (262145, 5000, 9, 4.0)])
def test_two_groups_within(gs, ctx, orc, na, nb, k, cap):
    a, b = _points(na, 1), _points(nb, 2)
    q = np.unique(np.linspace(0, na - 1, 300).astype(np.uint32))
    r_idx, r_dist = orc.knn_brute(a, b, k, False, queries=q, cap=cap)
    for idx, dist in _search(gs, ctx, a, b, k, (20, 20, 20), cap=cap, calls=2):
        np.testing.assert_array_equal(idx[:, q], r_idx[:, q])
        np.testing.assert_array_equal(dist[:, q], r_dist[:, q])


@pytest.mark.parametrize("n,cells,radius", [(500, (8, 8, 8), 1), (3000, (12, 12, 36), 1), (3000, (24, 1, 24), 1),
                                            (40000, (24, 24, 24), 1)])
def test_same_lists_as_one_lane(gs, ctx, n, cells, radius):
    """Also with coordinates that are infinite, not numbers, or so large that
    squared distances overflow."""
    pos = _points(n, 5)
    pos[3], pos[17], pos[40] = (np.inf, 1.0, 2.0), (np.nan, 5.0, 5.0), (1.0, -np.inf, np.nan)
    pos[100:110, 0], pos[200:204, 2] = 3e30, np.float32(1e-42)
    got = _search(gs, ctx, pos, None, 7, cells, radius, calls=2)
    try:
        ctx.set_shape(capi.GS_SHAPE_KNN, 128, 1)
        want = _search(gs, ctx, pos, None, 7, cells, radius, calls=2)
    finally:
        ctx.set_shape(capi.GS_SHAPE_KNN, 256, 1)
    for g, w in zip(got, want):
        np.testing.assert_array_equal(g[0], w[0])
        np.testing.assert_array_equal(g[1], w[1])


# Exhaustive, local then chunks, teams, one lane per query, the split scan; the
# group itself and another one.
@pytest.mark.parametrize("na,nb,k,cells", [(100, 0, 7, (8, 8, 8)), (700, 100, 3, (8, 8, 8)), (700, 3000, 7, (12, 12, 12)),
                                           (3000, 0, 7, (12, 12, 12)), (40000, 0, 16, (24, 24, 24)),
                                           (131073, 0, 7, (36, 36, 36)), (131073, 0, 4, (36, 36, 36)),
                                           (700, 3000, 20, (12, 12, 12))])
def test_seed_with_lost_positions(gs, ctx, na, nb, k, cells):
    """A neighbour of the previous result whose position is no number any more
    bounds nothing: the list is that of a search without a seed."""
    A, B = (_movers(gs, ctx, _points(n, n + k)) if n else None for n in (na, nb))
    bins = gs.KNNBinData(ctx, cells, (SIZE,) * 3, origin=(0.0, 0.0, 0.0))
    seeded, fresh = gs.KNNData(ctx, na, k), gs.KNNData(ctx, na, k)
    groups = [A] + ([B] if B else [])
    for step in range(2):
        for G in groups:
            if step:
                gs.updateGroup(G, 0.01, capi.GS_MODE_GPUREF)
            gs.updateKNNDatabase(G, bins)
        gs.findKNearestNeighbors(A, seeded, bins, B or A, 1)
    gs.findKNearestNeighbors(A, fresh, bins, B or A, 1, capi.GS_KNN_NO_SEED)
    assert np.isnan((B or A).download().pos()).any()
    got, want = seeded.download(), fresh.download()
    np.testing.assert_array_equal(got[0], want[0])
    np.testing.assert_array_equal(got[1], want[1])
    for h in [seeded, fresh, bins] + groups:
        h.close()


def _movers(gs, ctx, pos):
    """A group of which every 29th agent loses its position at the first update."""
    n = pos.shape[0]
    st = scenarios.make_agents(pos, np.tile([[0.0, 0.0, 1.0]], (n, 1)), np.ones(n), 0.5, 1.0, 1.0)
    st.arrays["speed"][::29] = np.nan
    return gs.AgentGroup(ctx, st)
