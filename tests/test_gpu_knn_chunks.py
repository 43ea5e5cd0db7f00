"""The exhaustive search over 64-slot chunks (small and sparse targets, small
groups over a wide reach): exact lists at the edges of chunks and of the
dispatch, with and without a bound to start from."""
import numpy as np
import pytest

from gpusteer_amd import scenarios

pytestmark = pytest.mark.gpu

SIZE = (200.0, 10.0, 200.0)


def _points(n, seed, spread=100.0):
    g = np.random.default_rng(seed)
    p = g.uniform(-spread, spread, (n, 3)) * [1.0, 0.0, 1.0]
    p[: n // 4] = [20.0, 0.0, -30.0] + 0.5 * g.normal(size=(n // 4, 3))
    if n > 8:
        p[-3:] = p[:3]
    return p.astype(np.float32)[g.permutation(n)]


def _group(gs, ctx, pos):
    n = pos.shape[0]
    return gs.AgentGroup(ctx, scenarios.make_agents(pos, np.tile([[0.0, 0.0, 1.0]], (n, 1)), np.zeros(n), 0.5, 1.0, 1.0))


def _check(gs, ctx, orc, a, b, k, cells, cap):
    """Unseeded, seeded, and seeded after both groups moved and were binned
    again (the chunk boxes are then the new snapshot's)."""
    bins = gs.KNNBinData(ctx, cells, SIZE)
    A = _group(gs, ctx, a)
    B = A if b is None else _group(gs, ctx, b)
    knn = gs.KNNData(ctx, a.shape[0], k)
    q = np.unique(np.linspace(0, a.shape[0] - 1, 200).astype(np.uint32))
    for step in range(3):
        if step != 1:
            for G in {A, B}:
                gs.updateKNNDatabase(G, bins)
        if cap is None:
            gs.findKNearestNeighbors(A, knn, bins, B, 1)
        else:
            gs.findKNearestNeighborsWithin(A, knn, bins, B, cap, 1)
        idx, dist = knn.download()
        pa, pb = A.download().pos(), B.download().pos()
        r_idx, r_dist = orc.knn_brute(pa, pb, k, b is None, queries=q, cap=float("inf") if cap is None else cap)
        np.testing.assert_array_equal(idx[:, q], r_idx[:, q])
        np.testing.assert_array_equal(dist[:, q], r_dist[:, q])
        if step == 1:
            for G in {A, B}:
                gs.wrapWorld(G, worldSize=(150.0, 20.0, 150.0))
    for h in (knn, bins, A) + (() if b is None else (B,)):
        h.close()


# Small targets (at most 256 points, the group itself among them); sparse
# targets (at most 4,096, fewer than one per 16 cells); small groups over a wide
# reach (at most 16,384 on both sides); both sides of 16 and 8 lanes a query.
@pytest.mark.parametrize("na,nb,k,cells,cap", [
    (1, 1, 1, (4, 1, 4), None), (5, 0, 7, (4, 1, 4), None), (64, 0, 7, (4, 1, 4), None), (65, 0, 16, (4, 1, 4), 30.0),
    (256, 0, 8, (16, 1, 16), None), (3000, 2, 3, (40, 1, 40), None), (3000, 63, 3, (40, 1, 40), 25.0),
    (24576, 64, 4, (40, 1, 40), None), (24577, 65, 9, (40, 1, 40), None), (140000, 256, 3, (40, 1, 40), 50.0),
    (5000, 1254, 3, (512, 1, 512), 140.0), (30000, 1254, 16, (512, 1, 512), 140.0), (5000, 4096, 7, (512, 1, 512), None),
    (5000, 5000, 7, (64, 1, 64), 62.0), (2000, 16384, 16, (64, 1, 64), None), (300, 10000, 1, (64, 1, 64), 200.0),
    (4096, 256, 7, (65, 1, 64), None), (4096, 257, 7, (65, 1, 64), None), (4097, 257, 7, (65, 1, 64), 60.0),
    (4096, 5000, 16, (64, 1, 64), None), (1000, 16384, 7, (100, 1, 100), None), (1000, 16384, 8, (100, 1, 100), 30.0),
    (140000, 1254, 16, (512, 1, 512), 140.0)])
def test_lists(gs, ctx, orc, na, nb, k, cells, cap):
    print(f"case na={na} nb={nb} k={k} cells={cells} cap={cap}", flush=True)
    _check(gs, ctx, orc, _points(na, na), _points(nb, nb + 1) if nb else None, k, cells, cap)


# Small groups by small groups: the cells around the query, wider boxes while
# they have no more columns than the target has chunks, then the chunks; the
# split scan for more than 16 neighbours.
@pytest.mark.parametrize("where", ["mixed", "apart", "one cluster"])
@pytest.mark.parametrize("na,nb,k,radius,cap", [
    (2000, 1025, 1, 1, 40.0), (2000, 1025, 7, 2, 75.0), (1999, 4096, 8, 1, None), (513, 1024, 9, 2, 1e6),
    (300, 10000, 16, 1, 60.0), (16384, 257, 7, 1, None), (8192, 3000, 7, 1, None), (8193, 3000, 16, 1, 1e6),
    (500, 16000, 7, 2, 150.0), (2000, 1025, 20, 1, 75.0), (1999, 4096, 32, 2, None), (513, 1024, 17, 1, 1e6)])
def test_small_groups(gs, ctx, orc, where, na, nb, k, radius, cap):
    print(f"case {where} na={na} nb={nb} k={k} radius={radius} cap={cap}", flush=True)
    g = np.random.default_rng(na + nb)
    lo, hi = {"mixed": (-100.0, 100.0), "apart": (60.0, 100.0), "one cluster": (-8.0, 8.0)}[where]
    a = g.uniform(-100.0, -60.0 if where == "apart" else 100.0, (na, 3)).astype(np.float32)
    b = g.uniform(lo, hi, (nb, 3)).astype(np.float32)
    bins = gs.KNNBinData(ctx, (23, 20, 24), (200.0, 200.0, 200.0))
    A, B = _group(gs, ctx, a), _group(gs, ctx, b)
    knn = gs.KNNData(ctx, na, k)
    limit = float("inf") if cap is None else cap
    for step in range(3):
        if step != 1:
            for G in (A, B):
                gs.updateKNNDatabase(G, bins)
        if cap is None:
            gs.findKNearestNeighbors(A, knn, bins, B, radius)
        else:
            gs.findKNearestNeighborsWithin(A, knn, bins, B, cap, radius)
        idx, dist = knn.download()
        q = np.unique(np.linspace(0, na - 1, 300).astype(np.uint32))
        r_idx, r_dist = orc.knn_brute(A.download().pos(), B.download().pos(), k, False, queries=q, cap=limit)
        np.testing.assert_array_equal(idx[:, q], r_idx[:, q])
        np.testing.assert_array_equal(dist[:, q], r_dist[:, q])
        if step == 1:  # part of each group goes to the opposite face: seeds far away
            for G in (A, B):
                gs.wrapWorld(G, worldSize=(150.0, 150.0, 150.0))
    for h in (knn, bins, A, B):
        h.close()


# Few targets of many queries, on both sides of the lines where a lane per query
# takes over: with a seed and without, by the targets and by those in reach.
@pytest.mark.parametrize("na,nb,k,cells,cap", [
    (4096, 1, 3, (40, 1, 40), None), (65536, 16, 7, (40, 1, 40), None), (65536, 17, 16, (40, 1, 40), 50.0),
    (65536, 64, 3, (40, 1, 40), None), (65535, 64, 3, (40, 1, 40), None), (131072, 33, 9, (40, 1, 40), None),
    (262144, 128, 7, (64, 1, 64), None), (262144, 129, 16, (64, 1, 64), None),
    (262144, 1254, 7, (512, 1, 512), 30.0), (524288, 1254, 3, (512, 1, 512), 12.0)])
def test_few_targets(gs, ctx, orc, na, nb, k, cells, cap):
    print(f"case na={na} nb={nb} k={k} cells={cells} cap={cap}", flush=True)
    _check(gs, ctx, orc, _points(na, na), _points(nb, nb + 1), k, cells, cap)


# Every point in one place: the bounds of all lanes and chunks are equal.
@pytest.mark.parametrize("na,nb,k,cells", [(300, 100, 7, (4, 1, 4)), (2000, 3000, 16, (16, 1, 16)),
                                           (9000, 3000, 7, (16, 4, 16)), (30000, 1000, 3, (200, 1, 200))])
def test_ties(gs, ctx, na, nb, k, cells):
    bins = gs.KNNBinData(ctx, cells, SIZE)
    A, B = _group(gs, ctx, _points(na, 8)), _group(gs, ctx, np.tile(np.float32([[7.0, 0.0, -11.0]]), (nb, 1)))
    knn = gs.KNNData(ctx, na, k)
    for G in (A, B):
        gs.updateKNNDatabase(G, bins)
    for _ in range(2):
        gs.findKNearestNeighbors(A, knn, bins, B, 1)
        idx, _ = knn.download()
        np.testing.assert_array_equal(idx, np.tile(np.arange(k, dtype=np.uint32)[:, None], (1, na)))
    for h in (knn, bins, A, B):
        h.close()


def test_far_targets_and_odd_coordinates(gs, ctx, orc):
    a, b = _points(3000, 3), _points(200, 4, spread=5.0) + np.float32([5e4, 0.0, -5e4])
    _check(gs, ctx, orc, a, b, 7, (40, 1, 40), None)
    # coordinates that are no numbers belong to no list and bound nothing
    b = _points(130, 5)
    bad = b.copy()
    bad[::3, 0] = np.nan
    bins = gs.KNNBinData(ctx, (40, 1, 40), SIZE)
    A, B = _group(gs, ctx, a), _group(gs, ctx, bad)
    knn = gs.KNNData(ctx, a.shape[0], 16)
    for G in (A, B):
        gs.updateKNNDatabase(G, bins)
    for _ in range(2):
        gs.findKNearestNeighbors(A, knn, bins, B, 1)
        idx, dist = knn.download()
        keep = np.nonzero(~np.isnan(bad[:, 0]))[0].astype(np.uint32)
        r_idx, r_dist = orc.knn_brute(a, b[keep], 16, False)
        np.testing.assert_array_equal(idx, keep[r_idx])
        np.testing.assert_array_equal(dist, r_dist)
    for h in (knn, bins, A, B):
        h.close()


def test_recorded_search_of_a_target_that_moves(gs, ctx, orc):
    """A recorded frame computes the boxes it reads, whatever was current when
    it was recorded."""
    a, b = _points(2000, 6), _points(200, 7)
    bins = gs.KNNBinData(ctx, (40, 1, 40), SIZE)
    A, B = _group(gs, ctx, a), _group(gs, ctx, b)
    knn = gs.KNNData(ctx, 2000, 7)

    def frame():
        for G in (A, B):
            gs.updateGroup(G, 0.0, gs.MODE_GPUREF)
            gs.wrapWorld(G, worldSize=(150.0, 20.0, 150.0))
            gs.updateKNNDatabase(G, bins)
        gs.findKNearestNeighbors(A, knn, bins, B, 1)

    def check():
        idx, dist = knn.download()
        r_idx, r_dist = orc.knn_brute(A.download().pos(), B.download().pos(), 7, False)
        np.testing.assert_array_equal(idx, r_idx)
        np.testing.assert_array_equal(dist, r_dist)

    frame(), frame()
    with ctx.record(lambda: (frame(), frame())) as f:
        for _ in range(3):
            f.launch(1)
            check()
            gs.findKNearestNeighbors(A, knn, bins, B, 1)  # between replays, from the boxes that are current
            check()
            gs.findKNearestNeighbors(A, knn, bins, B, 1)
    frame()
    check()
    for h in (knn, bins, A, B):
        h.close()
