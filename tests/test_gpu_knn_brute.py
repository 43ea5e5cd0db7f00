"""Brute-force search on the matrix cores: exact lists at the edges of its
tiles, and where its bound is loose, its buffer overflows or the coordinates
are not ordinary numbers."""
import numpy as np
import pytest

from gpusteer_amd import scenarios

pytestmark = pytest.mark.gpu


def _group(gs, ctx, pos):
    n = pos.shape[0]
    return gs.AgentGroup(ctx, scenarios.make_agents(pos, np.tile([[0.0, 0.0, 1.0]], (n, 1)), np.zeros(n), 0.5, 1.0, 1.0))


def _search(gs, ctx, a, b, k, bins=None):
    A = _group(gs, ctx, a)
    B = A if b is None else _group(gs, ctx, b)
    if bins is not None:  # storage order is then not agent order
        for G in {A, B}:
            gs.updateKNNDatabase(G, bins)
    knn = gs.KNNData(ctx, a.shape[0], k)
    gs.findKNearestNeighborsBruteForce(A, knn, B)
    out = knn.download()
    for h in (knn, A) + (() if b is None else (B,)):
        h.close()
    return out


def _reference(a, b, k, same, rows):
    """Keys (fp32 d2, index) with d2 a number, as the search defines them."""
    idx = np.full((k, len(rows)), 0xFFFFFFFF, np.uint32)
    dist = np.full((k, len(rows)), np.finfo(np.float32).max, np.float32)
    with np.errstate(all="ignore"):
        for c, r in enumerate(rows):
            d = a[r] - b
            d2 = (d[:, 0] * d[:, 0] + d[:, 1] * d[:, 1]) + d[:, 2] * d[:, 2]
            ok = ~np.isnan(d2)
            if same:
                ok[r] = False
            j = np.nonzero(ok)[0]
            j = j[np.lexsort((j, d2[j]))][:k]
            idx[:len(j), c], dist[:len(j), c] = j, np.sqrt(d2[j])
    return idx, dist


def _check(gs, ctx, a, b, k, bins=None):
    rows = np.unique(np.linspace(0, a.shape[0] - 1, 150).astype(np.int64))
    idx, dist = _search(gs, ctx, a, b, k, bins)
    r_idx, r_dist = _reference(a, a if b is None else b, k, b is None, rows)
    np.testing.assert_array_equal(idx[:, rows], r_idx)
    np.testing.assert_array_equal(dist[:, rows], r_dist)


@pytest.mark.parametrize("na,nb,k", [
    (1, 0, 3), (2, 0, 7), (15, 0, 16), (16, 0, 7), (17, 1, 7), (63, 0, 1), (64, 65, 32), (65, 64, 7), (300, 40, 32),
    (1000, 0, 32), (4096, 0, 7), (4097, 1023, 8), (8192, 0, 9), (8193, 5000, 16), (16389, 0, 7), (500, 20000, 4)])
def test_tile_edges(gs, ctx, na, nb, k):
    print(f"case na={na} nb={nb} k={k}", flush=True)
    g = np.random.default_rng(na + nb)
    a = g.uniform(-50, 50, (na, 3)).astype(np.float32)
    b = g.uniform(-50, 50, (nb, 3)).astype(np.float32) if nb else None
    _check(gs, ctx, a, b, k)
    bins = gs.KNNBinData(ctx, (7, 7, 7), (100.0,) * 3)
    _check(gs, ctx, a, b, k, bins)
    bins.close()


# Both sides of the line between a lane per query and the matrix cores.
@pytest.mark.parametrize("na,nb,k", [
    (100, 18, 7), (100, 19, 7), (17, 0, 7), (16384, 109, 7), (16384, 110, 7), (20000, 100, 16), (20000, 80, 32),
    (131072, 958, 7), (131072, 960, 7), (300001, 700, 5), (100000, 1, 16), (4097, 0, 1)])
def test_few_points_for_many_queries(gs, ctx, na, nb, k):
    print(f"case na={na} nb={nb} k={k}", flush=True)
    g = np.random.default_rng(na + nb)
    a = g.uniform(-50, 50, (na, 3)).astype(np.float32)
    b = g.uniform(-50, 50, (nb, 3)).astype(np.float32) if nb else None
    if nb > 20:
        b[:9], b[11] = b[9], (np.nan, 0.0, np.inf)
    bins = gs.KNNBinData(ctx, (7, 7, 7), (100.0,) * 3)
    _check(gs, ctx, a, b, k, bins)
    bins.close()


def _cases():
    g = np.random.default_rng(1)
    u = g.uniform(-1, 1, (2500, 3))
    yield "ties", np.round(u * 4)                                    # hundreds of points per position
    yield "one place", np.zeros((700, 3)) + 3.25
    yield "two far clusters", np.where(np.arange(2500)[:, None] % 2, u, u + 1e6)
    yield "far from the origin", u * 30 + [1e5, -2e5, 3e5]
    yield "tiny", u * 1e-22
    yield "a line", u * [1e4, 0.0, 0.0]
    far = u * 10
    far[::7] *= 1e18
    yield "squares that overflow", far * 1e2
    odd = u * 10
    odd[3], odd[50], odd[51], odd[1250] = (np.nan, 0, 0), (np.inf, 1, 1), (1, -np.inf, np.inf), (np.nan,) * 3
    yield "not numbers", odd


@pytest.mark.parametrize("name,pos", list(_cases()), ids=lambda v: v if isinstance(v, str) else "")
@pytest.mark.parametrize("k", [7, 32])
def test_positions(gs, ctx, name, pos, k):
    print(f"case {name} k={k}", flush=True)
    with np.errstate(all="ignore"):
        pos = pos.astype(np.float32)
    _check(gs, ctx, pos, None, k)
    _check(gs, ctx, pos[:900], pos, k)
