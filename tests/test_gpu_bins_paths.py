"""Bin builds at the sizes where they change their passes (scan and scatter in
one block; builds of a multi-step call whose inner order is free), against a
stable sort and against single-step calls."""
import numpy as np
import pytest

from gpusteer_amd import scenarios

from helpers import assert_state_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cells", [
    (1, (1, 1, 1)), (2000, (32, 32, 16)), (2000, (32, 32, 17)), (16384, (16, 16, 16)), (16385, (16, 16, 16)),
    (16384, (16385, 1, 1)), (16385, (128, 128, 1)), (50000, (1, 16383, 1)), (9000, (3, 2, 1)),
    (5120, (10240, 1, 1)), (5120, (1, 10242, 1)), (5121, (4, 4, 4)), (4096, (12288, 1, 1)), (4096, (1, 1, 12289)),
    (2048, (16384, 1, 1)), (2049, (16384, 1, 1))])
def test_build_is_the_stable_sort(gs, ctx, orc, n, cells):
    print(f"case n={n} cells={cells}", flush=True)
    g = np.random.default_rng(n)
    size = (30.0, 30.0, 30.0)
    bins = gs.KNNBinData(ctx, cells, size, origin=(0.0,) * 3)
    A = None
    for _ in range(2):  # the second build starts from a clean or a used count array
        pos = g.uniform(-1.0, 31.0, (n, 3)).astype(np.float32)
        pos[: n // 3] = 3.0  # one crowded cell
        pos = pos[g.permutation(n)]
        st = scenarios.make_agents(pos, np.tile([[0.0, 0.0, 1.0]], (n, 1)), np.zeros(n), 0.5, 1.0, 1.0)
        A = A or gs.AgentGroup(ctx)
        A.upload(st)
        for _ in range(2):
            gs.updateKNNDatabase(A, bins)
            key, start, perm, sp = A.download_bins(bins.num_cells)
            r_key, r_start, r_perm, r_sp = orc.bins_build(orc.grid((0.0,) * 3, size, cells), pos)
            np.testing.assert_array_equal(key, r_key)
            np.testing.assert_array_equal(start, r_start)
            np.testing.assert_array_equal(perm, r_perm)
            np.testing.assert_array_equal(sp, r_sp)
    for h in (A, bins):
        h.close()


@pytest.mark.parametrize("n,cells,wrap,mode", [
    (3000, (12, 12, 12), 1, 0), (20000, (16, 16, 16), 0, 1), (20001, (26, 26, 26), 0, 0), (40000, (32, 32, 32), 1, 0),
    (40000, (36, 36, 36), 1, 1), (70000, (32, 32, 64), 0, 0), (20000, (24, 24, 24), 1, 0), (20000, (1, 96, 128), 0, 0)])
def test_one_call_of_many_steps_equals_many_calls(gs, ctx, n, cells, wrap, mode):
    """The whole state, the storage order, the bins and the lists."""
    st, p = scenarios.boids_sphere(n=n)
    p.grid_cells, p.mode = cells, mode
    if wrap == 0:
        p.wrap_shape, p.wrap_size = 0, (80.0, 70.0, 90.0)
    got = []
    for parts in ((7,), (1,) * 7, (3, 4)):
        A = gs.AgentGroup(ctx, st)
        bins = gs.KNNBinData(ctx, p.grid_cells, p.grid_size, origin=p.grid_origin)
        knn = gs.KNNData(ctx, n, 7)
        for s in parts:
            gs.stepBoids(A, knn, bins, p, s)
        got.append((A.download(), A.download_bins(bins.num_cells), knn.download()))
        for h in (knn, bins, A):
            h.close()
    for other in got[1:]:
        assert_state_equal(got[0][0], other[0])
        for a, b in zip(got[0][1] + got[0][2], other[1] + other[2]):
            np.testing.assert_array_equal(a, b)
