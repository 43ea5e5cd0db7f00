"""Per-agent kernels run in blocks of one wavefront for small groups: sizes at
the edges of a wavefront and of that rule, the fused step and the same step by
separate calls, both modes."""
import numpy as np
import pytest

from gpusteer_amd import scenarios
from helpers import assert_state_equal
from test_gpu_step import _separate_calls_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 63, 64, 65, 32768, 32769])
@pytest.mark.parametrize("mode,k", [(0, 7), (1, 5)])
def test_step_at_block_edges(gs, ctx, orc, n, mode, k):
    print(f"case n={n} mode={mode} k={k}", flush=True)
    st, p = scenarios.boids_sphere(n=n, radius=50.0 if n > 100 else 10.0)
    p.mode, p.k = mode, k
    ref = st.copy()
    for _ in range(2):
        r_idx, r_dist = orc.boids_step(ref, p)
    for fused in (True, False):
        A = gs.AgentGroup(ctx, st)
        bins = gs.KNNBinData(ctx, p.grid_cells, p.grid_size, origin=p.grid_origin)
        knn = gs.KNNData(ctx, n, k)
        for _ in range(2):
            if fused:
                gs.stepBoids(A, knn, bins, p, 1)
            else:
                _separate_calls_step(gs, A, knn, bins, p)
        idx, dist = knn.download()
        np.testing.assert_array_equal(idx, r_idx)
        np.testing.assert_array_equal(dist, r_dist)
        assert_state_equal(A.download(), ref, what=f"fused {fused}: ")
        for h in (knn, bins, A):
            h.close()
