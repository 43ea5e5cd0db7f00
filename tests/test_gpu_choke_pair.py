"""Crowd frames phase by phase for both groups (gs_step_choke of small groups)
against the separate calls: the whole state, storage order and every list."""
import ctypes as C

import numpy as np
import pytest

from gpusteer_amd import _capi as capi
from gpusteer_amd import scenarios
from gpusteer_amd.ensemble import choke_step_calls, step_choke
from gpusteer_amd.state import WallState

from helpers import assert_state_equal

pytestmark = pytest.mark.gpu


def _world(gs, ctx, sc, k):
    bins = gs.KNNBinData(ctx, sc.grid_cells, sc.grid_size, origin=sc.grid_origin)
    G = [gs.AgentGroup(ctx, st) for st in sc.groups]
    W, O = gs.WallGroup(ctx, sc.walls), gs.ObstacleGroup(ctx, *sc.obstacles)
    for g in (W, O):
        gs.updateKNNDatabase(g, bins)
    knns = [[gs.KNNData(ctx, st.n, kk) for kk in (k, k, sc.knw, sc.kno)] for st in sc.groups]
    return bins, G, W, O, knns


def _result(G, knns, cells):
    return ([g.download() for g in G], [g.download_bins(cells) for g in G], [x.download() for ks in knns for x in ks])


def _equal(a, b):
    for x, y in zip(a[0], b[0]):
        assert_state_equal(x, y)
    for xs, ys in zip(a[1] + a[2], b[1] + b[2]):
        for x, y in zip(xs, ys):
            np.testing.assert_array_equal(x, y)


def _joint_frames(ctx):
    n = C.c_uint64()
    capi.check(capi.lib.gs_debug_joint_frames(ctx.h, C.byref(n)), "gs_debug_joint_frames")
    return n.value


def _scenario(n0, n1, gap, mode, cells, obstacles=50, walls=True):
    sc = scenarios.choke(n_total=2 * max(n0, n1), gap=gap, n_obstacles=obstacles, workload=n0 + n1)
    # the groups start across the wall from each other, so that they meet and touch it within a few frames
    for st, n in zip(sc.groups, (n0, n1)):
        st.arrays["pz"] *= np.float32(0.12)
    sc.groups = (sc.groups[0].subset(np.arange(n0)), sc.groups[1].subset(np.arange(n1)))
    sc.mode, sc.grid_cells = mode, cells
    if mode == 1:
        sc.sep = scenarios.FlockTerm(1.5, 3.0, -0.707, 10.0, 4096)
    if not walls:
        sc.walls = WallState({f: v[:0].copy() for f, v in sc.walls.arrays.items()})
    return sc


# The last two take the separate calls (a group or a lattice beyond one block's
# scan).
@pytest.mark.parametrize("n0,n1,k,mode,cells,obstacles,walls,other", [
    (1, 1, 7, 0, (40, 1, 40), 50, True, 3.5), (3, 700, 7, 1, (40, 1, 40), 2, True, 3.5),
    (1500, 1000, 8, 0, (40, 1, 40), 0, True, 3.5), (1000, 1501, 3, 1, (128, 1, 128), 50, False, 3.5),
    (2500, 2500, 7, 0, (40, 1, 40), 50, True, 0.0), (16384, 300, 7, 1, (100, 1, 100), 200, True, 3.5),
    (16385, 300, 7, 0, (100, 1, 100), 50, True, 3.5), (700, 700, 7, 0, (129, 1, 129), 50, True, 3.5)])
def test_equals_separate_calls(gs, ctx, n0, n1, k, mode, cells, obstacles, walls, other):
    print(f"case n={n0},{n1} k={k} mode={mode} cells={cells}", flush=True)
    sc = _scenario(n0, n1, 9.0, mode, cells, obstacles, walls)
    sc.other_radius = other if other > 0 else float("inf")
    frames = 12
    bins, G, W, O, knns = _world(gs, ctx, sc, k)
    for _ in range(frames):
        choke_step_calls(G, knns, W, O, bins, sc)
    want = _result(G, knns, bins.num_cells)
    moved = any((st["px"] != r["px"]).any() for st, r in zip(sc.groups, want[0]))
    assert moved
    bins2, G2, W2, O2, knns2 = _world(gs, ctx, sc, k)
    joint = 1 if max(n0, n1, bins.num_cells) <= 16384 else 0
    before = _joint_frames(ctx)
    for parts in ((frames,), (1, 4, frames - 5)):
        for g, st in zip(G2, sc.groups):
            g.upload(st)
        for p in parts:
            step_choke(G2, knns2, W2, O2, bins2, sc, p)
        _equal(_result(G2, knns2, bins2.num_cells), want)
    assert _joint_frames(ctx) - before == 2 * frames * joint
    # mixed with separate calls, and replayed from a recorded frame
    for g, st in zip(G2, sc.groups):
        g.upload(st)
    for _ in range(2):
        choke_step_calls(G2, knns2, W2, O2, bins2, sc)
        step_choke(G2, knns2, W2, O2, bins2, sc, 1)
    with ctx.record(lambda: step_choke(G2, knns2, W2, O2, bins2, sc, 2)) as f:
        f.launch((frames - 4) // 2)
    _equal(_result(G2, knns2, bins2.num_cells), want)
    for h in [bins, W, O, bins2, W2, O2] + G + G2 + [x for ks in knns + knns2 for x in ks]:
        h.close()


def test_buffers_end_as_with_separate_calls(gs, ctx):
    """A recorded frame can be replayed when it ends in the buffers in which it
    began: searches for display before the frame's own make it so, with the
    separate calls and with the joint frame."""
    sc = _scenario(900, 700, 9.0, 0, (40, 1, 40))
    results = []
    for calls in (choke_step_calls, step_choke):
        bins, G, W, O, knns = _world(gs, ctx, sc, 7)

        def frame():
            for g in G:
                gs.updateKNNDatabase(g, bins)
            for g, other, (own, oth, wall, obs) in zip(G, G[::-1], knns):
                gs.findKNearestNeighbors(g, own, bins, g, 1)
                gs.findKNearestNeighborsWithin(g, oth, bins, other, sc.other_radius, 1)
                gs.findKNearestNeighbors(g, wall, bins, W, 1)
                gs.findKNearestNeighbors(g, obs, bins, O, 1)
            calls(G, knns, W, O, bins, sc)

        for _ in range(2):
            frame()
        with ctx.record(frame) as f:
            f.launch(1)
            f.launch(5)
        results.append(_result(G, knns, bins.num_cells))
        for h in [bins, W, O] + G + [x for ks in knns for x in ks]:
            h.close()
    _equal(*results)
