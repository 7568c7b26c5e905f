"""The phase times of a call: the refinement's hold its kernels' device times, on every way a request can take, and the
phases together do not exceed the call."""
import time

import numpy as np
import pytest

import gsj

pytestmark = pytest.mark.gpu


def _mesh(n, seed, **kw):
    return gsj.generate("parcels_mesh", nx=n, ny=n, w=1 / 1549, h=1 / 1549, seed=seed, **kw)


def _timed(call):
    call()   # scratch of its size is there
    t = time.perf_counter()
    s = call().stats
    ms = 1e3 * (time.perf_counter() - t)
    assert s["traverse_ms"] + s["refine_ms"] + s["compact_ms"] + s["copy_ms"] <= ms
    assert s["compact_ms"] > 0
    return s


@pytest.mark.parametrize("maxv", [0, 16])
def test_points(ctx, maxv):
    M = _mesh(60, 1)
    lo, hi = M.xy.min(0), M.xy.max(0)
    P, L = ctx.points(lo + (hi - lo) * np.random.default_rng(2).random((2_000_000, 2))), ctx.polys(gsj.subdivide(M, maxv) if maxv else M)
    s = _timed(lambda: ctx.points_in_polygons(P, L))
    assert s["refine_ms"] >= s["k_small_ms"] > 0


# 32768 candidates at most: one wait for all classes and the rows; more: one after the classes
@pytest.mark.parametrize("n,kw", [(80, {}), (60, {"median": 40.0, "kmax": 400}), (100, {})])
@pytest.mark.parametrize("what", ["want_area", "want_relate"])
def test_joins(ctx, n, kw, what):
    L = ctx.polys(_mesh(n, n, **kw))
    s = _timed(lambda: ctx.join(L, L, upper=True, **{what: True}))
    kernels = max(s["k_screen_ms"], s["k_mixed_ms"]) + max(s["k_tiny_ms"], s["k_small_ms"], s["k_medium_ms"], s["k_large_ms"])
    assert s["refine_ms"] >= kernels > 0


def test_lists_refined_after_the_wait(ctx):
    # whole borders of 1200 edges in one window: their pairs are refined behind the first compaction
    L = ctx.polys(gsj.generate("regions_grid", nx=20, ny=20, kx=3, ky=3, edge_segs=300, seed=3))
    s = _timed(lambda: ctx.join(L, L, upper=True, want_area=True))
    assert s["refine_ms"] >= s["k_over_ms"] > 0
