"""Rows of points in subdivided layers: counted per point where the batch covers the points, sorted where it covers few of
them or a point meets more pieces than a run holds. Against the oracle to the bit, in the oracle's order of keys."""
import json

import numpy as np
import pytest

import gsj
from oracle import oracle as O
from conftest import sorted_rows

pytestmark = pytest.mark.gpu


def _mesh(n, seed, **kw):
    return gsj.generate("parcels_mesh", nx=n, ny=n, w=1 / 1549, h=1 / 1549, seed=seed, **kw)


def _stack(M, k):
    """k copies of the layer's polygons, so that every point meets k pieces at least"""
    sets = [M] * k
    ng, nr = M.n, len(M.rvo) - 1
    gro = np.concatenate([M.gro[:-1] + i * nr for i in range(k)] + [[k * nr]])
    rvo = np.concatenate([M.rvo[:-1] + i * len(M.xy) for i in range(k)] + [[k * len(M.xy)]])
    assert len(gro) == k * ng + 1
    return gsj.HostSet(gro.astype(np.uint64), rvo.astype(np.uint64), np.concatenate([s.xy for s in sets]))


def _check(ctx, xy, layer):
    got = ctx.points_in_polygons(ctx.points(xy), ctx.polys(layer))
    exp = O.points_join(O.Layer.points_layer(xy), O.Layer.polys(layer))
    g, e = sorted_rows(got.pairs, got.where), sorted_rows(exp["pairs"], exp["where"])
    assert np.array_equal(g[0], e[0]) and np.array_equal(g[1], e[1])
    return got, e


def _points(M, n, seed):
    """n points over the layer's box and some on its vertices and edge midpoints"""
    rng = np.random.default_rng(seed)
    lo, hi = M.xy.min(0), M.xy.max(0)
    return np.concatenate([lo + (hi - lo) * rng.random((n, 2)), M.xy[::5], 0.5 * (M.xy[:-1:7] + M.xy[1::7])])


# pieces with packed records only, and with long rings that have none; one point to more than a block of them
@pytest.mark.parametrize("maxv", [0, 5, 10, 64, 200])
@pytest.mark.parametrize("n", [1, 255, 257, 20000])
def test_points_per_piece_size(ctx, n, maxv):
    M = gsj.generate("regions_grid", nx=30, ny=30, kx=3, ky=3, edge_segs=100, seed=n) if maxv in (0, 200) else _mesh(20, n)
    got, e = _check(ctx, _points(M, n, n), gsj.subdivide(M, maxv) if maxv else M)
    assert (e[1] == 2).any()


# few of the points lie in the layer; from 8M points on the rows of such a batch are sorted
@pytest.mark.parametrize("far", [0, 6, 100, (8 << 20) - 2000, 8 << 20])
def test_points_mostly_elsewhere(ctx, far):
    M = _mesh(16, 4)
    xy = _points(M, 900, 4)
    out = np.random.default_rng(far).random((far, 2)) + [5.0, 0.0]
    _check(ctx, np.concatenate([out[: far // 2], xy, out[far // 2 :]]), gsj.subdivide(M, 8))


# 1 to 40 layers on top of each other: up to, at and beyond the length of a run (16 candidates)
@pytest.mark.parametrize("k", [1, 4, 8, 15, 16, 17, 40])
def test_points_in_stacked_pieces(ctx, k):
    M = _mesh(6, 9)
    got, _ = _check(ctx, _points(M, 3000, k), gsj.subdivide(_stack(M, k), 8))
    assert (np.diff(got.pairs[:, 0].astype(np.int64)) >= 0).all()


def test_stacked_pieces_take_one_way(ctx):
    # one point with more pieces than a run holds sends its batch to the sort; the counters and offsets that the other way
    # keeps for every point of the layer (12 bytes each) are then not set up at all, let alone run through
    M, n = _mesh(6, 9), 4 << 20
    S, near = gsj.subdivide(_stack(M, 17), 8), _points(M, 300, 2)
    xy = np.concatenate([np.random.default_rng(1).random((n, 2)) + [5.0, 0.0], near])
    own = gsj.Context(0)
    try:
        pts, plain, stacked = own.points(xy), own.polys(M), own.polys(S)
        own.points_in_polygons(pts, plain)   # the search's buffers; no subdivided layer, no fold
        free = json.loads(own.status())["mem_free_mb"]
        got = own.points_in_polygons(pts, stacked)
        assert (free - json.loads(own.status())["mem_free_mb"]) * 2**20 < 12 * n
        exp = O.points_join(O.Layer.points_layer(near), O.Layer.polys(S))
        g, e = sorted_rows(got.pairs, got.where), sorted_rows(exp["pairs"] + np.array([n, 0], np.uint32), exp["where"])
        assert len(e[0]) and np.array_equal(g[0], e[0]) and np.array_equal(g[1], e[1])
    finally:
        own.close()
