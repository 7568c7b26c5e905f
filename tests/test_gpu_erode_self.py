"""Eroded intersects of a layer with itself: a parent's pair with itself is settled by a point well inside it, and its
overlap area in pass 1 by its ring sum. The rows are the oracle's, which takes every pair through the whole test: shapes
around the width, area and edge counts where those shortcuts end, and rings that turn the wrong way."""
import numpy as np
import pytest

import gsj
from oracle import oracle as O
from conftest import sorted_rows

pytestmark = pytest.mark.gpu

LON, LAT = -95.2, 38.6


def _ring(xy):
    kx, ky = O.m_per_deg(LAT)
    r = np.array([LON, LAT]) + np.asarray(xy, float) / [kx, ky]
    return np.concatenate([r, r[:1]])


def _box(x, y, w, h):
    return _ring([(x, y), (x + w, y), (x + w, y + h), (x, y + h)])


def _circle(n, x, y, r):
    t = 2 * np.pi * np.arange(n) / n
    return _ring(np.stack([x + r * np.cos(t), y + r * np.sin(t)], axis=1))


def _star(n, x, y, r0, r1):
    t = np.pi * np.arange(2 * n) / n
    r = np.where(np.arange(2 * n) % 2, r0, r1)
    return _ring(np.stack([x + r * np.cos(t), y + r * np.sin(t)], axis=1))


def _layer(polys):
    rings = [r for p in polys for r in p]
    return gsj.HostSet(np.cumsum([0] + [len(p) for p in polys]), np.cumsum([0] + [len(r) for r in rings]), np.concatenate(rings))


def _check(ctx, polys, ra, rb, need=None):
    hs = _layer(polys)
    L, OL = ctx.polys(hs), O.Layer.polys(hs)
    exp = O.erode(OL, OL, ra, rb, same=True, upper=True, need_self=need)
    got = ctx.intersects_buffered(L, L, ra, rb, same=True, upper=True, need_self=need)
    assert np.array_equal(sorted_rows(got.pairs)[0], sorted_rows(exp["pairs"])[0])
    return got, exp


RADII = [(2.0, 2.0), (2.0, 1.0), (0.5, 2.0), (2.0, 0.0)]


@pytest.mark.parametrize("ra,rb", RADII)
def test_widths_around_the_radius(ctx, ra, rb):
    r = max(ra, rb)
    w = [2 * r * f for f in (0.5, 0.98, 1 - 1e-6, 1 - 1e-9, 1.0, 1 + 1e-9, 1 + 1e-6, 1.0005, 1.005, 1.02, 1.2, 3.0)]
    shapes = [[_box(40.0 * i, 0, w[i], 30)] for i in range(len(w))] + [[_box(40.0 * i, 100, 30, w[i])] for i in range(len(w))]
    shapes += [[_circle(4, 40.0 * i, 200, w[i])] for i in range(len(w))] + [[_circle(60, 40.0 * i, 300, w[i] / 2)] for i in range(len(w))]
    _, exp = _check(ctx, shapes, ra, rb)
    assert 0 < len(exp["pairs"]) < len(shapes)


@pytest.mark.parametrize("ra,rb", RADII)
def test_shapes_and_rings(ctx, ra, rb):
    L = _ring([(0, 0), (20, 0), (20, 3), (3, 3), (3, 20), (0, 20)])   # both arms thinner than two radii, the corner too
    polys = [[L], [_star(5, 60, 0, 4, 15)], [_star(9, 120, 0, 1, 15)], [_star(40, 180, 0, 14, 15)],
             [_box(220, -15, 30, 30), _box(232, -3, 6, 6)[::-1].copy()],              # a hole in the middle
             [_box(270, -15, 30, 30), _box(273, -12, 24, 24)[::-1].copy()],           # a frame 3 m wide
             [_box(320, -15, 30, 30), _box(330, -5, 10, 10)],                         # a hole turning the wrong way
             [_box(370, -15, 30, 30)[::-1].copy()],                                   # a shell turning the wrong way
             [_ring([(420, 0), (450, 30), (450, 0), (420, 30)])],                     # bow-ties, one lobe either way
             [_ring([(470, 0), (474, 30), (500, 0), (472, 32)])],
             [_box(520, 0, 30, 30), _box(535, 15, 30, 30)],                           # overlapping shells of one geometry
             [_box(600, 0, 30, 30), _box(640, 0, 3, 3), _box(650, 0, 30, 3)]]
    _check(ctx, polys, ra, rb)
    need = np.arange(len(polys)) % 2 == 0
    _check(ctx, polys, ra, rb, need.astype(np.uint8))


@pytest.mark.parametrize("n", [16, 17, 63, 64, 65, 129, 1022, 1023, 1024, 1500])
def test_edge_counts(ctx, n):
    polys = [[_circle(n, 0, 0, 30)], [_circle(n, 100, 0, 2.001)], [_circle(n, 200, 0, 30), _circle(max(3, n // 2), 200, 0, 27)[::-1].copy()],
             [_circle(n, 20, 20, 30)]]
    for ra, rb in ((1.0, 2.0), (20.0, 1.0)):
        _check(ctx, polys, ra, rb)


@pytest.mark.parametrize("side", [0.98 * np.sqrt(np.pi) * 2.0 * f for f in (0.9, 1 - 1e-4, 1 - 1e-7, 1.0, 1 + 1e-7, 1.1)])
def test_areas_around_the_bound(ctx, side):
    # squares whose area is about the one that pass 1 asks for (a disk of 0.98 radii), and longer boxes of the same area
    _check(ctx, [[_box(0, 0, side, side)], [_box(50, 0, side / 3, 3 * side)], [_box(100, 0, 40, 40)]], 2.0, 2.0)


def test_a_mesh_of_every_size(ctx):
    M = gsj.generate("parcels_mesh", nx=45, ny=41, w=1 / 1549, h=1 / 1549, seed=11, median=12.0)
    OL, L = O.Layer.polys(M), ctx.polys(M)
    for ra, rb in ((0.5, 0.75), (8.0, 1.0), (20.0, 20.0)):
        exp = O.erode(OL, OL, ra, rb, same=True, upper=True)
        got = ctx.intersects_buffered(L, L, ra, rb, same=True, upper=True)
        assert np.array_equal(sorted_rows(got.pairs)[0], sorted_rows(exp["pairs"])[0])


def test_more_pairs_than_one_row_of_blocks(ctx):
    # 8200 boxes on one spot: 67.2M candidates, the last of them in the grid's second row; every pair meets
    n = 8200
    box = _box(0, 0, 30, 20)
    hs = gsj.HostSet(np.arange(n + 1, dtype=np.uint64), 5 * np.arange(n + 1, dtype=np.uint64), np.tile(box, (n, 1)))
    own = gsj.Context(0)   # (its scratch goes with it)
    try:
        L = own.polys(hs)
        got = own.intersects_buffered(L, L, 2.0, 1.0, same=True)
        seen = np.zeros(n * n, bool)
        seen[got.pairs[:, 0].astype(np.int64) * n + got.pairs[:, 1]] = True
        assert got.stats["candidates"] == n * n == len(got.pairs) and seen.all()
        assert len(own.intersects_buffered(L, L, 11.0, 1.0, same=True).pairs) == 0
    finally:
        own.close()
