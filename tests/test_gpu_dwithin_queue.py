"""The distance joins' put-off work vs the oracle: edge pairs inside the error band (decided by a kernel of their own),
item queues that fill, overflow lists in LDS and beyond, and long pieces against points. Rows and distances are the
oracle's to the bit: both sides take the same FP64 operations of the shared geodesy, whatever kernel takes them."""
import numpy as np
import pytest

import gsj
from oracle import oracle as O
from conftest import sorted_rows

pytestmark = pytest.mark.gpu

LON, LAT = -95.2, 38.6


def _circle(n, x, y, r, phase=0.1):
    """closed CCW ring of n vertices, centre (x, y) and radius r in metres from (LON, LAT)"""
    kx, ky = O.m_per_deg(LAT)
    t = phase + 2 * np.pi * np.arange(n) / n
    ring = np.stack([LON + (x + r * np.cos(t)) / kx, LAT + (y + r * np.sin(t)) / ky], axis=1)
    return np.concatenate([ring, ring[:1]])


def _layer(polys):
    """polys: lists of rings"""
    rings = [r for p in polys for r in p]
    return gsj.HostSet(np.cumsum([0] + [len(p) for p in polys]), np.cumsum([0] + [len(r) for r in rings]), np.concatenate(rings))


def _same(got, exp, report):
    g, e = sorted_rows(got.pairs, got.dist if report else None), sorted_rows(exp["pairs"], exp["dist"] if report else None)
    assert np.array_equal(g[0], e[0])
    if report:
        assert np.array_equal(g[1], e[1])


def _polygons(ctx, A, B, d):
    a, b = _layer(A), _layer(B)
    LA, LB, OA, OB = ctx.polys(a), ctx.polys(b), O.Layer.polys(a), O.Layer.polys(b)
    for report in (False, True):
        exp = O.dwithin(OA, OB, d, report=report)
        got = ctx.dwithin(LA, LB, d, report_distance=report)
        _same(got, exp, report)
    return got, exp


def _points(ctx, xy, B, d):
    b = _layer(B)
    LP, LB, OP, OB = ctx.points(xy), ctx.polys(b), O.Layer.points_layer(xy), O.Layer.polys(b)
    for report in (False, True):
        exp = O.points_dwithin(OP, OB, d, report=report)
        got = ctx.points_dwithin(LP, LB, d, report_distance=report)
        _same(got, exp, report)
    return got, exp


# vertices of both sides: the tiny, small, medium, mixed and large classes' edges, the LDS overflow lists (129 to 448
# edges) and longer ones
@pytest.mark.parametrize("n,m", [(4, 15), (16, 16), (31, 31), (32, 63), (63, 63), (20, 90), (70, 130), (200, 400), (30, 447), (449, 700)])
def test_distance_at_the_threshold(ctx, n, m):
    A, B = [[_circle(n, 0, 0, 40)]], [[_circle(m, 120, 30, 50, 0.3)]]
    d0 = O.dwithin(O.Layer.polys(_layer(A)), O.Layer.polys(_layer(B)), 100.0, report=True)["dist"][0]
    for d in (d0, np.nextafter(d0, 0), d0 * (1 - 1e-9), d0 * (1 + 1e-9), d0 - 1.0, 5 * d0):
        _polygons(ctx, A, B, float(d))


@pytest.mark.parametrize("n", [16, 32, 64, 128, 300])
def test_more_items_than_the_queue_holds(ctx, n):
    # 20 km apart every edge pair lies inside the band of the closest one: n * n items of one pair
    got, _ = _polygons(ctx, [[_circle(n, 0, 0, 5)], [_circle(4, 0, 300, 5)]], [[_circle(n, 20000, 0, 5)], [_circle(5, 20000, 200, 5)]], 25000.0)
    assert len(got.pairs) == 4


@pytest.mark.parametrize("n", [3, 63, 64, 65, 128, 129, 1000])
def test_points_near_long_pieces(ctx, n):
    rng = np.random.default_rng(n)
    hole = _circle(max(3, n // 2), 0, 0, 20)[::-1].copy()
    B = [[_circle(n, 0, 0, 60), hole], [_circle(n, 200, 0, 60)], [_circle(5, 60, 130, 30)]]
    kx, ky = O.m_per_deg(LAT)
    xy = np.stack([LON + rng.uniform(-150, 350, 400) / kx, LAT + rng.uniform(-150, 200, 400) / ky], axis=1)
    xy[:6] = [B[0][0][1], B[0][0][0] * 0.5 + B[0][0][1] * 0.5, B[0][1][0], B[1][0][2], [LON, LAT], [LON + 100 / kx, LAT]]
    got, exp = _points(ctx, xy, B, 25.0)
    far = exp["dist"][exp["dist"] > 0]
    for d in far[:3]:   # the threshold at a reported distance, and just below it
        _points(ctx, xy, B, float(d))
        _points(ctx, xy, B, float(np.nextafter(d, 0)))


def test_points_with_more_items_than_the_queue_holds(ctx):
    kx, ky = O.m_per_deg(LAT)
    xy = np.stack([LON + (20000 + np.arange(400.0)) / kx, np.full(400, LAT)], axis=1)
    _points(ctx, xy, [[_circle(60, 0, 0, 5)], [_circle(90, 0, 50, 5)]], 25000.0)
