"""Joins of few candidates (all classes in two launches, one-block partition and scans, rows written into host memory) at
the edges of their ranges, against the oracle to the bit and against the no-allocation entry point, whose rows take the
other way to the host."""
import numpy as np
import pytest

import gsj
from oracle import oracle as O
from conftest import sorted_rows

pytestmark = pytest.mark.gpu


def _check(ctx, P, R, noalloc=True, **kw):
    LP, LR = ctx.polys(P), ctx.polys(R)
    exp = O.join(O.Layer.polys(P), O.Layer.polys(R), **kw)
    for got in [ctx.join(LP, LR, **kw)] + ([ctx.join(LP, LR, noalloc=True, **kw)] if noalloc else []):
        assert got.stats["candidates"] == exp["candidates"]
        col = "area" if kw.get("want_area") else "code"
        g, e = sorted_rows(got.pairs, getattr(got, col)), sorted_rows(exp["pairs"], exp[col])
        assert np.array_equal(g[0], e[0]) and np.array_equal(g[1], e[1])
    return got


# a parcel of a grid meets only itself: as many candidates as parcels. 1024: one element per thread of a block's scan or
# partition, 16384: their largest, 32768: the most that take the two stages
@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 1023, 1025, 2047, 16383, 16384, 16385, 32767, 32768, 32769])
def test_candidate_counts_at_the_edges(ctx, n):
    P = gsj.generate("parcels_grid", nx=n, ny=1, seed=n, x0=-100.0)   # (gaps of 1e-4 degrees: no float box meets the next)
    got = _check(ctx, P, P, noalloc=n <= 16385, want_area=True, upper=True)
    assert got.stats["candidates"] == n
    assert got.stats["n_tiny"] + got.stats["n_small"] == n


@pytest.mark.parametrize("n,median", [(3, 7.0), (12, 30.0), (30, 7.0), (50, 20.0)])
@pytest.mark.parametrize("what", ["want_area", "want_relate"])
def test_every_class_in_the_stages(ctx, n, median, what):
    # lognormal vertex counts: tiny to large pairs, spills and overflow lists among them
    M = gsj.generate("parcels_mesh", nx=n, ny=n, w=1 / 1549, h=1 / 1549, seed=n, median=median, kmax=400)
    _check(ctx, M, M, upper=True, **{what: True})


@pytest.mark.parametrize("segs", [3, 20, 110, 120, 300])
def test_lists_handed_to_the_host(ctx, segs):
    # whole borders in one window: 96, 448 and more edges per side; the longest lists are refined after the rows were
    # first compacted, and the rows are compacted again
    R = gsj.generate("regions_grid", nx=20, ny=20, kx=3, ky=3, edge_segs=segs, seed=segs)
    P = gsj.generate("parcels_grid", nx=20, ny=20, seed=1)
    got = _check(ctx, R, R, want_area=True, upper=True)
    if segs >= 120:
        assert got.stats["n_over"] > 0
    _check(ctx, P, R, want_relate=True)
