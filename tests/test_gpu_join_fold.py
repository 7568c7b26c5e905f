"""Piece pairs folded into parent pairs: in one block up to 4096 candidates, sorted by the radix sort beyond; rows written
into host memory or, by the no-allocation entry point, copied. Against the oracle to the bit."""
import numpy as np
import pytest

import gsj
from oracle import oracle as O
from conftest import sorted_rows

pytestmark = pytest.mark.gpu


def _mesh(n, seed, **kw):
    return gsj.generate("parcels_mesh", nx=n, ny=n, w=1 / 1549, h=1 / 1549, seed=seed, **kw)


def _check(ctx, P, R, upper, what, entries=(False,)):
    LP, LR = ctx.polys(P), ctx.polys(R)
    exp = O.join(O.Layer.polys(P), O.Layer.polys(R), upper=upper, **{what: True})
    col = "area" if what == "want_area" else "code"
    for noalloc in entries:
        got = ctx.join(LP, LR, upper=upper, noalloc=noalloc, **{what: True})
        g, e = sorted_rows(got.pairs, getattr(got, col)), sorted_rows(exp["pairs"], exp[col])
        assert np.array_equal(g[0], e[0]) and np.array_equal(g[1], e[1])
    return got


# from a handful of folded candidates to about a hundred thousand; 34 x 34 at 8 vertices lies around the block's 4096
@pytest.mark.parametrize("n,maxv", [(4, 8), (12, 16), (20, 8), (34, 8), (36, 8), (40, 32), (90, 8)])
@pytest.mark.parametrize("what", ["want_area", "want_relate"])
def test_self_join_of_pieces(ctx, n, maxv, what):
    S = gsj.subdivide(_mesh(n, n), maxv)
    _check(ctx, S, S, True, what, (False, True) if n <= 40 else (False,))


@pytest.mark.parametrize("sub", [(0, 8), (8, 0), (16, 8)])
def test_one_or_both_layers_subdivided(ctx, sub):
    P, R = (gsj.subdivide(M, s) if s else M for M, s in zip((_mesh(30, 5), _mesh(30, 6, jitter=0.05)), sub))
    for what in ("want_area", "want_relate"):
        _check(ctx, P, R, False, what)


def test_one_parent_of_many_pieces(ctx):
    # a region of 2000 edges cut to 8 vertices: hundreds of pieces of one parent, thousands of piece pairs in one row
    R = gsj.subdivide(gsj.generate("regions_grid", nx=30, ny=30, kx=1, ky=1, edge_segs=500, seed=1), 8)
    P = gsj.generate("parcels_grid", nx=30, ny=30, seed=2)
    for what in ("want_area", "want_relate"):
        _check(ctx, P, R, False, what)
        _check(ctx, R, R, True, what)


@pytest.mark.parametrize("n,maxv", [(12, 8), (70, 8), (70, 64)])
def test_clusters_of_pieces(ctx, n, maxv):
    S = gsj.subdivide(_mesh(n, 3 * n), maxv)
    assert np.array_equal(ctx.cluster(ctx.polys(S))[0], O.cluster(O.Layer.polys(S))["root"])
