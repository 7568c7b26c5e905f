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


FOLD_MAX = 4096   # the most candidates that one block folds


def _folded(ctx, P, R, upper):
    """the candidates that go to the fold: piece pairs that meet, of a parent of several pieces on either side"""
    pairs = ctx.join(ctx.polys(P), ctx.polys(R), upper=upper, want_area=True, no_agg=True).pairs
    several = [np.zeros(S.n, bool) if S.parent is None else np.bincount(S.parent - S.parent[0])[S.parent - S.parent[0]] > 1 for S in (P, R)]
    return int((several[0][pairs[:, 0]] | several[1][pairs[:, 1]]).sum())


def _check(ctx, P, R, upper, what, entries=(False,)):
    LP, LR = ctx.polys(P), ctx.polys(R)
    exp = O.join(O.Layer.polys(P), O.Layer.polys(R), upper=upper, **{what: True})
    col = "area" if what == "want_area" else "code"
    for noalloc in entries:
        got = ctx.join(LP, LR, upper=upper, noalloc=noalloc, **{what: True})
        g, e = sorted_rows(got.pairs, getattr(got, col)), sorted_rows(exp["pairs"], exp[col])
        assert np.array_equal(g[0], e[0]) and np.array_equal(g[1], e[1])
    return got


# from a handful of folded candidates to about a hundred thousand; 17 to 20 cells a side at 8 vertices lie around the
# block's 4096
@pytest.mark.parametrize("n,maxv", [(4, 8), (12, 16), (17, 8), (18, 8), (20, 8), (34, 8), (36, 8), (40, 32), (90, 8)])
@pytest.mark.parametrize("what", ["want_area", "want_relate"])
def test_self_join_of_pieces(ctx, n, maxv, what):
    S = gsj.subdivide(_mesh(n, n), maxv)
    assert (_folded(ctx, S, S, True) <= FOLD_MAX) == (n < 18 or maxv > 8)
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


def _bits(v):
    return max(1, int(v).bit_length())


def _key_bits(P, R):
    """bits of a folded candidate's key: both parents, and both pieces within their parents"""
    return sum(_bits(S.parent[-1]) + _bits(np.bincount(S.parent - S.parent[0]).max() - 1) for S in (P, R))


def _cells(k, last):
    """one parent, of id `last`, cut into k x k cells of unequal sizes; the cuts are synthetic edges"""
    rng = np.random.default_rng(k)
    x, y = (np.concatenate([[0.0], np.cumsum(0.5 + rng.random(k))]) * 1e-4 - o for o in (95.0, -38.0))
    i, j = (a.ravel() for a in np.meshgrid(np.arange(k), np.arange(k), indexing="ij"))
    x0, x1, y0, y1 = x[i], x[i + 1], y[j], y[j + 1]
    xy = np.stack([np.stack([x0, x1, x1, x0, x0], 1), np.stack([y0, y0, y1, y1, y0], 1)], 2)
    syn = np.stack([j > 0, i < k - 1, j < k - 1, i > 0, np.zeros(k * k, bool)], 1)
    n = k * k
    return gsj.HostSet(np.arange(n + 1, dtype=np.uint64), 5 * np.arange(n + 1, dtype=np.uint64), xy.reshape(-1, 2),
                       np.full(n, last, np.uint32), syn.reshape(-1).astype(np.uint8))


# the last piece of the last parent with itself, where both ids have all their bits set: its key is the largest there is,
# 64 bits of ones at 2^24 parents and 256 pieces
@pytest.mark.parametrize("bits", [23, 24, 25])
@pytest.mark.parametrize("what", ["want_area", "want_relate"])
def test_the_largest_key(ctx, bits, what):
    S = _cells(16, 2**bits - 1)
    assert _key_bits(S, S) == 2 * bits + 16
    _check(ctx, S, S, True, what, (False, True))


def _renumbered(S, step):
    """the pieces of S under parent ids `step` apart"""
    return gsj.HostSet(S.gro, S.rvo, S.xy, S.parent * np.uint32(step), S.syn)


# keys up to and beyond 63 bits (from 64 on the candidates are sorted twice, by piece pair and by parent pair), few and many
# candidates: regions of hundreds of pieces under ids millions apart, with themselves and with parcels of a few pieces
@pytest.mark.parametrize("k,segs", [(2, 110), (2, 250), (3, 500)])
@pytest.mark.parametrize("what", ["want_area", "want_relate"])
def test_wide_keys(ctx, k, segs, what):
    R = gsj.subdivide(gsj.generate("regions_grid", nx=30, ny=30, kx=k, ky=k, edge_segs=segs, seed=segs), 8)
    P = gsj.subdivide(gsj.generate("parcels_grid", nx=30, ny=30, seed=segs, kmin=9, kmax=30), 8)
    assert R.parent[-1] < P.parent[-1] and P.n > P.parent[-1] + 1
    last = int(R.parent[-1])
    for bits in (62, 64, 66):
        half = (bits - _key_bits(_renumbered(R, 1), _renumbered(R, 1))) // 2 + _bits(last)
        S = _renumbered(R, 2 ** (half - 1) // last + 1)
        assert _key_bits(S, S) == bits
        assert (_folded(ctx, S, S, True) > FOLD_MAX) == (segs > 110)
        _check(ctx, S, S, True, what, (False, True) if segs == 110 else (False,))
    narrow = max(q for q in range(9, 28) if _key_bits(_renumbered(P, 2 ** (q - 9)), _renumbered(R, 2**q)) <= 63)
    for q in (narrow, narrow + 1):
        _check(ctx, _renumbered(P, 2 ** (q - 9)), _renumbered(R, 2**q), False, what)
