"""Layer preparation where its kernels change over: geometries a lane takes and those a wave takes, few and many of them to
a wave, sorts of short and long tiles, clips of rings longer than one batch of loads. Against the oracle or the host."""
import numpy as np
import pytest

import gsj
from oracle import oracle as O

pytestmark = pytest.mark.gpu


def _rings(sizes, seed):
    """a star-shaped ring of each size (stored vertices, closed), some with a hole"""
    rng = np.random.default_rng(seed)
    gro, rvo, xy = [0], [0], []
    for i, m in enumerate(sizes):
        a = np.sort(rng.random(m - 1)) * 2 * np.pi
        for scale in (1.0, 0.3) if i % 3 == 0 else (1.0,):
            r = scale * (0.8 + 0.2 * rng.random(m - 1))[:, None]
            p = np.array([i % 100, i // 100]) * 2.5 - 95.0 + r * np.stack([np.cos(a), np.sin(a)], 1)
            xy.append(np.concatenate([p, p[:1]]))
            rvo.append(rvo[-1] + m)
        gro.append(len(rvo) - 1)
    return gsj.HostSet(np.array(gro, np.uint64), np.array(rvo, np.uint64), np.concatenate(xy))


def _check_prep(ctx, hs):
    d, o = ctx.polys(hs).export(), O.Layer.polys(hs).export()
    for k in ("origin", "ext", "bb", "q"):
        assert np.array_equal(d[k], o[k]), k
    return d, o


# boundary lengths: the device's hypot and the host's may differ in the last bit, but not for edges along an axis, whose
# sum then shows the order of its terms
@pytest.mark.parametrize("steps", [1, 30, 31, 32, 61, 62, 63, 64, 65, 1200])
def test_boundary_length_is_summed_in_order(ctx, steps):
    rng = np.random.default_rng(steps)
    rings = []
    for i in range(3):
        x, y = np.cumsum(rng.random(steps)), np.cumsum(rng.random(steps))
        stair = np.stack([np.repeat(x, 2), np.concatenate([[0.0], np.repeat(y, 2)[:-1]])], 1)
        p = np.concatenate([[[0.0, 0.0]], stair, [[x[-1], y[-1]], [0.0, y[-1]], [0.0, 0.0]]])
        rings.append(p + [0.0, 0.0])
    n = [len(r) for r in rings]
    hs = gsj.HostSet(np.arange(4, dtype=np.uint64), np.concatenate([[0], np.cumsum(n)]).astype(np.uint64), np.concatenate(rings))
    d, o = _check_prep(ctx, hs)
    assert np.array_equal(d["blen"], o["blen"])


# around the 128 vertices a lane takes, the 64 edges of a chunk and of a wave's round
@pytest.mark.parametrize("m", [4, 63, 64, 65, 66, 127, 128, 129, 130, 193, 2500])
@pytest.mark.parametrize("n", [1, 5])
def test_one_size(ctx, n, m):
    _check_prep(ctx, _rings([m] * n, m))


# one to a wave, several, 64; a few large ones among small ones
@pytest.mark.parametrize("n", [4095, 8191, 8193, 20000])
def test_mixed_sizes(ctx, n):
    sizes = np.random.default_rng(n).integers(4, 12, n)
    sizes[:: n // 7] = [500, 129, 70, 300, 64, 65, 1000, 128][: len(sizes[:: n // 7])]
    _check_prep(ctx, _rings(sizes, n))


@pytest.mark.parametrize("maxv", [8, 64])
@pytest.mark.parametrize("m", [9, 10, 17, 130, 2500])
def test_subdivided(ctx, m, maxv):
    hs = _rings([m, m + 1, m + 7, 5], m)
    a, b = gsj.subdivide(hs, maxv, ctx), gsj.subdivide(hs, maxv)
    for k in ("gro", "rvo", "xy", "parent", "syn"):
        assert np.array_equal(getattr(a, k), getattr(b, k)), k
    _check_prep(ctx, a)


# sorts of 1024-element tiles up to 64k elements, of 4096 beyond
@pytest.mark.parametrize("n", [2, 1023, 1025, 65536, 65537])
def test_dedup_sizes(ctx, n):
    x = np.random.default_rng(n).integers(0, max(n // 2, 2), n).astype(np.float64)[:, None]
    xy = np.stack([x + [0, 1, 1, 0, 0], x * 0 + [0, 0, 1, 1, 0]], 2).reshape(-1, 2) * 1e-4
    hs = gsj.HostSet(np.arange(n + 1, dtype=np.uint64), 5 * np.arange(n + 1, dtype=np.uint64), xy)
    a, b = gsj.dedup(hs, ctx), gsj.dedup(hs)
    assert np.array_equal(a[0].xy, b[0].xy) and np.array_equal(a[1], b[1]) and np.array_equal(a[2], b[2])
