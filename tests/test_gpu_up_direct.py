"""Upward adjacency written straight into the caller's arrays, from down maps
whose lows lie close together, far apart, and both in a wave; and where an output
array is the down map itself."""
import numpy as np
import pytest

from test_gpu_kernels import dev, lib  # noqa: F401  (fixtures)

pytestmark = pytest.mark.gpu

DEG = {(1, 0): 2, (2, 1): 3, (3, 0): 4, (3, 2): 4}


def lows_like(kind, n, nlows, rng):
    near = np.minimum(np.arange(n) // 5, nlows - 1)
    far = rng.integers(0, nlows, n)
    if kind == "near":
        return near
    if kind == "far":
        return far
    if kind == "one":
        return np.zeros(n, np.int64)
    # both in a wave
    lane = np.arange(n) % 64
    return np.where((lane < 8) if kind == "far, near" else (lane >= 24), far, near)


@pytest.mark.parametrize("kind", ["near", "far", "one", "far, near", "near, far"])
@pytest.mark.parametrize("hd,ld,nhighs,nlows", [(3, 0, 1, 4), (2, 1, 85, 60), (1, 0, 4097, 300), (3, 2, 3001, 9000)])
@pytest.mark.parametrize("into", ["apart", "the map"])
def test_up_from_down_into(lib, dev, kind, hd, ld, nhighs, nlows, into):  # noqa: F811
    deg = DEG[hd, ld]
    rng = np.random.default_rng([hd, ld])
    lows = lows_like(kind, nhighs * deg, nlows, rng).astype(np.uint32)
    p = dev.put(lows)
    po, pd = dev.empty(nlows + 1, np.uint32), dev.empty(len(lows), np.uint32)
    pa = p if into == "the map" else dev.empty(len(lows), np.uint32)
    assert lib.ohx_up_from_down(hd, ld, nhighs, nlows, p, po, pa, pd, None) == 0
    order = np.argsort(lows, kind="stable")
    want = np.concatenate([[0], np.cumsum(np.bincount(lows, minlength=nlows))]).astype(np.uint32)
    assert np.array_equal(dev.get(po, nlows + 1, np.uint32), want)
    assert np.array_equal(dev.get(pa, len(lows), np.uint32), (order // deg).astype(np.uint32))
    assert np.array_equal(dev.get(pd, len(lows), np.uint32), (order % deg).astype(np.uint32))
