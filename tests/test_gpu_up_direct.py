"""Upward adjacency written straight into the caller's arrays, from down maps
whose lows lie close together, far apart, and both in a wave; where an output
array is the down map itself, or is host memory, which the runtime copies to;
and no output array at all, which is refused."""
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


def small():
    lows = np.array([[0, 1, 2, 3], [1, 2, 3, 4]], dtype=np.uint32)
    order = np.argsort(lows.ravel(), kind="stable")
    offs = np.concatenate([[0], np.cumsum(np.bincount(lows.ravel(), minlength=5))])
    return lows, [a.astype(np.uint32) for a in (offs, order // 4, order % 4)]


@pytest.mark.parametrize("on_host", [(0,), (1,), (2,), (0, 1, 2)])
def test_up_from_down_into_host_memory(lib, dev, on_host):  # noqa: F811
    lows, want = small()
    p = dev.put(lows)
    host = [np.zeros(len(w), np.uint32) for w in want]
    out = [host[k].ctypes.data if k in on_host else dev.empty(len(want[k]), np.uint32) for k in range(3)]
    assert lib.ohx_up_from_down(3, 0, 2, 5, p, *out, None) == 0
    for k in range(3):
        got = host[k] if k in on_host else dev.get(out[k], len(want[k]), np.uint32)
        assert np.array_equal(got, want[k])


@pytest.mark.parametrize("missing", [0, 1, 2])
def test_up_from_down_without_an_output_array(lib, dev, missing):  # noqa: F811
    lows, want = small()
    p = dev.put(lows)
    out = [None if k == missing else dev.empty(len(want[k]), np.uint32) for k in range(3)]
    assert lib.ohx_up_from_down(3, 0, 2, 5, p, *out, None) == 0xFFFFFFFF
    assert lib.ohx_last_error()
    # no uses: only the offsets are written
    if missing:
        assert lib.ohx_up_from_down(3, 0, 0, 5, p, out[0], None, None, None) == 0
        assert not dev.get(out[0], 6, np.uint32).any()
