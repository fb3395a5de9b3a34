"""The independent set over a mesh's edges, whose neighbours are read from
the elements around each edge, against the oracle's, which reads the edge
star: the smallest boxes, odd sizes, and goodness with and without ties."""
import ctypes as C

import numpy as np
import pytest

import meshlib as ML

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n", [(2, 1), (2, 7), (2, 33), (3, 1), (3, 2), (3, 7)])
@pytest.mark.parametrize("levels", [1, 5, None])
@pytest.mark.parametrize("star", [False, True])
def test_edge_indset_through_elements(dim, n, levels, star):
    libs = [ML.load("product"), ML.load("oracle")]
    assert all(libs), "build first"
    # goodness of one level is one chain of ties over the whole mesh
    libs[0].dll.ohx_set_indset_max_rounds.argtypes = [C.c_uint]
    libs[1].dll.orc_set_indset_max_rounds.argtypes = [C.c_uint]
    libs[0].dll.ohx_set_indset_max_rounds(100000)
    libs[1].dll.orc_set_indset_max_rounds(100000)
    try:
        x, c = ML.box(dim, n)
        got = []
        for lib in libs:
            m = ML.Mesh(lib, dim, x, c)
            m.derive_model_full()
            if star:
                m.star(1, dim)
            rng = np.random.default_rng(n)
            ne = m.count(1)
            good = rng.random(ne) if levels is None else rng.integers(0, levels, ne).astype(float)
            got.append(m.find_indset(1, rng.random(ne) < 0.7, good))
        assert np.array_equal(got[0], got[1])
    finally:
        libs[0].dll.ohx_set_indset_max_rounds(0)
        libs[1].dll.orc_set_indset_max_rounds(0)


def test_edge_indset_reads_a_star_that_is_there():
    """The star holds each neighbour once, the elements once for each element
    they share: where the star is there already its rounds are the shorter."""
    lib = ML.load("product")
    d = lib.dll
    d.ohx_profile_get.argtypes = [C.c_char_p] + 3 * [C.c_void_p]
    m = ML.Mesh.box_on_device(lib, 3, 30)
    m.derive_model_full()
    rng = np.random.default_rng(7)
    cand, good = rng.random(m.count(1)) < 0.6, rng.random(m.count(1))

    def rounds():
        best = 1e9
        for _ in range(8):
            d.ohx_profile_enable(1)
            try:
                d.ohx_profile_reset()
                state = m.find_indset(1, cand, good)
                ms = C.c_double()
                d.ohx_profile_get(b"indset_round", C.byref(ms), C.byref(C.c_ulonglong()), C.byref(C.c_double()))
            finally:
                d.ohx_profile_enable(0)
            best = min(best, ms.value)
        return best, state

    through_elements, a = rounds()
    m.star(1, 3)
    through_star, b = rounds()
    assert np.array_equal(a, b)
    assert through_star < 0.9 * through_elements
