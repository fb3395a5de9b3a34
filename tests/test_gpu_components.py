"""Deriving a model where its components matter: several bodies, holes, single
elements and shuffled elements, against the oracle's search; and the element
dual of a mesh without sides, whose third element on a side is an error."""
import numpy as np
import pytest

import meshlib as ML
import parity_cases as P

pytestmark = pytest.mark.gpu


def parts(dim, x, c, keep):
    c = c[keep(x[c].mean(1))]
    used, i = np.unique(c, return_inverse=True)
    return x[used], i.reshape(c.shape).astype(np.uint32)


def case(name):
    rng = np.random.default_rng(5)
    if name in ("squares", "boxes"):
        dim = 2 if name == "squares" else 3
        x, c = ML.box(dim, 3)
        k = 5
        x = np.vstack([x + [2.0 * i, 0, 0] for i in range(k)])
        c = np.vstack([c + i * (len(x) // k) for i in range(k)])
        return dim, x, c[rng.permutation(len(c))]
    if name == "triangle":
        return 2, np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0.0]]), np.array([[0, 1, 2]])
    if name == "tet":
        return 3, np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0.0], [0, 0, 1]]), np.array([[0, 1, 2, 3]])
    if name == "frame":  # a square with a hole
        return (2,) + parts(2, *ML.box(2, 9), keep=lambda m: np.abs(m[:, :2] - 0.5).max(1) > 1 / 6)
    if name == "tunnel":  # a box with a hole through it, its faces rough
        x, c = parts(3, *ML.box(3, 6), keep=lambda m: np.abs(m[:, :2] - 0.5).max(1) > 1 / 6)
        return 3, x + 0.02 * (rng.random(x.shape) - 0.5), c[rng.permutation(len(c))]
    x, c = ML.box(3, 17)  # one component through many elements in any order
    return 3, x, c[rng.permutation(len(c))]


@pytest.mark.parametrize("name", ["triangle", "tet", "squares", "boxes", "frame", "tunnel", "shuffled"])
def test_derived_model(name):
    dim, x, c = case(name)
    got = []
    for which in ("product", "oracle"):
        lib = ML.load(which)
        assert lib, "build first"
        m = ML.Mesh(lib, dim, x, c.astype(np.uint32))
        m.derive_model_full()
        got.append(m)
    assert P.diff_states(*got) is None
    assert np.array_equal(got[0].dual(), got[1].dual())


def test_three_elements_on_a_side():
    """Three triangles on one edge: not a mesh whose sides can be derived."""
    x = np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0, -1, 0], [1, 1, 0.0]])
    m = ML.Mesh(ML.load("product"), 2, x, np.array([[0, 1, 2], [1, 0, 3], [0, 1, 4]], dtype=np.uint32))
    with pytest.raises(RuntimeError, match="non-manifold"):
        m.derive_model_full()
