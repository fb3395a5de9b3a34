"""Product uses take their places with one atomic per distinct low of a wave:
split and collapse passes whose products end inside a wave, fill many, or
repeat one low through whole waves leave maps equal to a fresh derivation."""
import numpy as np
import pytest

import meshlib as ML
import parity_cases as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,n", [(2, 1), (2, 9), (2, 40), (3, 1), (3, 3), (3, 9)])
@pytest.mark.parametrize("fine", [1, 0.3])
def test_patched_maps(dim, n, fine):
    got = []
    for which in ("product", "oracle"):
        lib = ML.load(which)
        assert lib, "build first"
        x, c = ML.box(dim, n)
        m = ML.Mesh(lib, dim, x, c)
        m.derive_model_full()
        # one fine corner: a few products; or fine throughout
        m.add_field(0, "adapt_size", np.where(x[:, 0] <= (0 if fine == 1 else 1), 0.4, 3.0) / n)
        m.last = m.adapt(max_ops=12)
        got.append(m)
    a, b = got
    assert a.last == b.last
    assert P.diff_states(a, b) is None
    fresh = a.clone()
    for low, high in ((0, 1), (0, dim), (1, dim)):
        for p, q in zip(a.up(low, high), fresh.up(low, high)):
            assert np.array_equal(p, q), (low, high)
