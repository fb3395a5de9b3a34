"""The qualities of candidate splits, listed per block of edges and measured
by groups of lanes: one split pass with scattered candidates equals the
oracle's, from a single element to meshes whose blocks take 32 and 64 edges,
none of them a multiple of it."""
import numpy as np
import pytest

import meshlib as ML
import parity_cases as P

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("share", [0.02, 0.5, 1.0])
@pytest.mark.parametrize("dim,n", [(2, 1), (2, 7), (2, 150), (2, 211), (3, 1), (3, 4), (3, 22), (3, 27)])
def test_scattered_splits(dim, n, share):
    got = []
    for which in ("product", "oracle"):
        lib = ML.load(which)
        assert lib, "build first"
        x, c = ML.box(dim, n)
        rng = np.random.default_rng([dim, n])
        step = (rng.random(x.shape) - 0.5) * (0.16 / n) * ((x[:, :dim] > 0) & (x[:, :dim] < 1)).all(1)[:, None]
        step[:, dim:] = 0
        m = ML.Mesh(lib, dim, x + step, c)
        m.derive_model_full()
        m.add_field(0, "adapt_size", np.where(rng.random(len(x)) < share, 0.5, 4.0) / n)
        m.last = m.refine_by_size(0.3)
        got.append(m)
    assert got[0].last == got[1].last
    assert P.diff_states(*got) is None
