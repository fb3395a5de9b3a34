"""The collapse-by-size loop carries what is known of its collapse qualities
from pass to pass; the meshes it leaves equal the oracle's, which measures
every direction in every pass: FP64, the FP32 screen and the certified FP32
pass (whose inexact values are carried too), sizes that collapse almost
everything and almost nothing, with and without ties."""
import ctypes as C

import numpy as np
import pytest

import meshlib as ML
import parity_cases as P
from omega_h_v1_amd import workloads as W
from test_gpu_swap_run import front

pytestmark = pytest.mark.gpu

# pinned variants of coarsen_quality_*_mixed: 1 lane certified, 4 lanes
# certified, 2 lanes screened (None: FP64)
MODES = {"fp64": None, "certified1": 33, "certified4": 36, "screen2": 18}


@pytest.fixture(scope="module")
def libs():
    got = [ML.load("product"), ML.load("oracle")]
    assert all(got), "build first"
    d = got[0].dll
    d.ohx_set_precision.argtypes = [C.c_int]
    d.ohx_tuning_force.argtypes = [C.c_char_p, C.c_int]
    d.ohx_set_indset_max_rounds.argtypes = [C.c_uint]
    got[1].dll.orc_set_indset_max_rounds.argtypes = [C.c_uint]
    d.ohx_set_indset_max_rounds(2000)
    got[1].dll.orc_set_indset_max_rounds(2000)
    yield got
    d.ohx_set_indset_max_rounds(0)
    got[1].dll.orc_set_indset_max_rounds(0)


def mesh(lib, dim, n, h, jitter, metric):
    x, c = ML.box(dim, n)
    inner = ((x[:, :dim] > 0) & (x[:, :dim] < 1)).all(1)
    step = (np.random.default_rng(n).random(x.shape) - 0.5) * (jitter / n) * inner[:, None]
    step[:, dim:] = 0
    m = ML.Mesh(lib, dim, x + step, c)
    m.derive_model_full()
    if metric:
        m.add_field(0, "metric", W.rotating_metric(x, h / n, 4.0, dim=dim).ravel())
    else:
        m.add_field(0, "adapt_size", W.uniform_size(len(x), h / n))
    return m


@pytest.mark.parametrize("mode", sorted(MODES))
@pytest.mark.parametrize("dim,n,h,jitter,metric", [
    (2, 3, 9.0, 0.0, False), (2, 17, 4.0, 0.16, False), (2, 16, 2.0, 0.16, True),
    (3, 2, 9.0, 0.0, False), (3, 6, 4.0, 0.0, False), (3, 7, 5.0, 0.16, False), (3, 6, 1.6, 0.16, True),
])
def test_collapse_loop(libs, mode, dim, n, h, jitter, metric):
    d = libs[0].dll
    name = ("coarsen_quality_%dd_mixed" % dim).encode()
    v = MODES[mode]
    try:
        d.ohx_set_precision(0 if v is None else 1)
        d.ohx_tuning_force(name, -1 if v is None else v)
        a, b = (mesh(lib, dim, n, h, jitter, metric) for lib in libs)
        for m in (a, b):
            m.last = m.adapt(max_ops=40)
        assert a.last == b.last
        assert P.diff_states(a, b) is None
    finally:
        d.ohx_set_precision(0)
        d.ohx_tuning_force(name, -1)


PEAK = 8.0e9  # bytes per millisecond


def test_bytes_of_what_is_measured(libs):
    """The bytes counted for the collapse qualities are those of the directions
    a pass measures: passes that know some of them count fewer than
    passes on their own, which measure every one; and neither they nor the
    swap run's kernels read more than the memory can give."""
    d = libs[0].dll
    d.ohx_profile_get.argtypes = [C.c_char_p] + 3 * [C.c_void_p]
    start = front(libs[0], 9, 0.16)
    floor = min(start.min_quality(), 0.3)
    while start.refine_by_size(floor):
        pass
    floor = min(start.min_quality(), 0.3)

    def counted(run, names):
        d.ohx_profile_enable(1)
        d.ohx_profile_reset()
        got = {}
        try:
            run()
            for name in names:
                ms, k, b = C.c_double(), C.c_ulonglong(), C.c_double()
                d.ohx_profile_get(name.encode(), C.byref(ms), C.byref(k), C.byref(b))
                if k.value:
                    got[name] = (k.value, b.value)
                    assert 0 < b.value < PEAK * ms.value, (name, b.value, ms.value)
        finally:
            d.ohx_profile_enable(0)
        return got

    a, b = start.clone(), start.clone()
    passes = 6
    every = counted(lambda: [a.coarsen_by_size(floor, 1 / 3) for _ in range(passes)],
                    ["coarsen_quality_f64"])["coarsen_quality_f64"]
    names = ["coarsen_quality_f64", "swap_quality_f64", "indset_round"]
    known = counted(lambda: b.adapt(max_ops=passes - 2), names)["coarsen_quality_f64"]
    assert P.diff_states(a, b) is None
    assert known[0] == every[0] and known[1] < every[1]
    # the whole of an adaptation, in both modes
    counted(lambda: start.clone().adapt(max_ops=1000), names)
    d.ohx_set_precision(1)
    try:
        counted(lambda: start.clone().adapt(max_ops=1000),
                names + ["coarsen_quality_mixed", "coarsen_quality_certified", "coarsen_quality_force"])
    finally:
        d.ohx_set_precision(0)
