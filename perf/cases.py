"""What the time of this library is measured on.

Every case is a call, or the few calls in a row, that a program using the
library makes: one mesh_adapt of a mesh it holds (2D and 3D, isotropic and
anisotropic, FP64 and FP32-mixed, with solution fields, several meshes at
once), one step of a moving-mesh loop, deriving a mesh's topology from vertices and elements, and two of the
kernel entry points over device arrays.

Meshes are Kuhn boxes whose interior vertices are moved at random, so that,
as in a solver's mesh, no two elements are alike.  A state holds the mesh the
program has before the call, and the arrays, with room to spare, in which it
wants the result; a pass adapts a copy of the mesh (mesh_adapt changes it),
copies the whole adapted mesh into those arrays and lets it go.
"""
import ctypes as C
import math

import numpy as np
import torch

from omega_h_v1_amd import seam as S
from omega_h_v1_amd import workloads as W

SIZE_FLOOR, GOOD_QUALITY, LAYERS = 1.0 / 3.0, 0.3, 4  # the adapt parameters of the reference's public call
INDSET_ROUNDS = 2000  # a limit, not a work amount: fields that are constant along a front make long chains of ties
POINTWISE, CONSERVE = 1, 2

_LIB = None


def lib():
    global _LIB
    if _LIB is None:
        torch.cuda.init()
        _LIB = S.product()
        d = _LIB.dll
        d.osh_init(None, None)
        for f in ("osh_down", "osh_up", "osh_up_offs", "osh_up_dirs", "osh_star", "osh_star_offs"):
            getattr(d, f).restype = C.c_void_p
            getattr(d, f).argtypes = [C.c_void_p, C.c_uint, C.c_uint]
        for f in ("osh_get_field", "osh_get_label"):
            getattr(d, f).restype = C.c_void_p
            getattr(d, f).argtypes = [C.c_void_p, C.c_uint, C.c_char_p]
        d.osh_new_field.restype = C.c_void_p
        d.osh_new_field.argtypes = [C.c_void_p, C.c_uint, C.c_char_p, C.c_uint, C.c_int]
        d.osh_components.argtypes = [C.c_void_p, C.c_uint, C.c_char_p]
        d.ohx_set_precision.argtypes = [C.c_int]
        d.ohx_set_indset_max_rounds.argtypes = [C.c_uint]
        d.ohx_last_error.restype = C.c_char_p
        d.ohx_element_qualities_f64.argtypes = [C.c_uint, C.c_uint] + 4 * [C.c_void_p]
        d.ohx_min_quality_f64.argtypes = [C.c_uint, C.c_uint] + 3 * [C.c_void_p]
        d.ohx_min_quality_f64.restype = C.c_double
        d.ohx_measure_edges_f64.argtypes = [C.c_uint] + 5 * [C.c_void_p]
        d.ohx_up_from_down.argtypes = 4 * [C.c_uint] + 5 * [C.c_void_p]
        d.ohx_set_indset_max_rounds(INDSET_ROUNDS)
    return _LIB


class _View:
    """A device array of a mesh for torch.as_tensor; keeps the mesh alive."""

    def __init__(self, mesh, ptr, shape, kind):
        self.mesh = mesh
        self.__cuda_array_interface__ = {"data": (ptr or 0, False), "shape": shape, "typestr": kind, "version": 2}


def view(mesh, ptr, shape, kind):
    if 0 in shape or not ptr:
        return torch.empty(shape, dtype=torch.float64 if kind == "<f8" else torch.int32, device="cuda")
    return torch.as_tensor(_View(mesh, ptr, shape, kind), device="cuda")


def real_tag(m, d, name):
    dll = lib().dll
    nc = dll.osh_components(m.h, d, name.encode())
    return view(m, dll.osh_get_field(m.h, d, name.encode()), (m.count(d), nc), "<f8")


def new_field(m, d, name, ncomps, transfer, values):
    """osh_new_field, filled on the device."""
    ptr = lib().dll.osh_new_field(m.h, d, name.encode(), ncomps, transfer)
    view(m, ptr, (m.count(d), ncomps), "<f8").copy_(values.reshape(-1, ncomps))
    torch.cuda.synchronize()


def int_tag(m, d, name):
    return view(m, lib().dll.osh_get_label(m.h, d, name.encode()), (m.count(d),), "<i4")


def down(m, h, l):
    return view(m, lib().dll.osh_down(m.h, h, l), (m.count(h), math.comb(h + 1, l + 1)), "<i4")


def arrays(m, fields=()):
    """The whole mesh: connectivity and classification of every dimension,
    the coordinates, and the named (dimension, field) pairs."""
    out = {"x": real_tag(m, 0, "coordinates")}
    for d in range(m.dim + 1):
        if d:
            out["down%d" % d] = down(m, d, 0)
        out["class_dim%d" % d] = int_tag(m, d, "class_dim")
        out["class_id%d" % d] = int_tag(m, d, "class_id")
    for d, name in fields:
        out["%s%d" % (name, d)] = real_tag(m, d, name)
    return out


def room(dim, elements, fields=()):
    """Arrays for a mesh of up to so many elements; fields: (dimension, name,
    components)."""
    e = int(elements) + 200
    n = [0.6 * e, 1.7 * e, e] if dim == 2 else [0.4 * e, 1.6 * e, 2.3 * e, e]
    n = [int(v) for v in n]
    out = {"x": torch.zeros(n[0], 3, dtype=torch.float64, device="cuda")}
    for d in range(dim + 1):
        if d:
            out["down%d" % d] = torch.zeros(n[d], d + 1, dtype=torch.int32, device="cuda")
        out["class_dim%d" % d] = torch.zeros(n[d], dtype=torch.int32, device="cuda")
        out["class_id%d" % d] = torch.zeros(n[d], dtype=torch.int32, device="cuda")
    for d, name, nc in fields:
        out["%s%d" % (name, d)] = torch.zeros(n[d], nc, dtype=torch.float64, device="cuda")
    return out


def take(meshes, into, fields):
    """The meshes' arrays, one mesh after the other, copied into the
    program's own; how many entities of every dimension there are."""
    at = dict.fromkeys(into, 0)
    to, of = [], []
    for m in meshes:
        for k, v in arrays(m, fields).items():
            n = at[k] + len(v)
            if n > len(into[k]):
                raise RuntimeError("the adapted mesh has %d %s, more than there is room for" % (n, k))
            to.append(into[k][at[k]:n])
            of.append(v)
            at[k] = n
    for kind in (torch.float64, torch.int32):
        same = [i for i, v in enumerate(of) if v.dtype == kind]
        torch._foreach_copy_([to[i] for i in same], [of[i] for i in same])
    out = dict(into)
    out["counts"] = np.array([at["class_dim%d" % d] for d in range(meshes[0].dim + 1)])
    torch.cuda.current_stream().synchronize()  # the meshes may go now
    return out


# ---------------------------------------------------------------- meshes
def counts(dim, n):
    """Entities of the Kuhn box of n cubes (squares) a side, by dimension."""
    if dim == 2:
        return [(n + 1) ** 2, 3 * n * n + 2 * n, 2 * n * n]
    v, t = (n + 1) ** 3, 6 * n ** 3
    f = (4 * t + 12 * n * n) // 2  # every face twice but those of the surface
    return [v, v + f - t - 1, f, t]


def mesh_bytes(dim, n):
    """One copy of a mesh: coordinates, one size, and for every dimension
    the vertices and the classification of each entity."""
    c = counts(dim, n)
    return 32 * c[0] + sum(8 * c[d] + (4 * (d + 1) * c[d] if d else 0) for d in range(dim + 1))


def moved(dim, n, x, rng):
    """Interior vertices of the box moved by up to 0.08 of the spacing."""
    inner = ((x[:, :dim] > 0) & (x[:, :dim] < 1)).all(1)
    step = (rng.random((len(x), 3)) - 0.5) * (0.16 / n)
    step[:, dim:] = 0
    return x + step * inner[:, None]


def box(dim, n, rng):
    """A classified, full box mesh on the GPU."""
    m = S.Mesh.box_on_device(lib(), dim, n)
    x = m.coords().reshape(-1, 3)
    real_tag(m, 0, "coordinates").copy_(torch.from_numpy(moved(dim, n, x, rng)))
    torch.cuda.synchronize()
    m.derive_model_full()
    return m


def warped(dim, n, h, warp, rng):
    """A box of uniform desired size h with a displacement field "warp"."""
    m = box(dim, n, rng)
    m.add_field(0, "adapt_size", W.uniform_size(m.count(0), h))
    x = m.coords().reshape(-1, 3)
    amount = rng.uniform(0.9, 1.1)
    if warp == "sine":
        w = W.sine_warp_2d(x, 0.1 * amount)
    else:
        w = W.rotation_warp(x, amount * math.pi / 4)
    m.add_field(0, "warp", w.ravel())
    return m


def front(n, steep, rng, eps=0.01, hmin=0.128, hmax=6.4):
    """A 3D box with the metric of a steep front's Hessian, the same shape
    of metric relative to the spacing at every n."""
    m = box(3, n, rng)
    x = m.coords().reshape(-1, 3)
    m.add_field(0, "hessian", W.tanh_front_hessian(x, a=steep * n, s0=rng.uniform(1.4, 1.6), dim=3).ravel())
    m.metric_from_hessian("hessian", eps, hmin / n, hmax / n)
    m.free_field(0, "hessian")
    return m


def add_solution(m):
    """Element fields that follow the mesh: two conserved, and in 3D two
    pointwise ones."""
    d = m.dim
    x = real_tag(m, 0, "coordinates")
    c = x[down(m, d, 0).long()].mean(1)
    new_field(m, d, "mass", 1, CONSERVE, 1.0 + c[:, 0] + 0.5 * c[:, 1] ** 2)
    new_field(m, d, "momentum", 3, CONSERVE, torch.stack([c[:, 1], -c[:, 0], 0.25 + 0 * c[:, 2]], 1))
    if d == 3:
        new_field(m, d, "velocity", 3, POINTWISE,
                  torch.stack([1 + 2 * c[:, 0] - c[:, 2], 0.5 * c[:, 1], 3 - c[:, 0] + c[:, 1]], 1))
        new_field(m, d, "temperature", 1, POINTWISE, torch.sin(3 * c[:, 0]) * torch.cos(2 * c[:, 2]))


def dye(x, dim):
    """A cone of height 1 at the left of the box, a negative one at the right."""
    z = 0.5 if dim == 3 else 0.0
    left = np.sqrt(((x - [0.25, 0.5, z]) ** 2).sum(1))
    right = np.sqrt(((x - [0.75, 0.5, z]) ** 2).sum(1))
    return np.where(left <= 0.25, 4 * (0.25 - left), np.where(right <= 0.25, -4 * (0.25 - right), 0.0))


def set_size_field(m, weight, min_h, max_h):
    """The size from the recovered Hessian of the dye, on the GPU."""
    d = m.dim
    m.free_field(0, "adapt_size")
    m.element_gradients("dye")
    m.recover_by_volume("grad_dye")
    m.free_field(d, "grad_dye")
    m.element_gradients("grad_dye")
    m.free_field(0, "grad_dye")
    m.recover_by_volume("grad_grad_dye")
    m.free_field(d, "grad_grad_dye")
    m.size_from_hessian("grad_grad_dye", [weight], min_h, max_h)
    m.free_field(0, "grad_grad_dye")


# ----------------------------------------------------------------- cases
def listed():
    return [
        # the smallest call: a coarse 2D mesh of a moving-domain run, where
        # every pass is a few launches and a decision on the host
        {"name": "adapt2d_512", "kind": "warp", "dim": 2, "n": 16, "h": 1.33, "warp": "sine"},
        # a moving-domain run's ordinary 2D mesh (131,072 triangles)
        {"name": "adapt2d_131k", "kind": "warp", "dim": 2, "n": 256, "h": 1.28, "warp": "sine"},
        # a small 3D mesh (3,072 tets) refined towards a uniform size
        {"name": "adapt3d_3k", "kind": "uniform", "dim": 3, "n": 8, "h": 0.4},
        # an ordinary 3D mesh of odd size in a boundary-layer-like metric, FP64
        {"name": "aniso3d_55k", "kind": "front", "n": 21, "steep": 0.78, "mixed": False},
        # a large 3D mesh (511,104 tets) in that metric, FP32-mixed
        {"name": "aniso3d_511k", "kind": "front", "n": 44, "steep": 0.78, "mixed": True},
        # a large mesh refined to a smaller size: 384,000 tets become about
        # 1.8 million, and memory bandwidth decides
        {"name": "adapt3d_384k", "kind": "uniform", "dim": 3, "n": 40, "h": 1.2},
        # solution transfer: an adapt that carries conserved and pointwise
        # element fields
        {"name": "transfer3d_10k", "kind": "transfer", "dim": 3, "n": 12, "h": 0.6},
        # one step of a moving-mesh loop: move, recover a size field from the
        # solution, adapt
        {"name": "step2d_20k", "kind": "step", "dim": 2, "n": 101},
        # from vertices and elements in host memory to a classified mesh with
        # the adjacencies a solver asks for
        {"name": "setup3d_664k", "kind": "setup", "dim": 3, "n": 48},
        # the kernel entry points on device arrays: qualities and edge
        # lengths, and the upward adjacency
        {"name": "quality3d_2m", "kind": "quality", "dim": 3, "n": 71},
        {"name": "up_from_down_vert_tet", "kind": "up", "high": 3, "low": 0, "n": 53, "ordered": False},
        # uneven meshes, each in a metric of its own, adapted at once on
        # several streams
        {"name": "many3d_16", "kind": "many", "count": 16, "hi": 20, "ratio": 20.0, "threads": 8},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["warp", "warp", "uniform", "uniform", "front", "front", "transfer", "step", "setup", "quality",
                       "up", "many"])
    # n / h spacings of the desired size fit across the box: the adapted mesh
    # has no more than about two million elements
    if kind == "warp":
        dim = rng.choice([2, 2, 3])
        n = _log(rng, 8, 256) if dim == 2 else _log(rng, 4, 20)
        return {"kind": kind, "dim": dim, "n": n, "h": round(rng.uniform(0.8, 1.4), 3),
                "warp": rng.choice(["sine", "rot"]) if dim == 2 else "rot"}
    if kind == "uniform":
        dim = rng.choice([2, 3])
        n = _log(rng, 16, 300) if dim == 2 else _log(rng, 4, 40)
        least = max(0.4, n / (320 if dim == 2 else 33))
        return {"kind": kind, "dim": dim, "n": n, "h": round(rng.uniform(least, least + 1.5), 3)}
    if kind == "front":
        return {"kind": kind, "n": _log(rng, 8, 42), "steep": round(rng.uniform(0.5, 0.9), 3), "mixed": rng.random() < 0.5}
    if kind == "transfer":
        dim = rng.choice([2, 3])
        n = _log(rng, 8, 100) if dim == 2 else _log(rng, 4, 16)
        return {"kind": kind, "dim": dim, "n": n, "h": round(rng.uniform(0.6, 1.6), 3)}
    if kind == "step":
        dim = rng.choice([2, 2, 3])
        return {"kind": kind, "dim": dim, "n": _log(rng, 24, 256) if dim == 2 else _log(rng, 6, 24)}
    if kind == "setup":
        dim = rng.choice([2, 3])
        return {"kind": kind, "dim": dim, "n": _log(rng, 8, 500) if dim == 2 else _log(rng, 4, 48)}
    if kind == "quality":
        dim = rng.choice([2, 3])
        return {"kind": kind, "dim": dim, "n": _log(rng, 8, 900) if dim == 2 else _log(rng, 4, 71)}
    if kind == "up":
        high, low = rng.choice([(1, 0), (2, 0), (2, 1), (3, 0), (3, 1), (3, 2)])
        return {"kind": kind, "high": high, "low": low, "n": _log(rng, 4, 53), "ordered": rng.random() < 0.3}
    return {"kind": kind, "count": rng.randint(3, 16), "hi": rng.randint(10, 20), "ratio": round(rng.uniform(4, 20), 2),
            "threads": rng.choice([2, 4, 8])}


def growth(case):
    """About how many elements an adapted mesh has for each one before."""
    if case["kind"] == "front":
        return 165.0 / case["n"]  # a front is a surface
    if case["kind"] == "many":
        return 14.0  # of the desired size in the mean, and anisotropic
    # an element of the desired size is smaller than the box's, whose edges
    # are 1 to sqrt(dim) spacings long
    return (3.1 if case["dim"] == 2 else 8.3) * case.get("h", 1.2) ** -case["dim"]


def many_sizes(case):
    """Cubes a side of the meshes: spread over their logarithm."""
    lo, hi = math.log(8), math.log(case["hi"])
    return [int(round(math.exp(lo + (hi - lo) * (k + 0.5) / case["count"]))) for k in range(case["count"])]


# --------------------------------------------------------------- prepare
def fields_of(case, dim):
    """The fields (dimension, name, components) of the adapted mesh."""
    kind = case["kind"]
    if kind in ("front", "many"):
        return [(0, "metric", 6)]
    if kind == "warp":
        return [(0, "adapt_size", 1), (0, "warp", 3)]
    if kind == "step":
        return [(0, "adapt_size", 1), (0, "warp", 3), (0, "dye", 1)]
    if kind == "transfer":
        more = [(3, "velocity", 3), (3, "temperature", 1)] if dim == 3 else []
        return [(0, "adapt_size", 1), (dim, "mass", 1), (dim, "momentum", 3)] + more
    return [(0, "adapt_size", 1)]


def prepare(case, seed):
    lib()
    rng = np.random.default_rng([seed, 77])
    kind = case["kind"]
    if kind in ("setup", "quality", "up"):
        return prepare_kernels(case, rng)
    if kind == "many":
        meshes = many(case, rng)
    else:
        meshes = [one(case, rng)]
    m = meshes[0]
    fields = fields_of(case, m.dim)
    elements = sum(m.count(m.dim) for m in meshes)
    s = {"case": case, "meshes": meshes, "fields": [f[:2] for f in fields],
         "room": room(m.dim, elements * 2 * max(1.0, growth(case)), fields)}
    torch.cuda.synchronize()
    return s


def one(case, rng):
    kind = case["kind"]
    if kind == "warp":
        return warped(case["dim"], case["n"], case["h"] / case["n"], case["warp"], rng)
    if kind in ("uniform", "transfer"):
        m = box(case["dim"], case["n"], rng)
        # a desired size that varies by a fifth over the domain
        x = m.coords().reshape(-1, 3)
        p = rng.uniform(0, 2 * math.pi)
        h = case["h"] / case["n"] * (1 + 0.2 * np.sin(5 * x[:, 0] + 3 * x[:, 1] + 2 * x[:, 2] + p))
        m.add_field(0, "adapt_size", h)
        if kind == "transfer":
            add_solution(m)
        return m
    if kind == "front":
        return front(case["n"], case["steep"], rng)
    dim, n = case["dim"], case["n"]
    m = warped(dim, n, 1.0 / n, "rot", rng)
    m.add_field(0, "dye", dye(m.coords().reshape(-1, 3), dim) * rng.uniform(0.9, 1.1))
    return m


def many(case, rng):
    """Boxes of different sizes, each in a constant metric of its own whose
    mean length is the mesh's spacing."""
    meshes = []
    for n in many_sizes(case):
        rot = W.random_rotation(rng)
        lengths = np.exp(rng.uniform(math.log(0.1 / case["ratio"]), math.log(0.1), size=3))
        m = box(3, n, rng)
        real_tag(m, 0, "coordinates").mul_(n * float(np.prod(lengths)) ** (1.0 / 3.0))
        torch.cuda.synchronize()
        m.add_field(0, "metric", W.constant_metric(m.count(0), rot, lengths).ravel())
        meshes.append(m)
    return meshes


def prepare_kernels(case, rng):
    kind = case["kind"]
    if kind == "setup":
        x, c = S.box(case["dim"], case["n"])
        return {"case": case, "x": moved(case["dim"], case["n"], x, rng), "elements": c}
    if kind == "quality":
        m = box(case["dim"], case["n"], rng)
        s = {"case": case, "x": real_tag(m, 0, "coordinates").clone(), "edges": down(m, 1, 0).clone(),
             "elems": down(m, m.dim, 0).clone(),
             "h": torch.from_numpy(rng.uniform(0.8, 1.2, m.count(0)) / case["n"]).cuda()}
        s["q"] = torch.empty(len(s["elems"]), dtype=torch.float64, device="cuda")
        s["len"] = torch.empty(len(s["edges"]), dtype=torch.float64, device="cuda")
        torch.cuda.synchronize()
        return s
    dim = max(2, case["high"])
    m = box(dim, case["n"], rng)
    lows = down(m, case["high"], case["low"]).clone()
    if not case["ordered"]:
        # entities in an arbitrary order, as meshes come from generators
        lows = lows[torch.from_numpy(rng.permutation(len(lows))).cuda()]
    nl = m.count(case["low"])
    s = {"case": case, "lows": lows, "nl": nl}
    uses = s["lows"].numel()
    s["offsets"] = torch.empty(nl + 1, dtype=torch.int32, device="cuda")
    s["highs"] = torch.empty(uses, dtype=torch.int32, device="cuda")
    s["dirs"] = torch.empty(uses, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    return s


# ------------------------------------------------------------------- run
def run(state):
    dll = lib().dll
    case = state["case"]
    kind = case["kind"]
    if kind == "setup":
        return run_setup(dll, state)
    if kind in ("quality", "up"):
        return run_kernels(dll, state)
    dll.ohx_set_precision(1 if case.get("mixed") else 0)
    meshes = [m.clone() for m in state["meshes"]]
    m = meshes[0]
    done = None
    if kind == "many":
        _, changed, _ = S.Mesh.adapt_many(lib(), meshes, SIZE_FLOOR, GOOD_QUALITY, LAYERS, 50, case["threads"])
    elif kind == "front":
        changed = m.adapt(SIZE_FLOOR, GOOD_QUALITY, LAYERS, 1000)
    elif kind == "warp":
        done = m.warp_to_limit(0.2)
        changed = m.adapt(SIZE_FLOOR, GOOD_QUALITY, LAYERS, 50)
    elif kind == "step":
        n = case["n"]
        done = m.warp_to_limit(0.1)
        set_size_field(m, 0.075 / n ** 2, 0.4 / n, 1.2 / n)
        changed = m.adapt(SIZE_FLOOR, 0.4, 0, 50)
    else:
        changed = m.adapt(SIZE_FLOOR, GOOD_QUALITY, LAYERS, 50)
    out = take(meshes, state["room"], state["fields"])
    out["changed"] = changed
    if done is not None:
        out["done"] = done
    return out


def run_setup(dll, state):
    m = S.Mesh(lib(), state["case"]["dim"], state["x"], state["elements"])
    m.derive_model_full()
    d = m.dim
    out = arrays(m)
    for h in range(2, d + 1):
        out["down%d%d" % (h, h - 1)] = down(m, h, h - 1)
    for l, h in [(0, 1), (0, d), (1, d)]:
        uses = m.count(h) * math.comb(h + 1, l + 1)
        out["up%d%d" % (l, h)] = view(m, dll.osh_up(m.h, l, h), (uses,), "<i4")
        out["up_offs%d%d" % (l, h)] = view(m, dll.osh_up_offs(m.h, l, h), (m.count(l) + 1,), "<i4")
        out["up_dirs%d%d" % (l, h)] = view(m, dll.osh_up_dirs(m.h, l, h), (uses,), "<i4")
    # vertex neighbours: the other end of every edge of a vertex
    out["star"] = view(m, dll.osh_star(m.h, 0, 1), (2 * m.count(1),), "<i4")
    out["star_offs"] = view(m, dll.osh_star_offs(m.h, 0, 1), (m.count(0) + 1,), "<i4")
    return out


def _ok(r, dll):
    if r == 0xFFFFFFFF or r == -1:
        raise RuntimeError(dll.ohx_last_error())


def run_kernels(dll, s):
    case = s["case"]
    if case["kind"] == "quality":
        d = case["dim"]
        n, ne = len(s["elems"]), len(s["edges"])
        _ok(dll.ohx_element_qualities_f64(d, n, s["elems"].data_ptr(), s["x"].data_ptr(), s["q"].data_ptr(), None), dll)
        low = dll.ohx_min_quality_f64(d, n, s["elems"].data_ptr(), s["x"].data_ptr(), None)
        _ok(dll.ohx_measure_edges_f64(ne, s["edges"].data_ptr(), s["x"].data_ptr(), s["h"].data_ptr(),
                                      s["len"].data_ptr(), None), dll)
        return {"q": s["q"], "len": s["len"], "min": low}
    _ok(dll.ohx_up_from_down(case["high"], case["low"], len(s["lows"]), s["nl"], s["lows"].data_ptr(),
                             s["offsets"].data_ptr(), s["highs"].data_ptr(), s["dirs"].data_ptr(), None), dll)
    return {k: s[k] for k in ("offsets", "highs", "dirs")}


# ---------------------------------------------------------- work and truth
def work(case):
    """A mesh read once and the adapted mesh written once; the adapted
    meshes are about as large as these expressions say."""
    kind = case["kind"]
    if kind == "quality":
        c = counts(case["dim"], case["n"])
        d = case["dim"]
        return {"bytes": c[d] * (4 * (d + 1) + 8) + 16 * c[1] + 32 * c[0],
                "flops": c[d] * (90 if d == 3 else 40) * 2 + 14 * c[1]}
    if kind == "up":
        c = counts(max(2, case["high"]), case["n"])
        uses = c[case["high"]] * math.comb(case["high"] + 1, case["low"] + 1)
        return {"bytes": 4 * (3 * uses + c[case["low"]] + 1), "flops": 0}
    if kind == "setup":
        d, n = case["dim"], case["n"]
        c = counts(d, n)
        maps = sum(4 * (h + 1) * c[h] for h in range(2, d + 1))
        ups = sum(4 * (c[l] + 1) + 8 * c[h] * math.comb(h + 1, l + 1) for l, h in [(0, 1), (0, d), (1, d)])
        return {"bytes": 24 * c[0] + 4 * (d + 1) * c[d] + mesh_bytes(d, n) + maps + ups + 4 * (c[0] + 1) + 8 * c[1],
                "flops": 0}
    if kind == "many":
        return {"bytes": sum((mesh_bytes(3, n) + 40 * (n + 1) ** 3) * (1 + growth(case)) for n in many_sizes(case)),
                "flops": 0}
    d = case.get("dim", 3)
    one = mesh_bytes(d, case["n"])
    if kind == "front":
        one += 40 * counts(3, case["n"])[0]
    elif kind == "step":
        one += 16 * counts(d, case["n"])[0]
    if kind == "transfer":
        one += (64 if d == 3 else 32) * counts(d, case["n"])[d]
    return {"bytes": one * (1 + growth(case)), "flops": 0}


def tolerance(case):
    """The library's FP64 path promises the reference's results bit for bit,
    and FP32-mixed the FP64 path's, so there is nothing to allow for."""
    return "exact"


def exact(case, seed):
    if case["kind"] == "up":
        s = prepare(case, seed)
        lows = s["lows"].cpu().numpy()
        deg = lows.shape[1]
        order = np.argsort(lows.ravel(), kind="stable")
        offs = np.concatenate([[0], np.cumsum(np.bincount(lows.ravel(), minlength=s["nl"]))])
        return {"offsets": torch.from_numpy(offs.astype(np.int32)),
                "highs": torch.from_numpy((order // deg).astype(np.int32)),
                "dirs": torch.from_numpy((order % deg).astype(np.int32))}
    if case["kind"] != "quality":
        return None  # a sequence of decisions, not a formula
    s = prepare(case, seed)
    x, e, t = s["x"].cpu(), s["edges"].long().cpu(), s["elems"].long().cpu()
    length = (x[e[:, 1]] - x[e[:, 0]]).square().sum(1).sqrt() / ((s["h"].cpu()[e[:, 0]] + s["h"].cpu()[e[:, 1]]) / 2)
    p = x[t]
    if case["dim"] == 3:
        # signed volume over the 3/2 power of the root mean square face area
        u, v, w = p[:, 1] - p[:, 0], p[:, 2] - p[:, 0], p[:, 3] - p[:, 0]
        vol = (torch.linalg.cross(u, v) * w).sum(1) / 6
        area2 = 0
        for f in ((0, 1, 2), (0, 1, 3), (0, 2, 3), (1, 2, 3)):
            a = torch.linalg.cross(p[:, f[1]] - p[:, f[0]], p[:, f[2]] - p[:, f[0]]) / 2
            area2 = area2 + a.square().sum(1)
        q = vol / (area2 / 4).sqrt() ** 1.5
        regular = (math.sqrt(2) / 12) / (math.sqrt(3) / 4) ** 1.5
    else:
        u, v = p[:, 1] - p[:, 0], p[:, 2] - p[:, 0]
        area = (u[:, 0] * v[:, 1] - u[:, 1] * v[:, 0]) / 2
        len2 = sum((p[:, b] - p[:, a]).square().sum(1) for a, b in ((0, 1), (1, 2), (2, 0)))
        q = area / len2
        regular = (math.sqrt(3) / 4) / 3
    q = q / regular
    return {"q": q, "len": length, "min": float(q[1:].min())}
