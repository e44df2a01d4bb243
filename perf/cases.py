"""The work a program gives this package, as cases that can be timed: which
calls, on which sizes, element types, boundaries and paddings.

A case is a dict of plain values; `listed()` holds fixed ones, `draw(rng)`
makes another of the same kinds and ranges, `prepare(case, seed)` makes what
a program holds before the call (device arrays filled from the seed, the
StencilArrays over them, a batch plan), `run(state)` is one call as a program
writes it, `work(case)` the bytes and operations it cannot do without, and
`exact(case, seed)` its result in 64-bit arithmetic with plain torch.

Kinds of calls:

- ``gather``: ``mapstencil(f, A)``, the reference's basic call (blocking,
  allocates its result).
- ``gauss``: ``mapstencil_(kernelproduct, dest, A)`` with a Gaussian
  ``Kernel(Window(R))`` into a buffer the program keeps (image filtering).
- ``life``: a Game of Life run, ``mapstencil_steps`` over a
  ``SwitchingStencilArray`` of bytes.
- ``heat2d`` / ``heat3d``: explicit diffusion, ``mapstencil_steps`` with
  ``Laplacian`` over VonNeumann(1) in 2-D or 3-D.
- ``batch``: one ``BatchPlan`` over many arrays of uneven sizes, three shapes
  and three reductions.
- ``steps_batch``: many 2-D heat runs with their own step counts in one call.
- ``water``: ``scatterstencil_`` of the downhill rules (a hydrology step).
- ``coupled``: ``mapstencil_`` of two arguments, diffusion with a source term.
"""
import math
import random
import sys
from pathlib import Path

import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "stencils.jl_amd"))
import stencils_hip as sh  # noqa: E402

DTYPES = {"f64": torch.float64, "f32": torch.float32, "bf16": torch.bfloat16,
          "u8": torch.uint8, "i32": torch.int32, "i64": torch.int64}
ASYNC = sh._abi.ASYNC


def listed():
    return [
        # the reference's README benchmark: a 3 x 3 mean of a 1000 x 1000
        # Float64 array, where a call's latency counts as much as its kernel
        {"name": "mean_f64_1000", "kind": "gather", "fold": "mean", "shape": "window1", "dtype": "f64",
         "n0": 1000, "n1": 1000, "boundary": "remove", "padding": "cond"},
        # the same call on a large raster whose rows are an odd number of cells
        {"name": "mean_f64_8191x8005", "kind": "gather", "fold": "mean", "shape": "window1", "dtype": "f64",
         "n0": 8191, "n1": 8005, "boundary": "remove", "padding": "cond"},
        # a dilation of a byte raster (an element type outside the build-time kernels)
        {"name": "max_u8_8192", "kind": "gather", "fold": "maximum", "shape": "moore2", "dtype": "u8",
         "n0": 8192, "n1": 8192, "boundary": "wrap", "padding": "cond"},
        # 7 x 7 Gaussian filters over padded arrays, in both storage types
        {"name": "gauss_f32_4096", "kind": "gauss", "radius": 3, "dtype": "f32", "n0": 4096, "n1": 4096,
         "boundary": "reflect", "padding": "halo"},
        {"name": "gauss_bf16_16384", "kind": "gauss", "radius": 3, "dtype": "bf16", "n0": 16384, "n1": 16384,
         "boundary": "reflect", "padding": "halo"},
        # the benchmark's Game of Life: a thousand generations on a large torus
        {"name": "life_8192_1000", "kind": "life", "n0": 8192, "n1": 8192, "steps": 1000, "rule": "conway",
         "boundary": "wrap", "padding": "halo"},
        # a mid-size run on a grid whose rows are no multiple of a vector
        {"name": "life_1501x1333_200", "kind": "life", "n0": 1501, "n1": 1333, "steps": 200, "rule": "conway",
         "boundary": "remove", "padding": "cond"},
        # diffusion runs: a 2-D field and a 3-D block
        {"name": "heat2d_f32_4096_100", "kind": "heat2d", "dtype": "f32", "n0": 4096, "n1": 4096, "steps": 100,
         "boundary": "wrap", "padding": "cond"},
        {"name": "heat3d_f32_256_100", "kind": "heat3d", "dtype": "f32", "n0": 256, "n1": 256, "n2": 256,
         "steps": 100, "boundary": "wrap", "padding": "cond"},
        # many small and mid-size arrays in one call, as the uneven batch of the benchmark
        {"name": "batch_f32_60", "kind": "batch", "dtype": "f32", "count": 60, "lo": 64, "hi": 2048, "mix": 1},
        # hydrology: water moving downhill on an elevation raster
        {"name": "water_f64_4096", "kind": "water", "dtype": "f64", "n0": 4096, "n1": 4096, "rule": "flow",
         "boundary": "remove"},
        # diffusion with a source field, one step
        {"name": "coupled_f32_4096", "kind": "coupled", "dtype": "f32", "n0": 4096, "n1": 4096,
         "boundary": "wrap", "padding": "cond"},
    ]


def _side(rng, lo, hi):
    """A side, uniform over its logarithm; every other one a multiple of 32."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    return n if rng.random() < 0.5 else max(lo, n // 32 * 32)


def _steps(rng, most):
    return max(1, min(int(most), int(round(math.exp(rng.uniform(0.0, math.log(max(2, most))))))))


def draw(rng):
    kind = rng.choice(["gather", "gather", "gauss", "life", "heat2d", "heat3d", "batch", "steps_batch", "water",
                       "coupled"])
    bc = rng.choice(["wrap", "remove", "reflect"])
    pad = rng.choice(["cond", "halo"])
    if kind == "gather":
        dtype = rng.choice(["f64", "f64", "f32", "f32", "bf16", "u8", "i32", "i64"])
        fold = rng.choice(["maximum", "minimum"] if dtype in ("u8", "i32") else
                          ["sum", "maximum"] if dtype == "i64" else ["mean", "sum", "maximum"])
        return {"kind": kind, "fold": fold, "shape": rng.choice(["window1", "moore1", "moore2", "vonneumann2",
                                                                 "circle3", "list6"]),
                "dtype": dtype, "n0": _side(rng, 64, 8192), "n1": _side(rng, 64, 8192), "boundary": bc, "padding": pad}
    if kind == "gauss":
        return {"kind": kind, "radius": rng.choice([1, 2, 3]), "dtype": rng.choice(["f32", "bf16"]),
                "n0": _side(rng, 128, 8192), "n1": _side(rng, 128, 8192), "boundary": bc, "padding": pad}
    if kind == "life":
        n0, n1 = _side(rng, 64, 8192), _side(rng, 64, 8192)
        return {"kind": kind, "n0": n0, "n1": n1, "steps": _steps(rng, min(1000, 2.0e10 / (n0 * n1))),
                "rule": rng.choice(["conway", "conway", "highlife"]), "boundary": bc, "padding": pad}
    if kind == "heat2d":
        n0, n1 = _side(rng, 64, 8192), _side(rng, 64, 8192)
        return {"kind": kind, "dtype": rng.choice(["f32", "f32", "f64", "bf16"]), "n0": n0, "n1": n1,
                "steps": _steps(rng, min(300, 1.6e9 / (n0 * n1))), "boundary": bc, "padding": pad}
    if kind == "heat3d":
        n0, n1, n2 = _side(rng, 32, 384), _side(rng, 32, 384), _side(rng, 32, 384)
        return {"kind": kind, "dtype": rng.choice(["f32", "f32", "f64", "bf16"]), "n0": n0, "n1": n1, "n2": n2,
                "steps": _steps(rng, min(300, 1.6e9 / (n0 * n1 * n2))), "boundary": bc, "padding": pad}
    if kind == "batch":
        return {"kind": kind, "dtype": rng.choice(["f32", "f32", "f64", "bf16"]), "count": rng.randrange(8, 61),
                "lo": 64, "hi": rng.choice([512, 1024, 2048]), "mix": rng.randrange(1, 1000)}
    if kind == "steps_batch":
        return {"kind": kind, "dtype": "f32", "count": rng.randrange(4, 31), "lo": 64, "hi": rng.choice([256, 512, 1024]),
                "most": rng.choice([40, 100]), "mix": rng.randrange(1, 1000)}
    if kind == "water":
        return {"kind": kind, "dtype": rng.choice(["f64", "f32"]), "n0": _side(rng, 64, 6000),
                "n1": _side(rng, 64, 6000), "rule": rng.choice(["flow", "downhill"]), "boundary": bc}
    return {"kind": kind, "dtype": rng.choice(["f32", "f64"]), "n0": _side(rng, 64, 8192), "n1": _side(rng, 64, 8192),
            "boundary": bc, "padding": pad}


# ------------------------------------------------------------------ inputs

def _device():
    return torch.device("cuda", torch.cuda.current_device())


def _generator(seed):
    return torch.Generator(device=_device()).manual_seed(int(seed))


def _column_major(a):
    """`a` as the package indexes it: the contiguous axis first."""
    return a.permute(*reversed(range(a.ndim)))


def _field(g, size, dtype, scale=1.0):
    """Uniform values: [0, scale) for floats, 0 .. 99 for integers."""
    if dtype.is_floating_point:
        a = torch.rand(size[::-1], generator=g, device=_device(),
                       dtype=torch.float64 if dtype == torch.float64 else torch.float32)
        a = (a * scale).to(dtype) if scale != 1.0 else a.to(dtype)
    else:
        a = torch.randint(0, 100, size[::-1], generator=g, device=_device(), dtype=torch.int32).to(dtype)
    return _column_major(a)


def _soup(g, size):
    """A Life soup: cells alive with probability 0.3."""
    return _column_major((torch.rand(size[::-1], generator=g, device=_device()) < 0.3).to(torch.uint8))


def _size(case):
    return tuple(case[k] for k in ("n0", "n1", "n2") if k in case)


def _boundary(case, dtype):
    if case["boundary"] == "remove":
        return sh.Remove(0.0 if dtype.is_floating_point else 0)
    return sh.Wrap() if case["boundary"] == "wrap" else sh.Reflect()


def _padding(case):
    return sh.Halo() if case["padding"] == "halo" else sh.Conditional()


# offsets of the stencil shapes (the package's `Positional` for the list)
LIST6 = ((-2, 0), (0, -1), (0, 0), (1, 1), (2, -2), (-1, 2))


def _stencil(shape):
    return {"window1": lambda: sh.Window(1), "moore1": lambda: sh.Moore(1), "moore2": lambda: sh.Moore(2),
            "vonneumann2": lambda: sh.VonNeumann(2), "circle3": lambda: sh.Circle(3),
            "list6": lambda: sh.Positional(*LIST6)}[shape]()


def _gauss_weights(R):
    a = torch.arange(-R, R + 1, dtype=torch.float64)
    w = torch.exp(-(a[:, None] ** 2 + a[None, :] ** 2) / (2 * (R / 2.0) ** 2))
    return (w / w.sum()).to(torch.float32)


FOLDS = {"mean": sh.mean, "sum": sh.sum, "maximum": sh.maximum, "minimum": sh.minimum}
BATCH_SHAPES = ("window1", "circle3", "vonneumann2")
BATCH_FOLDS = ("sum", "maximum", "mean")


def _batch_items(case):
    """(size, shape, fold, steps) of each array of a batch: sides uniform over
    their logarithm, aspect 0.5 .. 2."""
    rng = random.Random(case["mix"])
    items = []
    for _ in range(case["count"]):
        side = math.exp(rng.uniform(math.log(case["lo"]), math.log(case["hi"])))
        asp = rng.uniform(0.5, 2.0)
        size = (max(8, int(side * math.sqrt(asp))), max(8, int(side / math.sqrt(asp))))
        items.append((size, rng.choice(BATCH_SHAPES), rng.choice(BATCH_FOLDS), rng.randint(10, case.get("most", 10))))
    return items


ALPHA2, ALPHA3, SOURCE, FLOW = 0.2, 0.15, 0.0625, 0.125


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    if kind in ("batch", "steps_batch"):
        dtype = DTYPES[case["dtype"]]
        if kind == "batch":
            calls = []
            for size, shape, fold, _ in _batch_items(case):
                A = sh.StencilArray(_field(g, size, dtype), _stencil(shape), boundary=sh.Remove(0.0))
                calls.append((FOLDS[fold], sh.colmajor_empty(size, dtype, _device()), A))
            return {"kind": kind, "plan": sh.BatchPlan(calls), "dests": [c[1] for c in calls]}
        f = sh.Laplacian(ALPHA2)
        return {"kind": kind, "items": [
            (f, sh.SwitchingStencilArray(_field(g, size, dtype), sh.VonNeumann(1), boundary=sh.Wrap()), steps)
            for size, _, _, steps in _batch_items(case)]}
    size = _size(case)
    if kind == "life":
        A = sh.SwitchingStencilArray(_soup(g, size), sh.Moore(1), boundary=_boundary(case, torch.uint8),
                                     padding=_padding(case))
        f = sh.LifeRule() if case["rule"] == "conway" else sh.LifeRule(birth=(3, 6), survive=(2, 3))
        return {"kind": kind, "f": f, "A": A, "steps": case["steps"]}
    dtype = DTYPES[case["dtype"]]
    bc = _boundary(case, dtype)
    if kind == "gather":
        A = sh.StencilArray(_field(g, size, dtype), _stencil(case["shape"]), boundary=bc, padding=_padding(case))
        return {"kind": kind, "f": FOLDS[case["fold"]], "A": A}
    if kind == "gauss":
        K = sh.Kernel(sh.Window(case["radius"]), _gauss_weights(case["radius"]).numpy())
        A = sh.StencilArray(_field(g, size, dtype), K, boundary=bc, padding=_padding(case))
        return {"kind": kind, "A": A, "dest": sh.colmajor_empty(size, dtype, _device())}
    if kind in ("heat2d", "heat3d"):
        nd = len(size)
        A = sh.SwitchingStencilArray(_field(g, size, dtype), sh.VonNeumann(1, nd), boundary=bc, padding=_padding(case))
        return {"kind": "heat", "f": sh.Laplacian(ALPHA2 if nd == 2 else ALPHA3), "A": A, "steps": case["steps"]}
    if kind == "water":
        water = sh.StencilArray(_field(g, size, dtype), sh.Moore(1), boundary=bc)
        land = sh.StencilArray(_field(g, size, dtype, 10.0), sh.Moore(1), boundary=bc)
        f = sh.Scatter.downhill_flow(FLOW) if case["rule"] == "flow" else sh.Scatter.downhill(FLOW)
        return {"kind": kind, "f": f, "dest": sh.colmajor_empty(size, dtype, _device()), "water": water, "land": land}
    assert kind == "coupled"
    S = sh.SwitchingStencilArray(_field(g, size, dtype), sh.VonNeumann(1), boundary=bc, padding=_padding(case))
    f = sh.Terms(sh.Laplacian(ALPHA2), sh.Scaled(SOURCE, sh.center))
    return {"kind": kind, "f": f, "A": S, "source": _field(g, size, dtype)}


def run(state):
    kind = state["kind"]
    if kind == "gather":
        return sh.mapstencil(state["f"], state["A"])
    if kind == "gauss":
        return sh.mapstencil_(sh.kernelproduct, state["dest"], state["A"], flags=ASYNC)
    if kind in ("life", "heat"):
        A = state["A"] = sh.mapstencil_steps(state["f"], state["A"], state["steps"], flags=ASYNC)
        return [A.interior(A.source), A.interior(A.dest)]
    if kind == "batch":
        state["plan"].run(flags=ASYNC)
        return state["dests"]
    if kind == "steps_batch":
        arrays = sh.mapstencil_steps_batch(state["items"], flags=ASYNC)
        state["items"] = [(f, A, n) for (f, _, n), A in zip(state["items"], arrays)]
        return [x for A in arrays for x in (A.source, A.dest)]
    if kind == "water":
        return sh.scatterstencil_(state["f"], "+", state["dest"], state["water"], state["land"], flags=ASYNC)
    assert kind == "coupled"
    A = state["A"] = sh.mapstencil_(state["f"], state["A"], state["source"], flags=ASYNC)
    return A.interior(A.source)


# ------------------------------------------------------------ what it costs

LENGTHS = {"window1": 9, "moore1": 8, "moore2": 24, "vonneumann2": 12, "circle3": 37, "list6": 6}


def _esize(name):
    return torch.empty(0, dtype=DTYPES[name]).element_size()


def work(case):
    """Every input read once and every output written once; one operation per
    fold step (two where it multiplies), the Laplacian's three more."""
    kind = case["kind"]
    if kind in ("batch", "steps_batch"):
        es, cells, flops = _esize(case["dtype"]), 0, 0
        for size, shape, _, steps in _batch_items(case):
            n = size[0] * size[1]
            cells += n * (2 if kind == "steps_batch" else 1)
            flops += n * (LENGTHS[shape] if kind == "batch" else 7 * steps)
        return {"bytes": (3 * cells // 2 if kind == "steps_batch" else 2 * cells) * es, "flops": flops}
    cells = math.prod(_size(case))
    if kind == "life":
        return {"bytes": 3 * cells, "flops": 10 * cells * case["steps"]}
    es = _esize(case["dtype"])
    if kind == "gather":
        return {"bytes": 2 * es * cells, "flops": LENGTHS[case["shape"]] * cells}
    if kind == "gauss":
        return {"bytes": 2 * es * cells, "flops": 2 * (2 * case["radius"] + 1) ** 2 * cells}
    if kind in ("heat2d", "heat3d"):
        return {"bytes": 3 * es * cells, "flops": (7 if kind == "heat2d" else 9) * cells * case["steps"]}
    if kind == "water":
        return {"bytes": 4 * es * cells, "flops": 8 * 4 * cells}
    return {"bytes": 3 * es * cells, "flops": 9 * cells}


# ------------------------------------------------------- 64-bit restatement

def _offsets(shape):
    def box(R, keep):
        return [(i, j) for j in range(-R, R + 1) for i in range(-R, R + 1) if keep(i, j)]
    return {"window1": lambda: box(1, lambda i, j: True), "moore1": lambda: box(1, lambda i, j: i or j),
            "moore2": lambda: box(2, lambda i, j: i or j),
            "vonneumann2": lambda: box(2, lambda i, j: 0 < abs(i) + abs(j) <= 2),
            "circle3": lambda: box(3, lambda i, j: i * i + j * j <= 12), "list6": lambda: list(LIST6)}[shape]()


def _outside(a, R, boundary):
    """`a` with R cells around it: zeros, the wrapped or the mirrored cells."""
    for d in range(a.ndim):
        n = a.shape[d]
        i = torch.arange(-R, n + R, device=a.device)
        if boundary == "wrap":
            a = a.index_select(d, i % n)
        elif boundary == "reflect":
            a = a.index_select(d, torch.where(i < 0, -i, torch.where(i >= n, 2 * n - 2 - i, i)))
        else:
            size = list(a.shape)
            size[d] = R
            z = a.new_zeros(size)
            a = torch.cat([z, a, z], d)
    return a


def _at(p, o, R, size):
    return p[tuple(slice(R + o[d], R + o[d] + size[d]) for d in range(len(size)))]


def _fold(a, offs, boundary, fold, weights=None):
    R = max(max(abs(c) for c in o) for o in offs)
    p, acc = _outside(a, R, boundary), None
    for k, o in enumerate(offs):
        v = _at(p, o, R, a.shape)
        if weights is not None:
            v = v * weights[k]
        acc = v.clone() if acc is None else (torch.maximum(acc, v) if fold == "maximum" else
                                             torch.minimum(acc, v) if fold == "minimum" else acc.add_(v))
    return acc / len(offs) if fold == "mean" else acc


def _laplacian(a, alpha, boundary):
    nd = a.ndim
    offs = [tuple(s if e == d else 0 for e in range(nd)) for d in range(nd) for s in (-1, 1)]
    return a + alpha * (_fold(a, offs, boundary, "sum") - 2 * nd * a)


def _as_float(value, dtype):
    """A coefficient as an array of `dtype` (16-bit storage: Float32) holds it."""
    return float(torch.tensor(value, dtype=torch.float64 if dtype == torch.float64 else torch.float32))


def exact(case, seed):
    kind = case["kind"]
    if kind == "life" or case["dtype"] in ("u8", "i32", "i64"):
        return None  # whole numbers
    g = _generator(seed)
    dtype = DTYPES[case["dtype"]]
    if kind in ("batch", "steps_batch"):
        out = []
        for size, shape, fold, steps in _batch_items(case):
            a = _field(g, size, dtype).double()
            if kind == "batch":
                out.append(_fold(a, _offsets(shape), "remove", fold))
                continue
            prev = a
            for _ in range(steps):
                prev, a = a, _laplacian(a, _as_float(ALPHA2, dtype), "wrap")
            out += [a, prev]
        return out
    size = _size(case)
    a = _field(g, size, dtype).double()
    bc = case["boundary"]
    if kind == "gather":
        return _fold(a, _offsets(case["shape"]), bc, case["fold"])
    if kind == "gauss":
        R = case["radius"]
        w = _gauss_weights(R).double()
        offs = [(i, j) for j in range(-R, R + 1) for i in range(-R, R + 1)]
        return _fold(a, offs, bc, "sum", [float(w[i + R, j + R]) for i, j in offs])
    if kind in ("heat2d", "heat3d"):
        alpha, prev = _as_float(ALPHA2 if kind == "heat2d" else ALPHA3, dtype), a
        for _ in range(case["steps"]):
            prev, a = a, _laplacian(a, alpha, bc)
        return [a, prev]
    if kind == "water":
        land = _field(g, size, dtype, 10.0).double()
        # each cell sends along every offset; its target is the cell there,
        # wrapped, mirrored, or none outside the array
        out = torch.zeros_like(a)
        p = _outside(land, 1, bc)
        index = []
        for d in range(2):
            i = torch.arange(-1, size[d] + 1, device=a.device)
            index.append(i % size[d] if bc == "wrap" else
                         torch.where(i < 0, -i, torch.where(i >= size[d], 2 * size[d] - 2 - i, i)) if bc == "reflect" else i)
        for o in _offsets("moore1"):
            drop = land - _at(p, o, 1, size)
            v = torch.where(drop > 0, a * (drop if case["rule"] == "flow" else 1.0) * FLOW, torch.zeros_like(a))
            ti, tj = (index[d][1 + o[d]: 1 + o[d] + size[d]] for d in range(2))
            ki, kj = ((t >= 0) & (t < size[d]) for d, t in enumerate((ti, tj)))
            v, ti, tj = v[ki][:, kj], ti[ki], tj[kj]
            rows = torch.zeros((size[0], v.shape[1]), dtype=v.dtype, device=v.device).index_add_(0, ti, v)
            out.index_add_(1, tj, rows)
        return out
    source = _field(g, size, dtype).double()
    return _laplacian(a, _as_float(ALPHA2, dtype), bc) + SOURCE * source
