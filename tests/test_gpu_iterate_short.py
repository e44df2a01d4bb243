"""2-D iterations in launches of two steps (csrc/ymarch_kernel.hpp), which
arrays of few rows and short iterations run: both buffers, halos included,
equal the step-by-step oracle's (16-bit storage and runtime-compiled kernels:
single steps')."""
import numpy as np
import pytest

import stencils_hip as sh
from stencils_hip import _lib

pytestmark = pytest.mark.gpu

BOUNDS = {"remove": lambda v: sh.Remove(v), "wrap": lambda v: sh.Wrap(), "reflect": lambda v: sh.Reflect()}
# 3 to 15 rows, more than one chunk of 14 rows, more than one workgroup of
# four; rows of one cell more than a tile, ragged, of the fewest cells
SIZES = [(16, 3), (17, 4), (225, 5), (895, 14), (113, 15), (1119, 29), (450, 61)]
CASES = [(sh.VonNeumann(1), sh.Laplacian(0.2)), (sh.Window(1), sh.mean), (sh.Moore(1), sh.maximum)]


@pytest.fixture(autouse=True)
def two_steps(monkeypatch):
    monkeypatch.setenv("STH_STEPS_KERNEL", "ymarch/2")


@pytest.mark.parametrize("bname", list(BOUNDS))
@pytest.mark.parametrize("dtype", ["f32", "f64"])
@pytest.mark.parametrize("size", SIZES, ids=str)
def test_two_steps_per_launch(gpu, oracle, size, dtype, bname):
    npdt = {"f32": np.float32, "f64": np.float64}[dtype]
    A = np.random.default_rng(sum(size)).random(size).astype(npdt)
    for st, f in CASES:
        for steps, pad in [(5, sh.Conditional()), (6, sh.Halo()), (8, sh.Conditional()), (12, sh.Halo()),
                           (71, sh.Conditional())]:
            make = lambda: sh.SwitchingStencilArray(A.copy(order="F"), st, boundary=BOUNDS[bname](npdt(3)),  # noqa: E731
                                                    padding=pad)
            G = sh.mapstencil_steps(f, make(), steps)
            assert _lib.steps_kernel() == "ymarch/2"
            O = oracle.mapstencil_steps(f, make(), steps)
            np.testing.assert_array_equal(np.asarray(G.source), np.asarray(O.source), err_msg=f"{st!r} {steps} {pad!r}")
            np.testing.assert_array_equal(np.asarray(G.dest), np.asarray(O.dest), err_msg=f"{st!r} {steps} {pad!r}")


@pytest.mark.parametrize("bname", list(BOUNDS))
@pytest.mark.parametrize("dtype,size", [("bf16", (16, 3)), ("bf16", (902, 14)), ("bf16", (450, 29)),
                                        ("i32", (1 << 18, 5)), ("i32", (80001, 14))])
def test_two_steps_equal_single_steps(gpu, dtype, size, bname):
    import torch
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(size[0])
    t = torch.rand(size[::-1], generator=g, device=dev)
    t = (t.to(torch.bfloat16) if dtype == "bf16" else (t * 1e6).to(torch.int32)).T
    f = sh.Laplacian(0.2) if dtype == "bf16" else sh.maximum
    for pad in (sh.Conditional(), sh.Halo()):
        make = lambda: sh.SwitchingStencilArray(t.clone(), sh.VonNeumann(1),  # noqa: E731
                                                boundary=BOUNDS[bname](3.0 if dtype == "bf16" else 3), padding=pad)
        G = sh.mapstencil_steps(f, make(), 12)
        assert _lib.steps_kernel() == "ymarch/2"
        O = sh.mapstencil_steps(f, make(), 12, graph=False, flags=sh._abi.NO_FUSE)
        assert _lib.steps_kernel() == "single"
        assert torch.equal(G.source, O.source) and torch.equal(G.dest, O.dest), repr(pad)
