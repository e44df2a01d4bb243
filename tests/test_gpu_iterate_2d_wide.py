"""2-D iterations on rows of several ragged tiles (csrc/march_tiles.hpp): widths
whose spread tiles lie unequal distances apart."""
import numpy as np
import pytest

import stencils_hip as sh

pytestmark = pytest.mark.gpu

BOUNDS = {"remove": lambda v: sh.Remove(v), "wrap": lambda v: sh.Wrap(), "reflect": lambda v: sh.Reflect()}


@pytest.mark.parametrize("bname", list(BOUNDS))
@pytest.mark.parametrize("dtype,n0", [("f32", 895), ("f32", 1119), ("f32", 4001), ("f32", 8191), ("f64", 447),
                                      ("f64", 1501), ("f64", 4095), ("f64", 8191)])
def test_ragged_rows(gpu, oracle, dtype, n0, bname):
    npdt = {"f32": np.float32, "f64": np.float64}[dtype]
    A = np.random.default_rng(n0).random((n0, 17)).astype(npdt)
    for pad in (sh.Conditional(), sh.Halo()):
        make = lambda: sh.SwitchingStencilArray(A.copy(order="F"), sh.VonNeumann(1),  # noqa: E731
                                                boundary=BOUNDS[bname](npdt(3)), padding=pad)
        G = sh.mapstencil_steps(sh.Laplacian(0.2), make(), 19)
        O = oracle.mapstencil_steps(sh.Laplacian(0.2), make(), 19)
        np.testing.assert_array_equal(np.asarray(G.source), np.asarray(O.source), err_msg=repr(pad))
        np.testing.assert_array_equal(np.asarray(G.dest), np.asarray(O.dest), err_msg=repr(pad))


@pytest.mark.parametrize("bname", list(BOUNDS))
@pytest.mark.parametrize("dtype,n0", [("bf16", 1791), ("bf16", 4094), ("i32", 895), ("i32", 8191)])
def test_ragged_rows_equal_single_steps(gpu, dtype, n0, bname):
    """16-bit storage, and a runtime-compiled kernel (Int32, 2^20 cells and more)."""
    import torch
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(n0)
    t = torch.rand((17 if dtype == "bf16" else (1 << 20) // n0 + 7, n0), generator=g, device=dev)
    t = (t.to(torch.bfloat16) if dtype == "bf16" else (t * 1e6).to(torch.int32)).T
    f = sh.Laplacian(0.2) if dtype == "bf16" else sh.maximum
    for pad in (sh.Conditional(), sh.Halo()):
        make = lambda: sh.SwitchingStencilArray(t.clone(), sh.VonNeumann(1),  # noqa: E731
                                                boundary=BOUNDS[bname](3.0 if dtype == "bf16" else 3), padding=pad)
        G = sh.mapstencil_steps(f, make(), 19)
        O = sh.mapstencil_steps(f, make(), 19, graph=False, flags=sh._abi.NO_FUSE)
        assert torch.equal(G.source, O.source) and torch.equal(G.dest, O.dest), repr(pad)
