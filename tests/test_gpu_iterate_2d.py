"""2-D iterations with several steps per launch (csrc/ymarch_kernel.hpp): both
buffers, halos included, equal the step-by-step oracle's (16-bit storage: the
one-step-per-launch path's)."""
import numpy as np
import pytest

import stencils_hip as sh

pytestmark = pytest.mark.gpu

# widths around one and two tiles of 56 vectors (224 f32, 112 f64, 448 bf16
# cells) and around the width from which ragged tiles are spread
WIDTHS = {"f32": [16, 17, 223, 224, 225, 231, 233, 451, 1001], "f64": [16, 19, 111, 113, 119, 122, 227, 448],
          "bf16": [16, 18, 446, 450, 460, 902], "i32": [17, 224, 229, 500]}
BOUNDS = {"remove": lambda t: sh.Remove(t(3)), "wrap": lambda t: sh.Wrap(), "reflect": lambda t: sh.Reflect()}
CASES = [(sh.VonNeumann(1), sh.Laplacian(0.2)), (sh.Window(1), sh.mean), (sh.Moore(1), sh.maximum)]


def _same(a, b, msg):
    np.testing.assert_array_equal(np.asarray(a), np.asarray(b), err_msg=msg)


@pytest.mark.parametrize("bname", list(BOUNDS))
@pytest.mark.parametrize("dtype", ["f32", "f64"])
def test_steps_per_launch(gpu, oracle, dtype, bname):
    npdt = {"f32": np.float32, "f64": np.float64}[dtype]
    rng = np.random.default_rng(17)
    for w, n0 in enumerate(WIDTHS[dtype]):
        A = rng.random((n0, (16, 37, 201)[w % 3])).astype(npdt)
        for st, f in CASES:
            # fewer steps than one launch takes, one launch, and many
            for steps, pad in [(3, sh.Conditional()), (5, sh.Halo("out")), (9, sh.Conditional()), (10, sh.Halo("out")),
                               (31, sh.Conditional()), (29, sh.Halo("in"))]:
                if isinstance(pad, sh.Halo) and pad.mode == "in" and min(A.shape) < 18:
                    continue
                make = lambda: sh.SwitchingStencilArray(A.copy(order="F"), st, boundary=BOUNDS[bname](npdt),  # noqa: E731
                                                        padding=pad)
                G = sh.mapstencil_steps(f, make(), steps, graph=steps > 9)
                O = oracle.mapstencil_steps(f, make(), steps, nthreads=4)
                msg = f"{A.shape} {st!r} {f!r} {steps} {pad!r}"
                _same(G.source, O.source, msg)
                _same(G.dest, O.dest, msg)


@pytest.mark.parametrize("bname", list(BOUNDS))
def test_steps_per_launch_long(gpu, oracle, bname):
    """Enough launches that 32 of them replay as one graph."""
    A = np.random.default_rng(3).random((70, 40)).astype(np.float32)
    make = lambda: sh.SwitchingStencilArray(A.copy(order="F"), sh.VonNeumann(1),  # noqa: E731
                                            boundary=BOUNDS[bname](np.float32))
    G = sh.mapstencil_steps(sh.Laplacian(0.2), make(), 661)
    O = oracle.mapstencil_steps(sh.Laplacian(0.2), make(), 661)
    _same(G.source, O.source, "661 steps")
    _same(G.dest, O.dest, "661 steps")


@pytest.mark.parametrize("bname", list(BOUNDS))
@pytest.mark.parametrize("dtype", ["bf16", "i32"])
def test_steps_per_launch_equal_single_steps(gpu, dtype, bname):
    import torch
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(11)
    bc = {"remove": sh.Remove(3.0 if dtype == "bf16" else 3), "wrap": sh.Wrap(), "reflect": sh.Reflect()}[bname]
    cases = CASES if dtype == "bf16" else [(sh.VonNeumann(1), sh.maximum)]
    for w, n0 in enumerate(WIDTHS[dtype]):
        # Int32 runs a runtime-compiled kernel, on arrays of 2^20 cells and more
        shape = (n0, (16, 37, 120)[w % 3] if dtype == "bf16" else (1 << 20) // n0 + 7)
        t = torch.rand(shape[::-1], generator=g, device=dev)
        t = (t.to(torch.bfloat16) if dtype == "bf16" else (t * 1e6).to(torch.int32)).T
        for st, f in cases:
            for pad in (sh.Conditional(), sh.Halo()):
                make = lambda: sh.SwitchingStencilArray(t.clone(), st, boundary=bc, padding=pad)  # noqa: E731
                G = sh.mapstencil_steps(f, make(), 22)
                O = sh.mapstencil_steps(f, make(), 22, graph=False, flags=sh._abi.NO_FUSE)
                same = torch.equal(G.source, O.source), torch.equal(G.dest, O.dest)
                assert all(same), f"{shape} {st!r} {f!r} {pad!r}"
