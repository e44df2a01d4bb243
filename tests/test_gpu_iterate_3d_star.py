"""3-D star iterations with up to four steps per launch (csrc/zmarch_kernel.hpp),
with that kernel forced: every boundary, padding, 4-byte and 16-bit storage,
sizes around its tiles (56 cells of columns and rows) and its smallest axis."""
import numpy as np
import pytest

import stencils_hip as sh
from stencils_hip import _lib

pytestmark = pytest.mark.gpu

# the last two: enough planes for several chunks, a last row tile of one and of two rows
SIZES = [(16, 16, 16), (56, 57, 17), (57, 56, 33), (64, 17, 40), (113, 60, 23), (20, 120, 19), (60, 113, 90), (17, 58, 300)]
BOUNDS = {"remove": lambda: sh.Remove(0.25), "wrap": sh.Wrap, "reflect": sh.Reflect}


@pytest.fixture(autouse=True)
def star(monkeypatch):
    monkeypatch.setenv("STH_STEPS_KERNEL", "zmarch/4")


@pytest.mark.parametrize("pad", ["cond", "halo"])
@pytest.mark.parametrize("bname", list(BOUNDS))
@pytest.mark.parametrize("size", SIZES, ids=str)
def test_star_f32(gpu, oracle, size, bname, pad):
    A = np.asfortranarray(np.random.default_rng(sum(size)).random(size).astype(np.float32))
    padding = sh.Conditional() if pad == "cond" else sh.Halo()
    bc = sh.Remove(np.float32(0.25)) if bname == "remove" else BOUNDS[bname]()
    for i, steps in enumerate((5, 6, 7, 8, 9, 10, 23)):
        f = sh.Laplacian(0.15) if i % 3 else sh.mean
        g, o = (sh.SwitchingStencilArray(A.copy(order="F"), sh.VonNeumann(1, 3), boundary=bc, padding=padding)
                for _ in range(2))
        g = sh.mapstencil_steps(f, g, steps)
        assert _lib.steps_kernel() == "zmarch/4"
        o = oracle.mapstencil_steps(f, o, steps)
        np.testing.assert_array_equal(g.source, o.source, err_msg=f"{steps} steps, source")
        np.testing.assert_array_equal(g.dest, o.dest, err_msg=f"{steps} steps, dest")


@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("bname", list(BOUNDS))
def test_star_16_bit(gpu, bname, dtype):
    """16-bit storage against single steps."""
    import torch
    gen = torch.Generator(device="cuda").manual_seed(3)
    for size in SIZES:
        a = torch.rand(size[::-1], generator=gen, device="cuda").to(getattr(torch, dtype)).permute(2, 1, 0)
        for pad, steps in ((sh.Conditional(), 14), (sh.Halo(), 9)):
            make = lambda: sh.SwitchingStencilArray(a.clone(), sh.VonNeumann(1, 3), boundary=BOUNDS[bname](),  # noqa: E731
                                                    padding=pad)
            g = sh.mapstencil_steps(sh.Laplacian(0.15), make(), steps)
            assert _lib.steps_kernel() == "zmarch/4"
            h = sh.mapstencil_steps(sh.Laplacian(0.15), make(), steps, graph=False, flags=sh._abi.NO_FUSE)
            assert _lib.steps_kernel() == "single"
            assert torch.equal(g.source, h.source) and torch.equal(g.dest, h.dest), f"{size} {pad!r}"
