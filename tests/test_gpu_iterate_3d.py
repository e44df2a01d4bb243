"""Iterations of 3-D star stencils that run several steps per launch against
the oracle's step-by-step loop, bit for bit, for both buffers and their
halos: sizes around the kernel's tiles (56 cells of columns and rows, its
smallest axis), uneven axes, step counts that leave every remainder."""
import numpy as np
import pytest

import stencils_hip as sh

pytestmark = pytest.mark.gpu

SIZES = [(16, 16, 16), (56, 57, 17), (57, 56, 33), (64, 17, 40), (113, 60, 23), (20, 120, 19)]


@pytest.mark.parametrize("pad", ["cond", "halo"])
@pytest.mark.parametrize("bname", ["remove", "wrap", "reflect"])
@pytest.mark.parametrize("size", SIZES, ids=str)
def test_iterate_3d(gpu, oracle, size, bname, pad):
    rng = np.random.default_rng(sum(size))
    for i, steps in enumerate((3, 4, 5, 6, 7, 8, 9, 10, 23)):
        f = sh.Laplacian(0.15) if i % 3 else sh.mean
        A = np.asfortranarray(rng.random(size).astype(np.float32))
        bc = {"remove": sh.Remove(np.float32(0.25)), "wrap": sh.Wrap(), "reflect": sh.Reflect()}[bname]
        padding = sh.Conditional() if pad == "cond" else sh.Halo()
        g, o = (sh.SwitchingStencilArray(A.copy(order="F"), sh.VonNeumann(1, 3), boundary=bc, padding=padding)
                for _ in range(2))
        g = sh.mapstencil_steps(f, g, steps)
        o = oracle.mapstencil_steps(f, o, steps)
        np.testing.assert_array_equal(g.source, o.source, err_msg=f"{steps} steps, source")
        np.testing.assert_array_equal(g.dest, o.dest, err_msg=f"{steps} steps, dest")


@pytest.mark.parametrize("bname", ["remove", "wrap", "reflect"])
def test_iterate_3d_bf16(gpu, bname):
    """bfloat16 storage: the multi-step launches equal single steps."""
    import torch
    a = torch.rand((40, 61, 70), device="cuda").to(torch.bfloat16).permute(2, 1, 0)
    bc = {"remove": sh.Remove(0.5), "wrap": sh.Wrap(), "reflect": sh.Reflect()}[bname]
    g = sh.SwitchingStencilArray(a.clone(), sh.VonNeumann(1, 3), boundary=bc)
    h = sh.SwitchingStencilArray(a.clone(), sh.VonNeumann(1, 3), boundary=bc)
    g = sh.mapstencil_steps(sh.Laplacian(0.15), g, 14)
    for _ in range(14):
        h = sh.mapstencil_(sh.Laplacian(0.15), h)
    assert torch.equal(g.source, h.source) and torch.equal(g.dest, h.dest)
