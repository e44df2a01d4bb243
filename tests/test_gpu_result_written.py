"""mapstencil's result is written whole: memory that held another pattern
before shows nowhere, at sizes with ragged tiles and in every dimension."""
import pytest
import torch

import stencils_hip as sh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,st", [((3,), sh.Window(1, 1)), ((257,), sh.Window(1, 1)), ((5, 3), sh.Moore(1)),
                                      ((64, 33), sh.Circle(3)), ((1025, 31), sh.Window(2)),
                                      ((7, 5, 3), sh.VonNeumann(1, 3)), ((130, 9, 5), sh.Moore(1, 3))],
                         ids=lambda v: str(v))
@pytest.mark.parametrize("dtype", [torch.float32, torch.float64, torch.int32])
def test_no_cell_keeps_old_memory(gpu, shape, st, dtype):
    dev = torch.device("cuda")
    src = sh.colmajor_empty(shape, dtype, dev)
    src.fill_(1)
    A = sh.StencilArray(src, st, boundary=sh.Remove(1))
    n = src.numel()
    for _ in range(3):
        poison = [torch.full((n,), 77, dtype=dtype, device=dev) for _ in range(4)]
        del poison  # the allocator hands this memory out again
        out = sh.mapstencil(sh.maximum, A)
        assert bool((out == 1).all())
        del out
