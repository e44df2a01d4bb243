"""A batch of several 2-D variants is one launch of the kernel that holds them
all: every shape and reduction it can be given, more jobs than one look at the
job table covers (64), sizes around a tile, against one call per job, bit for
bit (both run the same fold expressions)."""
import numpy as np
import pytest

import stencils_hip as sh

pytestmark = pytest.mark.gpu

SHAPES = [sh.Window(1), sh.Window(2), sh.Window(3), sh.Moore(1), sh.Moore(2), sh.VonNeumann(1), sh.VonNeumann(2),
          sh.VonNeumann(3), sh.Circle(1), sh.Circle(2), sh.Circle(3)]
FOLDS = [sh.sum, sh.mean, sh.minimum, sh.maximum]


@pytest.mark.parametrize("dtype", ["float32", "float64", "bfloat16"])
@pytest.mark.parametrize("njobs", [2, 45, 64, 65, 200])
def test_merged_batch(gpu, njobs, dtype):
    import torch
    dt = getattr(torch, dtype)
    g = torch.Generator(device="cuda").manual_seed(njobs)
    every = [(f, st) for st in SHAPES for f in FOLDS] + [(sh.Laplacian(0.2), sh.VonNeumann(1))]
    sizes = [(8, 9), (256, 16), (257, 17), (1023, 33), (64, 300), (513, 129)]
    calls, alone = [], []
    for i in range(njobs):
        f, st = every[(i * 7) % len(every)]
        n0, n1 = sizes[i % len(sizes)]
        a = torch.rand((n1, n0), generator=g, device="cuda", dtype=torch.float32).to(dt).T
        bc = (sh.Remove(0.5), sh.Wrap(), sh.Reflect())[i % 3]
        A = sh.StencilArray(a, st, boundary=bc, padding=sh.Halo() if i % 4 == 3 else sh.Conditional())
        calls.append((f, sh.colmajor_empty((n0, n1), dt, "cuda"), A))
        alone.append((f, sh.colmajor_empty((n0, n1), dt, "cuda"), A))
    sh.BatchPlan(calls).run()
    for f, d, A in alone:
        sh.mapstencil_(f, d, A)
    for i, (x, y) in enumerate(zip(calls, alone)):
        np.testing.assert_array_equal(x[1].float().cpu().numpy(), y[1].float().cpu().numpy(),
                                      err_msg=f"job {i}: {x[0]!r} {x[2]!r}")


def test_large_batch_stays_apart(gpu):
    """Variants of more than 8192 tiles on average keep a launch each."""
    import torch
    g = torch.Generator(device="cuda").manual_seed(1)
    calls, alone = [], []
    for i in range(24):
        a = torch.rand((1800, 2001), generator=g, device="cuda").T
        f, st = (sh.sum, sh.Window(1)) if i % 2 else (sh.maximum, sh.Circle(3))
        A = sh.StencilArray(a, st, boundary=sh.Wrap())
        calls.append((f, sh.colmajor_empty((2001, 1800), torch.float32, "cuda"), A))
        alone.append((f, sh.colmajor_empty((2001, 1800), torch.float32, "cuda"), A))
    sh.BatchPlan(calls).run()
    for (f, x, _), (_, y, A) in zip(calls, alone):
        sh.mapstencil_(f, y, A)
        assert torch.equal(x, y)
