"""What a first call compiles: a single gather its own kernel and no kernel of
an iteration, an iteration both."""
import numpy as np
import pytest

import stencils_hip as sh

pytestmark = pytest.mark.gpu


def test_single_gather_compiles_one_kernel(gpu, tmp_path, monkeypatch):
    monkeypatch.setenv("STH_JIT_CACHE", str(tmp_path))
    # a shape no other test uses: the process remembers what it has compiled
    st = sh.Positional((1, 1), (-1, 0), (0, 1), (1, -1))
    A = np.asfortranarray(np.random.default_rng(0).integers(0, 99, (1024, 1030)).astype(np.int32))
    for bc in (sh.Wrap(), sh.Reflect()):
        sh.mapstencil(sh.maximum, sh.StencilArray(A.copy(order="F"), st, boundary=bc))
    assert len(list(tmp_path.glob("*.name"))) == 1
    S = sh.SwitchingStencilArray(A.copy(order="F"), st, boundary=sh.Wrap())
    sh.mapstencil_steps(sh.maximum, S, 9)
    assert len(list(tmp_path.glob("*.name"))) == 2
