"""The one-byte extremes kernel (csrc/bytes_kernel.hpp), forced, with four and
with eight rows per lane: sizes whose last lane starts one to fifteen cells
after its neighbour, row ends inside a word, few rows, many."""
import numpy as np
import pytest

import stencils_hip as sh
from stencils_hip import _lib

pytestmark = pytest.mark.gpu

SHAPES = [sh.Moore(2), sh.Window(1), sh.Positional((0, 2), (0, -1)), sh.Positional((-2, 0), (1, 0), (2, 2)), sh.Circle(3)]
SIZES = [(1024, 1024), (1041, 1033), (32, 32771), (33, 32001), (34, 31001), (47, 22501), (2047, 513), (149797, 7)]


@pytest.mark.parametrize("rows", [4, 8])
@pytest.mark.parametrize("pad", ["cond", "halo"])
@pytest.mark.parametrize("bname", ["remove", "wrap", "reflect"])
@pytest.mark.parametrize("size", SIZES, ids=str)
def test_rows_per_lane(gpu, oracle, monkeypatch, size, bname, pad, rows):
    import torch
    monkeypatch.setenv("STH_BYTES_KY", str(rows))
    _lib.set_variant("/bytes")
    try:
        for i, st in enumerate(SHAPES):
            dt, f = ((np.uint8, sh.maximum), (np.int8, sh.minimum), (np.int8, sh.maximum), (np.uint8, sh.minimum))[
                (i + len(bname) + size[0]) % 4]
            info = np.iinfo(dt)
            A = np.asfortranarray(np.random.default_rng(i).integers(info.min, info.max + 1, size).astype(dt))
            bc = {"remove": sh.Remove(dt(3)), "wrap": sh.Wrap(), "reflect": sh.Reflect()}[bname]
            padding = sh.Conditional() if pad == "cond" else sh.Halo()
            t = sh.colmajor_empty(size, torch.from_numpy(A[:1, :1]).dtype, torch.device("cuda"))
            t.copy_(torch.from_numpy(np.ascontiguousarray(A.T)).T)
            dest = sh.colmajor_empty(size, t.dtype, t.device)
            chosen = sh.autotune(f, dest, sh.StencilArray(t, st, boundary=bc, padding=padding))
            wide = max(abs(c) for o in st.offsets() for c in o) > 2
            assert chosen.endswith(f"/bytes{4 if wide else rows}"), chosen
            o = oracle.mapstencil(f, sh.StencilArray(A, st, boundary=bc, padding=padding))
            np.testing.assert_array_equal(dest.cpu().numpy(), o, err_msg=f"{st!r} {f!r}")
    finally:
        _lib.set_variant("")
