"""Maximum and minimum of one-byte integers on arrays that compile a
specialisation: the kernel that keeps two cells per register against the
oracle, cell for cell (whole numbers: no tolerance), at row lengths around its
16 cells per lane, narrow and wide, for shapes with and without holes."""
import numpy as np
import pytest

import stencils_hip as sh

pytestmark = pytest.mark.gpu

SHAPES = [sh.Moore(2), sh.Window(1), sh.Circle(3), sh.Positional((0, 2), (0, -1)),
          sh.Positional((-3, 0), (1, 0), (3, 3), (2, -1)), sh.VonNeumann(2)]
SIZES = [(1024, 1024), (1043, 1031), (16, 65549), (17, 65537), (32, 32771), (35, 31001), (34, 32001), (2047, 513), (33, 47, 701)]


@pytest.mark.parametrize("pad", ["cond", "halo"])
@pytest.mark.parametrize("bname", ["remove", "wrap", "reflect"])
@pytest.mark.parametrize("size", SIZES, ids=str)
def test_byte_extremes(gpu, oracle, size, bname, pad):
    for i, st in enumerate(SHAPES):
        dt, f = ((np.uint8, sh.maximum), (np.int8, sh.minimum), (np.int8, sh.maximum), (np.uint8, sh.minimum))[
            (i + len(bname) + len(pad) + size[0]) % 4]
        if len(size) == 3 and pad == "halo":
            pytest.skip("a halo of a 2-D stencil over 3-D arrays is covered by the general tests")
        info = np.iinfo(dt)
        rng = np.random.default_rng(i)
        A = np.asfortranarray(rng.integers(info.min, info.max + 1, size).astype(dt))
        bc = {"remove": sh.Remove(dt(3)), "wrap": sh.Wrap(), "reflect": sh.Reflect()}[bname]
        padding = sh.Conditional() if pad == "cond" else sh.Halo()
        ga, oa = (sh.StencilArray(A.copy(order="F"), st, boundary=bc, padding=padding) for _ in range(2))
        np.testing.assert_array_equal(sh.mapstencil(f, ga), oracle.mapstencil(f, oa), err_msg=repr(st))
    assert any("/bytes" in v for v in sh._lib.tuning_table().values())


@pytest.mark.parametrize("bname", ["remove", "wrap", "reflect"])
def test_byte_extremes_eight_rows(gpu, oracle, bname):
    """From 2^25 cells a lane owns eight rows (reach up to 2)."""
    rng = np.random.default_rng(7)
    A = np.asfortranarray(rng.integers(0, 256, (8211, 4099)).astype(np.uint8))
    bc = {"remove": sh.Remove(np.uint8(3)), "wrap": sh.Wrap(), "reflect": sh.Reflect()}[bname]
    ga, oa = (sh.StencilArray(A, sh.Moore(2), boundary=bc) for _ in range(2))
    np.testing.assert_array_equal(sh.mapstencil(sh.maximum, ga), oracle.mapstencil(sh.maximum, oa))
