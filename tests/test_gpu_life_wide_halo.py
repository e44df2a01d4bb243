"""Life over a stencil whose radius is larger than its offsets reach: the halo
is as wide as the radius, and every cell of it is refreshed."""
import numpy as np
import pytest

import stencils_hip as sh

pytestmark = pytest.mark.gpu


class Ring(sh.Moore):
    """The eight neighbours, with a radius of its own."""

    def __init__(self, radius):
        super().__init__(radius, 2)

    def _offsets(self):
        return sh.Moore(1).offsets()


@pytest.mark.parametrize("radius", [1, 2, 3])
@pytest.mark.parametrize("bname", ["remove", "wrap", "reflect", "use"])
@pytest.mark.parametrize("size", [(48, 32), (41, 33), (100, 77), (256, 64)], ids=str)
def test_halo_as_wide_as_the_radius(gpu, oracle, size, bname, radius):
    A = (np.random.default_rng(radius).random(size) < 0.4).astype(np.uint8)
    bc = {"remove": sh.Remove(np.uint8(1)), "wrap": sh.Wrap(), "reflect": sh.Reflect(), "use": sh.Use()}[bname]
    for rule in (sh.LifeRule(), sh.LifeRule((3, 6), (2, 3))):
        for pad in (sh.Halo("out"), sh.Halo("in")):
            for steps in (1, 2, 7, 12, 30):
                g, o = (sh.SwitchingStencilArray(A.copy(order="F"), Ring(radius), boundary=bc, padding=pad)
                        for _ in range(2))
                g = sh.mapstencil_steps(rule, g, steps)
                o = oracle.mapstencil_steps(rule, o, steps)
                np.testing.assert_array_equal(g.source, o.source, err_msg=f"{rule!r} {pad!r} {steps}")
                np.testing.assert_array_equal(g.dest, o.dest, err_msg=f"{rule!r} {pad!r} {steps}")
