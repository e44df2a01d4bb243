"""Life iterations on packed bits (csrc/lifep_kernel.hpp) against the
step-by-step oracle: both buffers, halos included, must be equal."""
import numpy as np
import pytest

import stencils_hip as sh

pytestmark = pytest.mark.gpu

BOUNDS = {"remove": sh.Remove(np.uint8(0)), "remove1": sh.Remove(np.uint8(1)), "wrap": sh.Wrap(),
          "reflect": sh.Reflect()}
PADS = {"cond": sh.Conditional(), "halo_out": sh.Halo("out"), "halo_in": sh.Halo("in")}

# rows of 2, 3 and 62 packed words, one cell more and one strip more, with
# and without a partial last word; 3 rows (a Halo{:in} interior, mapped several times over), one
# row tile, and enough tiles for 1 to 12 rows per wave
SHAPES = [(66, 5), (65, 40), (95, 17), (1984, 41), (1985, 161), (2016, 700), (1501, 1333), (4001, 1500),
          (3000, 5000)]


@pytest.mark.parametrize("bname", list(BOUNDS))
@pytest.mark.parametrize("shape", SHAPES)
def test_packed_life_iterations(gpu, oracle, shape, bname):
    rng = np.random.default_rng(shape[0] * 7 + shape[1])
    # any nonzero byte is alive
    A = np.where(rng.random(shape) < 0.35, rng.integers(1, 256, shape), 0).astype(np.uint8)
    big = A.size > 1 << 20
    for rule, pad, steps in [(sh.LifeRule(), "cond", 8), (sh.LifeRule(), "halo_out", 9),
                             (sh.LifeRule((3, 6), (2, 3)), "halo_in", 11), (sh.LifeRule((0, 8), (0, 4, 8)), "cond", 10),
                             (sh.LifeRule(), "cond", 21 if big else 67), (sh.LifeRule(), "halo_out", 24 if big else 1100)]:
        make = lambda: sh.SwitchingStencilArray(A.copy(order="F"), sh.Moore(1), boundary=BOUNDS[bname],  # noqa: E731
                                                padding=PADS[pad])
        G = sh.mapstencil_steps(rule, make(), steps, graph=steps % 2 == 1 or steps > 1000)
        O = oracle.mapstencil_steps(rule, make(), steps, nthreads=8)
        msg = f"{rule!r} {pad} {steps} steps"
        np.testing.assert_array_equal(G.source, O.source, err_msg=msg)
        np.testing.assert_array_equal(G.dest, O.dest, err_msg=msg)


@pytest.mark.parametrize("bname", ["remove1", "wrap", "reflect", "use"])
@pytest.mark.parametrize("shape", [(18, 9), (33, 5), (63, 34), (1025, 7), (1039, 33)])
def test_single_steps_on_rows_of_any_length(gpu, oracle, shape, bname):
    """Rows that are no multiple of 16 cells: the last lane's chunk overlaps
    its neighbour's (csrc/life_kernel.hpp), every rows-per-lane variant."""
    from stencils_hip import _lib
    rng = np.random.default_rng(shape[0] + shape[1])
    A = np.where(rng.random(shape) < 0.4, rng.integers(1, 256, shape), 0).astype(np.uint8)
    bc = sh.Use() if bname == "use" else BOUNDS[bname]
    for rule in (sh.LifeRule(), sh.LifeRule((1, 3, 6), (2, 3, 5))):
        for pad in ("halo_in",) if bname == "use" else PADS:
            make = lambda: sh.SwitchingStencilArray(A.copy(order="F"), sh.Moore(1), boundary=bc,  # noqa: E731
                                                    padding=PADS[pad])
            O = oracle.mapstencil_steps(rule, make(), 3)
            for ky in ("ky2", "ky4", "ky8", "ky16"):
                _lib.set_variant(ky)
                try:
                    G = sh.mapstencil_steps(rule, make(), 3)
                finally:
                    _lib.set_variant("")
                np.testing.assert_array_equal(G.source, O.source, err_msg=f"{rule!r} {pad} {ky}")
                np.testing.assert_array_equal(G.dest, O.dest, err_msg=f"{rule!r} {pad} {ky}")


def test_packed_life_rows_of_a_view(gpu, oracle):
    """A grid inside a larger device tensor: rows start on any byte, and the
    cells between the rows are not the iteration's to write."""
    import torch
    rng = np.random.default_rng(5)
    P = rng.integers(0, 2, (301, 90)).astype(np.uint8)
    for lead in (0, 1, 7):
        bufs = []
        for _ in range(2):
            t = sh.colmajor_empty(P.shape, torch.uint8, torch.device("cuda"))
            t.copy_(torch.from_numpy(P))
            bufs.append(t)
        views = [t[lead:lead + 203, 3:80] for t in bufs]
        S = sh.SwitchingStencilArray(stencil=sh.Moore(1), boundary=sh.Wrap(), padding=sh.Conditional(),
                                     _buffers=tuple(views))
        S = sh.mapstencil_steps(sh.LifeRule(), S, 30)
        O = sh.SwitchingStencilArray(np.asfortranarray(P[lead:lead + 203, 3:80]), sh.Moore(1), boundary=sh.Wrap())
        O = oracle.mapstencil_steps(sh.LifeRule(), O, 30)
        np.testing.assert_array_equal(S.source.cpu().numpy(), O.source)
        np.testing.assert_array_equal(S.dest.cpu().numpy(), O.dest)
        for t in bufs:
            rest = t.cpu().numpy()
            rest[lead:lead + 203, 3:80] = P[lead:lead + 203, 3:80]
            np.testing.assert_array_equal(rest, P)
