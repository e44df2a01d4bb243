"""A float32 result stored as bfloat16 rounds to nearest, ties to even, for
every kind of value: ties and near-ties, overflow to infinity, subnormals,
infinities and NaN."""
import pytest
import torch

import stencils_hip as sh

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shift", [1, 255, 8 * 128 + 37, 16 * 128 + 1])
def test_sum_of_two_rounds_like_torch(shift):
    """x + y over all 65536 patterns of x, each with the pattern `shift`
    further on as y: exponent distances from 0 to 16 put the exact sum
    anywhere between two neighbouring bfloat16 values."""
    pat = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    rows = torch.stack([pat, pat.roll(-shift)])            # (2, 65536)
    want = (rows[0].float() + rows[1].float()).to(torch.bfloat16)
    t = sh.colmajor_empty((2, 65536), torch.bfloat16, torch.device("cuda"))
    t.copy_(rows)
    A = sh.StencilArray(t, sh.Positional((0, 0), (1, 0)), boundary=sh.Wrap())
    got = sh.mapstencil(sh.sum, A).cpu()[0]
    assert bool((torch.isnan(got) == torch.isnan(want)).all())
    ok = torch.isnan(want) | (got == want)
    assert bool(ok.all()), (~ok).nonzero()[:5]
