"""The gates' quotient n / (1 + e^-z) over the whole range of z: against 64 bits, and what a division makes of infinities and NaN."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def silu(x):
    from aphrodite_engine_amd import mixer_ops as mops
    return mops.act_and_mul(torch.cat([x, torch.ones_like(x)], 1).contiguous(), 0)


@pytest.mark.parametrize("low,high", [(1e-37, 1e-3), (1e-3, 1.0), (1.0, 87.3), (87.3, 88.7)])
def test_silu_against_64_bits(low, high):
    x = torch.logspace(math.log10(low), math.log10(high), 8192, dtype=torch.float64).float().to(DEV).view(2, 4096)
    for z in (x, -x):
        d = z.double()
        # e^-z as 2^(z log2 e): log2 e is 0.22 x 2^-24 off and the product rounds by up to 2^-24, |z| times that of the power, whose own last
        # place is 2 x 2^-24; the sum, the quotient and the product with one round once each
        bound = (1.25 * d.abs() + 2) * torch.sigmoid(-d) + 3
        want = torch.nn.functional.silu(d)
        assert ((silu(z).double() - want).abs() <= bound * 2.0 ** -24 * want.abs() + 2.0 ** -148).all()


def test_silu_of_the_smallest():
    """Half of z, rounded once, down to the least number there is."""
    n = torch.cat([torch.arange(1, 4097), torch.logspace(12, 26.7, 4096, base=2, dtype=torch.float64).long()]).to(torch.int32)      # 1.4e-45 .. 5e-38
    z = n.view(torch.float32).to(DEV).view(2, 4096)
    for x in (z, -z):
        assert torch.equal(silu(x), (x.double() / 2).float())


def test_silu_of_edges():
    inf, nan = float("inf"), float("nan")
    z = torch.tensor([[0.0, -0.0, inf, -inf, nan, 3e38, -3e38, -89.0]], device=DEV)
    got = silu(z).cpu()[0]
    assert got[0] == 0 and got[1] == 0 and torch.signbit(got[1]) and got[2] == inf and got[3].isnan() and got[4].isnan()
    assert got[5] == z[0, 5].item() and got[6] == 0 and got[7].abs() < 1e-36
