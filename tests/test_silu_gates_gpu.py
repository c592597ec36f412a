"""SiluAndMul's quotient for every 16-bit gate: numbers of every size, zeros, infinities and NaN."""
import pytest
import torch

from aphrodite_engine_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_every_gate(dtype):
    gate = torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(dtype)
    out = torch.empty(1024, 64, device="cuda", dtype=dtype)
    ops.silu_and_mul(out, torch.cat([gate.view(1024, 64), torch.ones(1024, 64, device="cuda", dtype=dtype)], 1))
    got, g = out.view(-1), gate.double()
    want = g / (1 + torch.exp(-g))
    want[g < -128 / 1.4426950408889634] = -0.0              # e^-gate is beyond fp32
    want[g == -float("inf")] = float("nan")
    nan = want.isnan()
    assert torch.equal(got.isnan(), nan)
    ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    # one rounding to the type; the exponential's argument and value in fp32; the smallest numbers' spacing
    bound = want.abs() * (ulp + 2.0 ** -22 + g.abs().clamp(max=100) * 2.0 ** -24) + (2.0 ** -25 if dtype == torch.float16 else 2.0 ** -134)
    finite = ~nan & ~want.isinf()
    assert bool(((got.double() - want).abs() <= bound)[finite].all())
    assert torch.equal(got[want.isinf()].double(), want[want.isinf()])
    assert torch.equal(torch.signbit(got[~nan]), torch.signbit(gate[~nan]))
