"""SiluAndMul's quotient for every 16-bit gate: numbers of every size, zeros, infinities and NaN.  The op by itself divides; the quantising form and the
products' epilogues have a reciprocal and a correction instead (silu_quotient) and have to give the op's bits."""
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


def _every(dtype):
    return torch.arange(65536, device="cuda", dtype=torch.int32).to(torch.int16).view(dtype)


def _same_bits(got, want):
    nan = want.isnan()
    assert torch.equal(got.isnan(), nan)
    assert torch.equal(got.view(torch.int16)[~nan], want.view(torch.int16)[~nan])


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("up", [1.0, -0.75])
def test_every_gate_of_the_quantising_form(dtype, up):
    x = torch.cat([_every(dtype).view(64, 1024), torch.full((64, 1024), up, device="cuda", dtype=dtype)], 1)
    want = torch.empty(64, 1024, device="cuda", dtype=dtype)
    ops.silu_and_mul(want, x)
    for scale in (None, torch.ones(1, device="cuda")):
        _same_bits(ops.silu_and_mul_quant_fp8(x, static_scale=scale, want_out=True)[2], want)


# weights of one in units of a column's scale and a row that picks one of them: the gates are the scales
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("m,n", [(70, 16384), (200, 16384), (1300, 32768)])
def test_every_gate_of_an_int4_product(dtype, m, n):
    gates = _every(dtype)
    gates = gates[gates.isfinite() & (gates != 0)]              # (a sum of products loses the sign of zero)
    gates = torch.cat([gates, gates[:-len(gates) % (n // 2)]])
    a = torch.zeros(m, 256, device="cuda", dtype=dtype)
    a[:, 5] = 1
    qw = torch.full((32, n), 0x99999999 - 2 ** 32, device="cuda", dtype=torch.int32)
    qz = torch.full((2, n // 8), 0x77777777, device="cuda", dtype=torch.int32)
    assert ops.wna16_gemm_large_silu_supported(m, n, 256, 2)
    for part in gates.view(-1, n // 2):
        sc = torch.stack([part, torch.ones_like(part)], 1).view(1, n).repeat(2, 1)
        got = ops.wna16_gemm_large_silu(a, qw, qz, sc, 1)
        want = torch.empty(1, n // 2, device="cuda", dtype=dtype)
        ops.silu_and_mul(want, torch.cat([part, torch.ones_like(part)])[None])
        if dtype == torch.bfloat16:                          # (f16 weights: bf16 scales of another range saturate or round there)
            seen = part.float().half().float() == part.float()
            got, want = got[:, seen], want[:, seen]
        _same_bits(got, want.expand_as(got).contiguous())
