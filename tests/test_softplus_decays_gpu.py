"""Decays exp(-rate softplus(a)) over the whole range of a, as the delta rule's scan and its chunks apply them: a state that only decays."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("chunks", [False, True])
@pytest.mark.parametrize("channel", [False, True])
def test_decays_over_the_range_of_their_gates(monkeypatch, chunks, channel):
    from aphrodite_engine_amd import mixer_ops as mops
    monkeypatch.setattr(mops, "DELTA_CHUNKED_FROM", 1 if chunks else 1 << 30)
    monkeypatch.setattr(mops, "delta_chunks_pay", lambda *a: chunks)
    H, d, e = 4, 64, 16
    edges = [-float("inf"), -110.0, -88.0, -87.0, -20.0, -1e-3, -0.0, 1e-30, 1.0, 19.99, 20.01, 88.0, 89.0, 3e38]
    x = torch.cat([torch.tensor(edges), torch.linspace(-30, 30, H * d - len(edges))]).to(DEV).view(H, d)
    na = H * d if channel else H
    a = x.reshape(1, -1) if channel else x[:, ::5][:, :1].reshape(1, -1)
    i32 = lambda v: torch.tensor([v], dtype=torch.int32, device=DEV)
    for rate in (1e-3, 0.7, 16.0):
        state = torch.ones(1, H, d, e, device=DEV)
        z = torch.zeros(1, H * d, device=DEV)
        mops.gated_delta_scan(z, z, torch.zeros(1, H * e, device=DEV), torch.full((1, H), -200.0, device=DEV), a.contiguous(),
                              torch.full((H,), rate, device=DEV).log(), torch.zeros(na, device=DEV), state, i32(0), i32(0), i32(1), i32(1), H, H, 1.0)
        r = torch.full((H,), rate, device=DEV).log().double().exp().cpu()[:, None]      # (the rounded logarithm's)
        ln = -r * torch.nn.functional.softplus(a.double().cpu().view(H, -1), threshold=1e9).nan_to_num(posinf=3e38)
        want = ln.exp().expand(H, d)
        got = state[0].double().cpu()
        assert torch.equal(got, got[:, :, :1].expand_as(got))
        # g = e^ln: an error of (softplus 2.3, exp of a_log 1.5, the product 0.5) x 2^-24 of ln, 1.5 x 2^-24 of g; below 2^-120 fp32 itself runs out
        bound = want * ((4.3 * ln.abs()).clamp(max=1e3) + 1.5) * 2.0 ** -24 + 2.0 ** -140
        assert (got[:, :, 0] - want).abs().le(bound).all(), (rate, ((got[:, :, 0] - want).abs() / bound).max())


@pytest.mark.parametrize("low,high", [(-87.3, -20.0), (-20.0, -1.0), (-1.0, 0.0), (0.0, 0.54), (0.54, 20.0), (20.0, 1e4)])
def test_softplus_against_64_bits(low, high):
    """A state-space memory's first token writes softplus(step size) k v^T: with ones for k and v, softplus itself."""
    from aphrodite_engine_amd import mixer_ops as mops
    T, H, d = 256, 128, 16
    g = torch.Generator(device=DEV).manual_seed(7)
    z = torch.rand(T, H, generator=g, device=DEV) * (high - low) + low
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    one = torch.ones(T, H * d, device=DEV)
    state = torch.zeros(mops.memory_state_shapes(T, H, d, d, mops.MEMORY_STATE_SPACE)[0], device=DEV)
    zero = torch.zeros(H, device=DEV)
    mops.outer_memory_scan(one[:, :d].contiguous(), one[:, :d].contiguous(), one, (state, ), i32(range(T)), i32(range(T)), i32([1] * T), i32([0] * T), H,
                           mops.MEMORY_STATE_SPACE, gate_i=z, qk_heads=1, a_log=zero, dt_bias=zero, skip=zero)
    got, x = state[:, :, 0, 0].double(), torch.exp(-z.double().abs())
    want = z.double().clamp(min=0) + torch.log1p(x)
    ulp = lambda v: torch.exp2(v.log2().floor() - 23).clamp(min=2.0 ** -149)
    # rounded once itself; e^-|z| is right to a last place, of which 1 / (1 + x) arrives; what follows a number's first part rounds below 0.06 x 2^-24 of it
    bound = ulp(want) / 2 + ulp(x.clamp(min=1e-45)) / (1 + x) + 0.06 * 2.0 ** -24 * torch.log1p(x)
    err = (got - want).abs()
    assert (err <= bound).all(), float((err / bound).max())
