"""Short segments of the gated delta rule (csrc/mixers/delta_rule.hip, gated_delta_rows_kernel): against the recurrence in 64 bits, token by
token, over segment lengths around its stages, row and column counts around its tiles, both kinds of decay, fresh and continued slots;
value heads of no multiple of 4, which take the other form, beside them."""
import pytest
import torch
from torch.nn import functional as F

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64


def run(lens, heads, kv_heads, d, e, channel, dtype=torch.bfloat16, seed=0):
    from aphrodite_engine_amd import mixer_ops as mops
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    T, n, per = sum(lens), len(lens), heads // kv_heads
    ctxs = [0 if i % 3 == 1 else 7 for i in range(n)]
    q, k = rnd(T, kv_heads * d + 8).to(dtype)[:, :kv_heads * d], rnd(T, kv_heads * d).to(dtype)
    v, b, a = rnd(T, heads * e).to(dtype), rnd(T, heads).to(dtype), rnd(T, heads * (d if channel else 1)).to(dtype)
    a_log, dt_bias = rnd(heads) * 0.3, rnd(heads * (d if channel else 1)) * 0.3
    state = rnd(n + 2, heads, d, e)
    before = state.clone()
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    slots, starts = list(range(n, 0, -1)), [sum(lens[:i]) for i in range(n)]
    out = mops.gated_delta_scan(q, k, v, b, a, a_log, dt_bias, state, i32(slots), i32(starts), i32(lens), i32(ctxs), heads, kv_heads, d ** -0.5,
                                max_q_len=max(lens))
    unit = lambda x: x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)
    Q, K = (unit(x.to(F64).view(T, kv_heads, d)).repeat_interleave(per, 1) for x in (q, k))
    Q, V, B = Q * d ** -0.5, v.to(F64).view(T, heads, e), torch.sigmoid(b.to(F64))
    G = torch.exp(-torch.exp(a_log.to(F64))[:, None] * F.softplus(a.to(F64) + dt_bias.to(F64)).view(T, heads, -1))
    want, left = torch.empty(T, heads, e, dtype=F64, device=DEV), before.to(F64)
    for i, slot in enumerate(slots):
        S = left[slot] * (ctxs[i] > 0)
        for t in range(starts[i], starts[i] + lens[i]):
            S = G[t][:, :, None] * S
            S = S + K[t][:, :, None] * (B[t][:, None] * (V[t] - (S * K[t][:, :, None]).sum(1)))[:, None, :]
            want[t] = (S * Q[t][:, :, None]).sum(1)
        left[slot] = S
    err = lambda x, y: float((x.to(F64) - y).norm() / y.norm())
    # fp32 sums of up to 256 products over 31 steps: far below 1e-5 of the whole
    assert err(out.view(T, heads, e), want) < 1e-5 and err(state, left) < 1e-5
    assert torch.equal(state[[0, n + 1]], before[[0, n + 1]])


@pytest.mark.parametrize("channel", [False, True])
@pytest.mark.parametrize("heads,kv_heads", [(3, 3), (4, 2)])
@pytest.mark.parametrize("d,e", [(64, 128), (128, 128), (16, 4), (31, 60), (33, 68), (100, 72), (130, 132), (256, 48), (64, 66), (20, 7)])
@pytest.mark.parametrize("lens", [[1], [1] * 5, [7, 1, 8, 9, 1, 31]])
def test_recurrence(channel, heads, kv_heads, d, e, lens):
    run(lens, heads, kv_heads, d, e, channel, seed=d + e)


@pytest.mark.parametrize("channel", [False, True])
def test_fp32_activations(channel):
    run([1, 3, 1], 2, 1, 96, 80, channel, dtype=torch.float32)
