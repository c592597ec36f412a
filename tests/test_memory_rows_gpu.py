"""Short segments of the gated outer-product memories (csrc/mixers/outer_memory.hip, outer_memory_rows_kernel): against the recurrence in 64
bits, token by token, over segment lengths around its stages, row and column counts around its tiles, fresh and continued slots; value
heads of no multiple of 4, which take the other form, beside them."""
import pytest
import torch
from torch.nn import functional as F

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64


def run(mode, lens, heads, d, e, groups=0, dtype=torch.bfloat16, seed=0):
    from aphrodite_engine_amd import mixer_ops as mops
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    T, n, qk = sum(lens), len(lens), groups or heads
    ctxs = [0 if i % 3 == 1 else 7 for i in range(n)]
    q, k, v = rnd(T, qk * d + 8).to(dtype)[:, :qk * d], rnd(T, qk * d).to(dtype), rnd(T, heads * e).to(dtype)
    state = tuple(rnd(*s) for s in mops.memory_state_shapes(n + 2, heads, d, e, mode))
    for s in state[1:]:                                      # kept once per 16 value columns, all the same
        s.copy_(s[:, :, :1].expand_as(s).clone())
    before = tuple(s.clone() for s in state)
    kw = {0: dict(decay=torch.linspace(0.75, 0.99, heads, device=DEV)),
          1: dict(gate_i=rnd(T, heads).to(dtype), gate_f=(rnd(T, heads) + 2).to(dtype), q_scale=d ** -0.5, gate_cap=15.0),
          2: dict(gate_i=rnd(T, heads).to(dtype), qk_heads=qk, a_log=rnd(heads) * 0.3, dt_bias=rnd(heads) * 0.3, skip=rnd(heads))}[mode]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    slots, starts = list(range(n, 0, -1)), [sum(lens[:i]) for i in range(n)]
    out = mops.outer_memory_scan(q, k, v, state, i32(slots), i32(starts), i32(lens), i32(ctxs), heads, mode, max_q_len=max(lens), **kw)
    q, k, v = (x.to(F64) for x in (q, k, v))
    if mode == 0:
        q, k, v = F.silu(q), F.silu(k), F.silu(v)
    q, k = (x.view(T, qk, d).repeat_interleave(heads // qk, 1) for x in (q, k))
    v = v.view(T, heads, e)
    w = {name: x.to(F64) if torch.is_tensor(x) else x for name, x in kw.items()}
    want, left = torch.empty(T, heads, e, dtype=F64, device=DEV), [s.to(F64) for s in before]
    for i, slot in enumerate(slots):
        S = left[0][slot] * (ctxs[i] > 0)
        N, M = (left[1][slot, :, 0] * (ctxs[i] > 0), left[2][slot, :, 0] * (ctxs[i] > 0)) if mode == 1 else (0, 0)
        for t in range(starts[i], starts[i] + lens[i]):
            a, b = (w["decay"], torch.ones_like(w["decay"])) if mode == 0 else (None, None)
            if mode == 1:
                gi, gf = 15 * torch.tanh(w["gate_i"][t] / 15), F.logsigmoid(15 * torch.tanh(w["gate_f"][t] / 15))
                m = torch.maximum(gf + M, gi)
                a, b, M = torch.exp(gf + M - m), torch.exp(gi - m), m
                N = a[:, None] * N + b[:, None] * k[t]
            if mode == 2:
                b = F.softplus(w["gate_i"][t] + w["dt_bias"])
                a = torch.exp(-torch.exp(w["a_log"]) * b)
            S = a[:, None, None] * S + (b[:, None] * k[t])[:, :, None] * v[t][:, None, :]
            y = (S * q[t][:, :, None] * (d ** -0.5 if mode == 1 else 1)).sum(1)
            if mode == 1:
                y = y / (torch.maximum(((N * q[t]).sum(1) * d ** -0.5).abs(), torch.exp(-M)) + 1e-6)[:, None]
            want[t] = y + w["skip"][:, None] * v[t] if mode == 2 else y
        left[0][slot] = S
        if mode == 1:
            left[1][slot], left[2][slot] = N[:, None], M[:, None]
    # fp32 sums of up to 256 products and 31 steps, and the division by a sum that may be small: far below 1e-4 of the whole
    err = lambda x, y: float((x.to(F64) - y).norm() / y.norm())
    assert err(out.view(T, heads, e), want) < 1e-4
    for s, y in zip(state, left):
        assert err(s, y) < 1e-5
    untouched = [0, n + 1]
    assert all(torch.equal(s[untouched], x[untouched]) for s, x in zip(state, before))


@pytest.mark.parametrize("mode,heads,groups", [(0, 3, 0), (1, 2, 0), (2, 6, 2)])
@pytest.mark.parametrize("d,e", [(64, 128), (128, 256), (16, 4), (24, 60), (31, 64), (33, 68), (100, 72), (130, 132), (256, 48), (64, 66), (20, 7)])
@pytest.mark.parametrize("lens", [[1], [1] * 5, [7, 1, 8, 9, 1, 31]])
def test_recurrence(mode, heads, groups, d, e, lens):
    run(mode, lens, heads, d, e, groups, seed=d + e)


@pytest.mark.parametrize("mode", [0, 1, 2])
def test_fp32_activations(mode):
    run(mode, [1, 3, 1], 2, 96, 80, dtype=torch.float32)
