"""Prompt portions over keys and values made from the latents they see: against 64-bit math on the module's own weights, beside decoded
rows, behind contexts, with windows, sinks and both kinds of gate; the gathered rows alone; when it runs."""
import pytest
import torch

from aphrodite_engine_amd import mixers as M
from aphrodite_engine_amd import mixer_ops as mops
from aphrodite_engine_amd.step_batch import StepBatch

pytestmark = pytest.mark.gpu
WIDTH, R, D = 256, 192, 128


def _module(heads, q_rank=0, gate="head", window=0, sink=True, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    with torch.device("cuda"):
        m = M.LatentAttention(WIDTH, heads, D, 0, D, q_rank, R, D ** -0.5, M.RotaryFrequencies(0, 1.0), 1e-5, torch.bfloat16, gate=gate,
                              window=window, sink=sink, project=False)
    for p, std in ((m.in_proj.weight, WIDTH ** -0.5), (m.w_uk, R ** -0.5), (m.w_uv, R ** -0.5)) + (((m.uq.weight, q_rank ** -0.5), ) if q_rank else ()):
        p.data.copy_(torch.randn(p.shape, generator=g, device="cuda") * std)
    if sink:
        m.sink.data.copy_(torch.randn(heads, generator=g, device="cuda"))
    m.finalize()
    return m


def _batch(segments, block, seed=1):
    need = [(c + n + block - 1) // block for c, n in segments]
    order = torch.randperm(sum(need) + 3, generator=torch.Generator().manual_seed(seed)).tolist()
    tables, a = [], 0
    for k in need:
        tables.append(order[a:a + k])
        a += k
    return StepBatch.build([[1] * n for _, n in segments], [c for c, _ in segments], tables, list(range(len(segments))), block,
                           torch.device("cuda")), tables, len(order)


def _exact(m, h, cache, tables, block, segments):
    """The module in 64 bits over the cache its own launch has written."""
    H, x = m.heads, h.double() @ m.in_proj.weight.double().t()
    q = x[:, :m.splits[0]]
    if m.q_rank:
        q = q / torch.sqrt((q * q).mean(-1, keepdim=True) + m.eps) * m.q_norm.double()
        q = q @ m.uq.weight.double().t()
    q, gate = q.view(-1, H, D), x[:, m.splits[0] + R:]
    out, a = [], 0
    for (c, n), t in zip(segments, tables):
        rows = torch.tensor([t[i // block] * block + i % block for i in range(c + n)], device="cuda")
        lat = cache.view(-1, R)[rows].double()
        k = (lat @ m.w_uk.double().view(H * D, R).t()).view(-1, H, D).transpose(0, 1)
        v = torch.matmul(lat, m.w_uv.double())
        s = torch.matmul(q[a:a + n].transpose(0, 1), k.transpose(1, 2).contiguous()) * m.scale
        gap = torch.arange(c, c + n, device="cuda")[:, None] - torch.arange(c + n, device="cuda")[None]
        s = s.masked_fill((gap < 0) | ((gap >= m.window) if m.window else False), float("-inf"))
        if m.sink is not None:
            s = torch.cat([s, m.sink.double().view(H, 1, 1).expand(H, n, 1)], -1)
        p = torch.softmax(s, -1)[..., :c + n].contiguous()
        out.append(torch.matmul(p, v).transpose(0, 1).reshape(n, H * D))
        a += n
    o = torch.cat(out)
    if m.head_gate:
        return (o.view(-1, H, D) * torch.sigmoid(gate[:, :H])[:, :, None]).reshape(-1, H * D)
    return o * torch.sigmoid(gate[:, :H * D]) if m.gated else o


CASES = [(4, [(0, 32)], 16, {}), (4, [(0, 33), (0, 1), (0, 257)], 16, {}), (8, [(5, 130), (0, 7), (40, 61), (90, 1), (3, 1)], 16, {}),
         (6, [(0, 200), (64, 1)], 13, {}), (4, [(300, 140)], 8, {"window": 50}), (4, [(17, 129), (10, 1)], 32, {"gate": True, "sink": False}),
         (4, [(0, 65)], 16, {"gate": False, "q_rank": 64}), (16, [(1000, 400), (0, 2)], 64, {"window": 500, "q_rank": 64})]


@pytest.mark.parametrize("heads,segments,block,form", CASES)
def test_expanded(heads, segments, block, form, monkeypatch):
    m = _module(heads, **form)
    b, tables, pool = _batch(segments, block)
    h = torch.randn(b.num_tokens, WIDTH, generator=torch.Generator(device="cuda").manual_seed(2), device="cuda").to(torch.bfloat16)
    cache = torch.randn(pool, block, R, generator=torch.Generator(device="cuda").manual_seed(3), device="cuda").to(torch.bfloat16)
    rows = torch.tensor([b.num_tokens - 1, 3, 0], device="cuda")
    errors = []
    for pairs in (0.0, float("inf")):                          # every portion expanded, none
        monkeypatch.setattr(M, "LATENT_EXPAND_PAIRS", pairs)
        monkeypatch.setattr(M, "LATENT_EXPAND_WORK", 0)
        monkeypatch.setattr(M, "LATENT_EXPAND_ROWS", 1 if pairs == 0.0 else 1 << 40)
        assert (m.expanded_segments(b) > 0) == (pairs == 0.0)
        wide = torch.full((b.num_tokens, heads * D + 16), 7.0, dtype=torch.bfloat16, device="cuda")
        got = m.attend(h, cache, b, wide[:, 8:8 + heads * D])
        want = _exact(m, h, cache, tables, block, segments)
        errors.append(float((got.double() - want).norm() / want.norm()))
        assert bool((wide[:, :8] == 7).all()) and bool((wide[:, 8 + heads * D:] == 7).all())
        assert torch.equal(m.attend(h, cache, b), got)
        some = m.attend(h, cache, b, rows=rows)
        # (the product behind the latent attention sums in another order for three rows than for all)
        assert float((some.double() - got[rows].double()).norm()) <= 2.0 ** -8 * float(got[rows].double().norm())
    # projected rows, keys, probabilities, values, results and gated results are rounded to bf16 on either way, up to eight roundings of
    # 2^-9 / sqrt(3) in the mean and independent: 1.7 * 2^-9, and half as much again for what the exponentials make of the scores' share
    assert errors[0] <= 2.5 * 2.0 ** -9 and errors[0] <= 1.1 * errors[1]


def test_gathered_rows():
    segments, block = [(3, 14), (0, 16), (40, 1), (0, 1)], 8
    b, tables, pool = _batch(segments, block)
    cache = torch.randn(pool, block, R, device="cuda").to(torch.bfloat16)
    rows, own = mops.latent_gather(cache, b.block_tables, b.q_len, b.ctx_len, [c + n for c, n in segments])
    assert rows.shape[0] == 32 + 16 + 48 + 16
    for s, ((c, n), t) in enumerate(zip(segments, tables)):
        want = torch.stack([cache[t[i // block], i % block] for i in range(c + n)])
        got = torch.stack([rows[int(own[s, i // 16]) * 16 + i % 16] for i in range(c + n)])
        assert torch.equal(got, want)


def test_when_it_runs(monkeypatch):
    m = _module(4)
    assert m.expanded_segments(_batch([(0, 4100), (90, 1)], 16)[0]) == 1          # 6.5e9 of heads * kv_rank * pairs
    assert m.expanded_segments(_batch([(0, 3900), (90, 1)], 16)[0]) == 0          # 5.8e9
    monkeypatch.setattr(M, "LATENT_EXPAND_WORK", 0)
    assert m.expanded_segments(_batch([(0, 100), (90, 1)], 16)[0]) == 1
    assert m.expanded_segments(_batch([(0, 95)], 16)[0]) == 0                    # few rows
    assert m.expanded_segments(_batch([(2000, 100)], 16)[0]) == 0                 # few rows for the keys
    assert m.expanded_segments(_batch([(90, 1)] * 40, 16)[0]) == 0               # decoded rows
    m.w_uv.data = m.w_uv.data.float()
    assert m.expanded_segments(_batch([(0, 400)], 16)[0]) == 0
