"""Prompt attention of 128-wide rows by one group of waves a row tile and by two that take its key tiles in turn: numbers of key tiles from one up, odd and
even, behind cached keys, under windows and chunks, with every operand of the score -- against attention in 64 bits."""
import pytest
import torch

from aphrodite_engine_amd import mixer_ops as mo

pytestmark = pytest.mark.gpu
DEV, D = "cuda", 128

# (query heads, kv heads, [(cached keys, rows)], block size, what else)
CASES = [
    (4, 1, [(0, 256)], 16, {}), (4, 1, [(0, 257)], 16, dict(bias=True)), (8, 2, [(65, 320)], 32, dict(bias=True, softcap=20.0)),
    (16, 4, [(700, 33)], 16, dict(window=300)), (16, 4, [(0, 700)], 16, dict(window=130, sink=True)), (6, 3, [(0, 449)], 16, dict(gate=1)),
    (3, 3, [(129, 513)], 64, dict(gate=2)), (8, 2, [(0, 1000), (300, 9), (250, 1)], 16, dict(bias=True)), (16, 4, [(0, 640)], 16, dict(chunk=192)),
    (16, 4, [(10, 300)], 8, {}), (16, 4, [(0, 2100)], 16, dict(bias=True)), (32, 8, [(0, 2100)], 16, {}), (32, 8, [(0, 700)] * 4, 16, dict(gate=2)),
    (16, 4, [(40, 200)], 16, dict(bias=True)), (32, 8, [(2200, 1100)], 16, dict(bias=True)), (32, 8, [(5000, 1100)], 16, {}), (32, 8, [(0, 1100)], 16, dict(window=300)),
    (32, 8, [(0, 1100)], 16, dict(window=400)), (32, 8, [(100, 1100), (3000, 1)], 16, {})]


@pytest.mark.parametrize("heads,kv_heads,segs,bs,kw", CASES)
def test_against_64_bits(heads, kv_heads, segs, bs, kw):
    g = torch.Generator(device=DEV).manual_seed(heads * 1000 + sum(q for _, q in segs))
    rows = sum(q for _, q in segs)
    blocks = [(c + q + bs - 1) // bs for c, q in segs]
    q = torch.randn(rows, heads * D, generator=g, device=DEV).bfloat16()
    kc, vc = (torch.randn(sum(blocks) + 1, bs, kv_heads, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    order = torch.randperm(sum(blocks), generator=g, device=DEV).int()
    vc[-1] = float("nan")
    table = torch.full((len(segs), max(blocks)), sum(blocks), dtype=torch.int32, device=DEV)       # (what is no segment's lies in a page of NaN)
    at = 0
    for i, n in enumerate(blocks):
        table[i, :n] = order[at:at + n]
        at += n
    for i, (c, n) in enumerate(segs):                                       # rows past a segment's end, too
        tail = (c + n) % bs
        if tail:
            vc[table[i, blocks[i] - 1].long(), tail:] = float("nan")
    window, chunk, softcap = kw.get("window", 0), kw.get("chunk", 0), kw.get("softcap", 0.0)
    lut = torch.randn(heads, 300, generator=g, device=DEV) if kw.get("bias") else None
    sink = torch.randn(heads, generator=g, device=DEV) if kw.get("sink") else None
    gate = torch.randn(rows, heads * (D if kw["gate"] == 2 else 1), generator=g, device=DEV).bfloat16() if kw.get("gate") else None
    ql, cl = [n for _, n in segs], [c for c, _ in segs]
    start = [sum(ql[:i]) for i in range(len(ql))]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    out = torch.full((rows, heads * D), float("nan"), device=DEV, dtype=torch.bfloat16)
    mo.distance_bias_attention(out, q, gate, kc, vc, table, i32(start), i32(ql), i32(cl), torch.repeat_interleave(i32(list(range(len(ql)))), i32(ql).long()).int(),
                               (min(ql), max(ql)), heads, D ** -0.5, lut, max_kv_len=max(c + n for c, n in segs), window=window, chunk=chunk, softcap=softcap, sink=sink)
    for i, (c, n) in enumerate(segs):
        r = slice(start[i], start[i] + n)
        k, v = (x[table[i, :blocks[i]].long()].reshape(-1, kv_heads, D)[:c + n].double().repeat_interleave(heads // kv_heads, 1).transpose(0, 1) for x in (kc, vc))
        s = torch.matmul(q[r].double().view(n, heads, D).transpose(0, 1), k.transpose(1, 2).contiguous()) * D ** -0.5
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        pos, key = torch.arange(c, c + n, device=DEV)[:, None], torch.arange(c + n, device=DEV)[None]
        if lut is not None:
            s = s + lut.double()[:, (pos - key).clamp(0, lut.shape[1] - 1)]
        seen = key <= pos
        if window:
            seen &= key > pos - window
        if chunk:
            seen &= key // chunk == pos // chunk
        s = s.masked_fill(~seen, float("-inf"))
        if sink is not None:
            s = torch.cat([s, sink.double()[:, None, None].expand(heads, n, 1)], 2)
        p = torch.softmax(s, 2)[..., :c + n]
        want = torch.matmul(p, v).transpose(0, 1).reshape(n, heads, D)
        if gate is not None:
            want = want * torch.sigmoid(gate[r].double().view(n, heads, -1))
        # probabilities and results are bf16: 2^-9 of a value each, the probabilities' against values of up to the largest; products of 128 in fp32
        err, top = (out[r].double().view(n, heads, D) - want).abs(), v.abs().max()
        assert (err <= 2.0 ** -8 * (want.abs() + 2.0 ** -1 * top)).all(), float((err / (want.abs() + 0.5 * top)).max())
        assert float(err.norm() / want.norm()) < 6e-3
