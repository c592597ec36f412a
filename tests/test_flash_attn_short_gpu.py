"""Prompt attention over rows of 128 below 4096 keys (csrc/flash_attn_short.hip): against a 64-bit softmax at lengths around its 32-row and
64-key tiles, for head groupings, both types, strided rows, with and without the causal mask, behind cached contexts; and ALiBi and what it leaves to the
other kernels (windows)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, D = "cuda", 128
LENS = [[1], [31], [32], [33], [63, 64, 65], [127, 1, 300], [129, 511], [1000, 2], [2111, 65]]


def reference(q, k, v, heads, kv_heads, causal, off=0, slopes=None, window=0):
    n, m = q.shape[0], k.shape[0]
    q, k, v = (x.double().view(x.shape[0], -1, D).transpose(0, 1).contiguous() for x in (q, k, v))
    k, v = (x.repeat_interleave(heads // kv_heads, 0) for x in (k, v))
    dist = torch.arange(n, device=DEV)[:, None] + off - torch.arange(m, device=DEV)[None]
    s = torch.matmul(q, k.transpose(1, 2).contiguous()) * D ** -0.5
    if slopes is not None:
        s = s - slopes.double()[:, None, None] * dist
    seen = (dist >= 0) if causal else torch.ones_like(dist, dtype=torch.bool)
    if window:
        seen = seen & (dist < window)
    return torch.matmul(torch.softmax(s.masked_fill(~seen, float("-inf")), -1), v).transpose(0, 1)


def bound(dtype):
    # probabilities and the result are rounded: an ulp's root mean square each
    return 2 ** 0.5 * (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8) / 3 ** 0.5 * 1.15


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads,kv_heads", [(8, 2), (4, 2), (3, 3), (32, 8), (6, 1)])
@pytest.mark.parametrize("lens", LENS)
@pytest.mark.parametrize("causal", [True, False])
def test_lengths(dtype, heads, kv_heads, lens, causal):
    from aphrodite_engine_amd import _custom_ops as ops
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + heads)
    T = sum(lens)
    qkv = torch.randn(T, (heads + 2 * kv_heads) * D + 8, generator=g, device=DEV).to(dtype)
    q, k, v = qkv[:, :-8].split([heads * D, kv_heads * D, kv_heads * D], -1)
    starts = [sum(lens[:i]) for i in range(len(lens) + 1)]
    out = ops.flash_attn_varlen(q.view(T, heads, D), k.view(T, kv_heads, D), v.view(T, kv_heads, D),
                                torch.tensor(starts, dtype=torch.int32, device=DEV), max(lens), D ** -0.5, causal=causal)
    for a, b in zip(starts, starts[1:]):
        want = reference(q[a:b], k[a:b], v[a:b], heads, kv_heads, causal)
        assert float((out[a:b].double() - want).norm() / want.norm()) < bound(dtype)


@pytest.mark.parametrize("kw", [dict(alibi=True), dict(window=40), dict()])
@pytest.mark.parametrize("lens", [[70, 33], [300], [1090]])
def test_forms_beside_it(kw, lens):
    from aphrodite_engine_amd import _custom_ops as ops
    heads, kv_heads, T = 8, 2, sum(lens)
    g = torch.Generator(device=DEV).manual_seed(3)
    q, k, v = (torch.randn(T, n * D, generator=g, device=DEV).half() for n in (heads, kv_heads, kv_heads))
    slopes = torch.rand(heads, generator=g, device=DEV) if kw.get("alibi") else None
    starts = [sum(lens[:i]) for i in range(len(lens) + 1)]
    w = kw.get("window", 0)
    out = ops.flash_attn_varlen(q.view(T, heads, D), k.view(T, kv_heads, D), v.view(T, kv_heads, D),
                                torch.tensor(starts, dtype=torch.int32, device=DEV), max(lens), D ** -0.5, causal=True, alibi_slopes=slopes,
                                window_size=(w - 1, 0) if w else (-1, -1))
    for a, b in zip(starts, starts[1:]):
        want = reference(q[a:b], k[a:b], v[a:b], heads, kv_heads, True, 0, slopes, w)
        assert float((out[a:b].double() - want).norm() / want.norm()) < bound(torch.float16)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("ctxs,lens", [([0, 5, 300], [40, 1, 100]), ([63, 64], [65, 200]), ([700], [17]), ([1500, 3], [100, 40])])
def test_behind_cached_contexts(dtype, ctxs, lens):
    from aphrodite_engine_amd import _custom_ops as ops
    heads, kv_heads, block, T = 8, 2, 16, sum(lens)
    g = torch.Generator(device=DEV).manual_seed(7)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    q, k, v = rnd(T, heads, D), rnd(T, kv_heads, D), rnd(T, kv_heads, D)
    need = [(c + n + block - 1) // block for c, n in zip(ctxs, lens)]
    tables = torch.zeros(len(lens), max(need), dtype=torch.int32, device=DEV)
    order, at = torch.randperm(sum(need) + 2, generator=g, device=DEV).int(), 0
    for i, m in enumerate(need):
        tables[i, :m] = order[at:at + m]
        at += m
    kc, vc = rnd(len(order), kv_heads, D // 8, block, 8), rnd(len(order), kv_heads, D, block)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    starts = [sum(lens[:i]) for i in range(len(lens) + 1)]
    out = torch.empty_like(q)
    ops.context_attention_fwd(q, k, v, out, "auto", kc, vc, tables, i32(starts), i32([c + n for c, n in zip(ctxs, lens)]), i32(ctxs), max(lens))
    for i, (c, n) in enumerate(zip(ctxs, lens)):
        slot = torch.arange(c, device=DEV)
        blk = tables[i][slot // block].long()
        keys = torch.cat([kc.permute(0, 3, 1, 2, 4).reshape(len(order), block, kv_heads, D)[blk, slot % block], k[starts[i]:starts[i] + n]])
        vals = torch.cat([vc.permute(0, 3, 1, 2)[blk, slot % block], v[starts[i]:starts[i] + n]])
        want = reference(q[starts[i]:starts[i] + n].reshape(n, -1), keys.reshape(c + n, -1), vals.reshape(c + n, -1), heads, kv_heads, True, c)
        got = out[starts[i]:starts[i] + n].double()
        assert float((got - want).norm() / want.norm()) < bound(dtype)
