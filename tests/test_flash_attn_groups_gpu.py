"""Prompt attention on 32 x 32 tiles at the edges of what its launch chooses: one group of waves a row tile and two that take the key tiles in turn, exact and
deferred maxima, prompts behind cached keys, rows so far apart that 32-bit offsets do not reach -- against attention in 64 bits."""
import pytest
import torch

from aphrodite_engine_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu
DEV, D = "cuda", 128


def _check(out, q, k, v, cu, scale, causal, slopes, dtype, cached=0):
    heads, rep = q.shape[1], q.shape[1] // k.shape[1]
    for a, b in zip(cu[:-1], cu[1:]):
        n = b - a
        kk, vv = (x[a:b + cached].double().repeat_interleave(rep, 1).transpose(0, 1) for x in (k, v))
        s = torch.matmul(q[a:b].double().transpose(0, 1), kk.transpose(1, 2).contiguous()) * scale
        i, j = torch.arange(cached, cached + n, device=DEV)[:, None], torch.arange(cached + n, device=DEV)[None]
        if slopes is not None:
            s = s + slopes.double()[:, None, None] * (j - i)
        if causal:
            s = s.masked_fill(j > i, float("-inf"))
        want = torch.matmul(torch.softmax(s, 2), vv).transpose(0, 1)
        # probabilities and results are rounded to the type: u of a value each, the probabilities' against values of up to the largest
        u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
        err = (out[a:b].double() - want).abs()
        assert (err <= 2 * u * (want.abs() + vv.abs().max() / 2)).all()
        assert float(err.norm() / want.norm()) < 1.2 * u


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads,kv,lens,causal,alibi,first", [
    (8, 2, [256], True, False, 4096), (8, 2, [257, 65], True, False, 4096), (32, 8, [1024], True, False, 4096), (32, 8, [2048], True, False, 4096),
    (32, 8, [2080], True, False, 4096), (6, 3, [321], False, False, 4096), (3, 3, [449, 1], True, True, 4096), (8, 2, [1100, 40, 700], True, False, 1024),
    (32, 8, [1500], True, True, 1024), (4, 4, [1090], False, False, 1024), (32, 8, [1200, 1300, 64], True, False, 1024),
    (8, 2, [1057, 31, 32, 33], True, False, 1024), (8, 2, [1057, 31, 32, 33], False, False, 1024), (4, 4, [1089, 127, 128, 129], True, False, 1024),
    (6, 3, [1025, 63, 64, 65, 1], True, False, 1024), (6, 3, [1025, 63, 64, 65, 1], False, True, 1024)])
def test_forms(heads, kv, lens, causal, alibi, first, dtype):
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + heads)
    t = sum(lens)
    qkv = torch.randn(t, (heads + 2 * kv) * D, generator=g, device=DEV).to(dtype)
    q, k, v = (x.view(t, -1, D) for x in qkv.split([heads * D, kv * D, kv * D], 1))
    cu = [sum(lens[:i]) for i in range(len(lens) + 1)]
    slopes = torch.rand(heads, generator=g, device=DEV) * 0.05 if alibi else None
    with ops.knob("APHRO_FA_V4_MIN_KEYS", first):
        out = ops.flash_attn_varlen(q, k, v, torch.tensor(cu, dtype=torch.int32, device=DEV), max(lens), D ** -0.5, causal=causal, alibi_slopes=slopes)
    _check(out, q, k, v, cu, D ** -0.5, causal, slopes, dtype)


@pytest.mark.parametrize("heads,kv,rows,cached,first", [
    (32, 8, 1300, 650, 4096), (32, 8, 1300, 1300, 4096), (32, 8, 1030, 686, 1024), (32, 8, 1030, 687, 1024), (32, 8, 300, 2000, 4096), (8, 8, 400, 79, 4096),
    (8, 1, 3000, 6001, 4096), (4, 4, 1033, 8000, 4096)])
def test_behind_cached_keys(heads, kv, rows, cached, first):
    """One prompt behind cached keys, on both sides of where its chains count as uneven."""
    g = torch.Generator(device=DEV).manual_seed(rows + cached)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV).bfloat16()
    q, k, v, bs = rnd(rows, heads, D), rnd(cached + rows, kv, D), rnd(cached + rows, kv, D), 16
    blocks = (cached + bs - 1) // bs
    order = torch.randperm(blocks + 1, generator=g, device=DEV)
    kc, vc = torch.full((blocks + 1, kv, D // 8, bs, 8), float("nan"), device=DEV).bfloat16(), torch.full((blocks + 1, kv, D, bs), float("nan"), device=DEV).bfloat16()
    at, off = order[torch.arange(cached, device=DEV) // bs], torch.arange(cached, device=DEV) % bs
    kc[at, :, :, off], vc[at, :, :, off] = k[:cached].view(cached, kv, D // 8, 8), v[:cached]
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    out = torch.empty_like(q)
    with ops.knob("APHRO_FA_V4_MIN_KEYS", first):
        ops.context_attention_fwd(q, k[cached:], v[cached:], out, "auto", kc, vc, order[None, :blocks].int().contiguous(), i32([0, rows]), i32([cached + rows]),
                                  i32([cached]), rows, max_seq_len=cached + rows, total_kv_tokens=cached + rows)
    _check(out, q, k, v, [0, rows], D ** -0.5, True, None, torch.bfloat16, cached)


@pytest.mark.parametrize("first", [1024, 4096])
def test_rows_far_apart(first):
    """A key every 2 MB: 1100 of them do not lie within 32-bit offsets of the first."""
    g = torch.Generator(device=DEV).manual_seed(first)
    n, stride = 1100, 1 << 20
    room = torch.empty(n * stride, dtype=torch.bfloat16, device=DEV)
    qkv = room.view(n, stride)[:, :6 * D]
    qkv.copy_(torch.randn(n, 6 * D, generator=g, device=DEV))
    q, k, v = (x.view(n, -1, D) for x in (qkv[:, :4 * D], qkv[:, 4 * D:5 * D], qkv[:, 5 * D:]))
    with ops.knob("APHRO_FA_V4_MIN_KEYS", first):
        out = ops.flash_attn_varlen(q, k, v, torch.tensor([0, n], dtype=torch.int32, device=DEV), n, D ** -0.5)
    _check(out, q, k, v, [0, n], D ** -0.5, True, None, torch.bfloat16)


def test_maxima_that_jump():
    """Keys far above all before them, in either group's tiles and at the diagonal, with deferred maxima and exact ones."""
    g = torch.Generator(device=DEV).manual_seed(1)
    n, heads, kv = 1500, 8, 2
    q, k, v = (torch.randn(n, h, D, generator=g, device=DEV) for h in (heads, kv, kv))
    for pos, gain in ((130, 8.0), (700, 6.0), (701, 14.0), (1100, 12.0), (1400, 20.0)):
        k[pos] = q.view(n, kv, heads // kv, D)[:, :, 0].mean(0) * gain + k[pos] * 0.1
    q, k, v = q.half(), k.half(), v.half()
    for first in (1024, 4096):
        with ops.knob("APHRO_FA_V4_MIN_KEYS", first):
            out = ops.flash_attn_varlen(q, k, v, torch.tensor([0, n], dtype=torch.int32, device=DEV), n, 0.3)
        _check(out, q, k, v, [0, n], 0.3, True, None, torch.float16)
