"""The 128-wide prompt attention of the sequence mixers (csrc/mixers/biased_attention_fast.h, dba_prefill32_kernel): against a 64-bit
softmax over segments cut anywhere, head groupings, cache block sizes, masks, caps, sinks, gates, bias tables and strides."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
D = 128


def run(lens, ctxs, heads, kv_heads, block, bias=0, temp=0.0, window=0, chunk=0, softcap=0.0, sink=False, gate=None, pad=0, seed=0, fill=None, shift=0):
    from aphrodite_engine_amd import mixer_ops as mops
    g = torch.Generator(device=DEV).manual_seed(seed)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    T, n = sum(lens), len(lens)
    need = [(c + l + block - 1) // block for c, l in zip(ctxs, lens)]
    order = torch.randperm(sum(need) + 3, generator=g, device=DEV).to(torch.int32)
    tables = torch.zeros(n, max(need), dtype=torch.int32, device=DEV)
    at = 0
    for i, k in enumerate(need):
        tables[i, :k] = order[at:at + k]
        at += k
    size = len(order) * block * kv_heads * D
    kc, vc = (rnd(size + shift).bfloat16()[shift:].view(len(order), block, kv_heads, D) for _ in range(2))
    if fill is not None:                                     # what lies in blocks and slots that no key has
        used = torch.zeros(len(order), block, dtype=torch.bool, device=DEV)
        for i, k in enumerate(need):
            for j in range(k):
                used[tables[i, j].long(), :min(block, ctxs[i] + lens[i] - j * block)] = True
        kc[~used], vc[~used] = fill, fill
    q = rnd(T, heads * D + 8).bfloat16()[:, :heads * D]
    gt = None if gate is None else rnd(T, (heads * D if gate == "columns" else heads) + pad).bfloat16()[:, :heads * D if gate == "columns" else heads]
    lut = rnd(heads, bias).float() if bias else None
    sk = rnd(heads).float() if sink else None
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    starts = [sum(lens[:i]) for i in range(n)]
    out = torch.full((T, heads * D + pad), 7.0, device=DEV).bfloat16()
    seq_of = torch.repeat_interleave(torch.arange(n, device=DEV, dtype=torch.int32), i32(lens))
    mops.distance_bias_attention(out[:, :heads * D], q, gt, kc, vc, tables, i32(starts), i32(lens), i32(ctxs), seq_of, (min(lens), max(lens)), heads,
                                 D ** -0.5, lut, temp, 64, 0.5, max(c + l for c, l in zip(ctxs, lens)), window, chunk, softcap, sk)
    assert pad == 0 or bool((out[:, heads * D:] == 7.0).all())
    got = out[:, :heads * D].double().view(T, heads, D)
    worst = 0.0
    for i in range(n):
        total = ctxs[i] + lens[i]
        slot = torch.arange(total, device=DEV)
        blk = tables[i][slot // block].long()
        k, v = kc[blk, slot % block].double(), vc[blk, slot % block].double()
        k, v = (x.repeat_interleave(heads // kv_heads, 1).transpose(0, 1).contiguous() for x in (k, v))
        rows = slice(starts[i], starts[i] + lens[i])
        pos = ctxs[i] + torch.arange(lens[i], device=DEV)
        qq = q[rows].double().view(lens[i], heads, D).transpose(0, 1).contiguous()
        s = torch.matmul(qq, k.transpose(1, 2).contiguous()) * D ** -0.5
        if temp:
            s = s * (1 + temp * torch.log(((pos + 1) // 64 + 1).double()))[None, :, None]
        if softcap:
            s = softcap * torch.tanh(s / softcap)
        dist = pos[:, None] - slot[None, :]
        if bias:
            s = s + lut.double()[:, dist.clamp(0, bias - 1)]
        seen = dist >= 0
        if window:
            seen = seen & (dist < window)
        if chunk:
            seen = seen & (slot[None, :] >= pos[:, None] // chunk * chunk)
        s = s.masked_fill(~seen, float("-inf"))
        if sink:
            s = torch.cat([s, sk.double()[:, None, None].expand(heads, lens[i], 1)], 2)
        p = torch.softmax(s, -1)[..., :total]
        want = torch.matmul(p, v).transpose(0, 1) * 0.5
        if gate == "heads":
            want = want * torch.sigmoid(gt[rows].double())[..., None]
        elif gate == "columns":
            want = want * torch.sigmoid(gt[rows].double()).view(lens[i], heads, D)
        worst = max(worst, float((got[rows] - want).norm() / want.norm()))
    # probabilities and the result are rounded to bfloat16: an ulp's root mean square each, 2^-8 / sqrt(3)
    assert worst < 2 ** 0.5 * 2 ** -8 / 3 ** 0.5 * 1.15
    return out


GROUPS = [(8, 2), (4, 2), (3, 3), (16, 2), (32, 8), (6, 1)]


@pytest.mark.parametrize("heads,kv_heads", GROUPS)
@pytest.mark.parametrize("lens,ctxs", [([8], [0]), ([31], [5]), ([32], [64]), ([33, 64, 65], [0, 63, 100]), ([129, 8, 300], [70, 511, 0]), ([1025], [0])])
@pytest.mark.parametrize("block", [16, 8, 24, 128])
def test_plain(heads, kv_heads, lens, ctxs, block):
    run(lens, ctxs, heads, kv_heads, block, seed=sum(lens), fill=float("nan"))


@pytest.mark.parametrize("heads,kv_heads", GROUPS)
@pytest.mark.parametrize("kw", [dict(bias=1), dict(bias=50, temp=0.1), dict(bias=4096, gate="heads"), dict(window=1), dict(window=40, bias=64), dict(chunk=48),
                                dict(softcap=5.0, bias=16, sink=True), dict(window=100, chunk=64, sink=True, gate="columns"), dict(gate="columns"),
                                dict(gate="columns", pad=1), dict(softcap=2.0, window=64, gate="heads", pad=3)])
def test_forms(heads, kv_heads, kw):
    run([200, 9, 70], [33, 300, 0], heads, kv_heads, 16, seed=heads, **kw)


@pytest.mark.parametrize("kw", [dict(bias=64), dict(window=600, sink=True), dict(gate="columns", pad=1)])
@pytest.mark.parametrize("block,ctx", [(16, 8), (24, 700)])
def test_short_segments_beside_prompt_portions(kw, block, ctx):
    """Decoded rows and portions of up to 7 tokens before, among and behind prompt portions, more than 64 segments of them; with the longer
    contexts their key ranges are split."""
    lens = [2] + [1] * 70 + [90] + [3] * 5 + [40, 7, 1]
    run(lens, [i * 13 % 37 + ctx for i in range(len(lens))], 8, 2, block, fill=0.0, **kw)


@pytest.mark.parametrize("kw", [dict(), dict(bias=64, gate="heads"), dict(window=100, sink=True), dict(gate="columns", pad=1)])
@pytest.mark.parametrize("block", [16, 24])
def test_caches_that_are_not_16_byte_aligned(kw, block):
    """The older prompt kernel, which loads through registers, has these."""
    run([200, 9, 70], [33, 300, 0], 8, 2, block, fill=0.0, shift=4, **kw)


def test_a_row_s_bits_do_not_depend_on_the_batch():
    """A segment by itself and between others, its rows cut at the same places: workgroups are numbered and ordered otherwise, the sums are not."""
    from aphrodite_engine_amd import mixer_ops as mops
    heads, G, block, lens, ctxs = 8, 2, 16, [70, 257, 1, 400], [33, 90, 500, 0]
    g = torch.Generator(device=DEV).manual_seed(1)
    kc, vc = (torch.randn(128, block, G, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    q = torch.randn(sum(lens), heads * D, generator=g, device=DEV).bfloat16()
    lut = torch.randn(heads, 64, generator=g, device=DEV)
    tables = torch.randperm(128, generator=g, device=DEV).to(torch.int32)[:4 * 32].view(4, 32)

    def go(segs):
        rows = torch.cat([torch.arange(sum(lens[:s]), sum(lens[:s + 1]), device=DEV) for s in segs])
        n = [lens[s] for s in segs]
        i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
        out = torch.empty(len(rows), heads * D, device=DEV).bfloat16()
        mops.distance_bias_attention(out, q[rows], None, kc, vc, tables[segs].contiguous(), i32([sum(n[:i]) for i in range(len(n))]), i32(n),
                                     i32([ctxs[s] for s in segs]), torch.repeat_interleave(torch.arange(len(n), device=DEV, dtype=torch.int32), i32(n)),
                                     (min(n), max(n)), heads, D ** -0.5, lut, max_kv_len=501)
        at = sum(n[:segs.index(1)])
        return out[at:at + lens[1]]
    want = go([1])
    for segs in ([0, 1, 2, 3], [3, 1], [1, 2]):
        assert torch.equal(go(segs), want)
