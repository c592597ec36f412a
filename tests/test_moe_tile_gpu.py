"""The prompt-sized expert GEMM (csrc/wna16_moe_tile.hip) and its routing: against the experts' products in 64 bits and against the decode-sized
path, at block edges, with experts that no token chose, both block sizes, K slices, both 16-bit types."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def experts_of(e, hidden, inter, dtype, layout, seed):
    from aphrodite_engine_amd.moe import Wna16Experts
    g = torch.Generator(device=DEV).manual_seed(seed)

    def words(*shape):
        return torch.randint(-2 ** 31, 2 ** 31 - 1, shape, generator=g, device=DEV, dtype=torch.int64).to(torch.int32)

    def one(k, n):
        qw = words(k // 8, n) if layout == "gptq" else words(k, n // 8)
        sc = (torch.rand(k // 128, n, generator=g, device=DEV) * 0.5 + 0.75) / (6.7 * k ** 0.5)
        return qw, words(k // 128, n // 8), sc.to(dtype)
    a, b = [one(hidden, 2 * inter) for _ in range(e)], [one(inter, hidden) for _ in range(e)]
    return Wna16Experts(a, b, zero_offset=1 if layout == "gptq" else 0, layout=layout), a, b


def dense(t, layout):
    qw, qz, sc = t
    order = range(8) if layout == "gptq" else (0, 4, 1, 5, 2, 6, 3, 7)

    def nib(w, dim, o):
        return torch.stack([(w >> (4 * i)) & 15 for i in o], dim + 1).flatten(dim, dim + 1)
    q = nib(qw, 0, range(8)) if layout == "gptq" else nib(qw, 1, order)
    z = nib(qz, 1, order) + (1 if layout == "gptq" else 0)
    rows = torch.arange(q.shape[0], device=DEV) // 128
    return (q - z[rows]).double() * sc.double()[rows]


@pytest.mark.parametrize("dtype,layout", [(torch.float16, "gptq"), (torch.float16, "awq"), (torch.bfloat16, "gptq")])
@pytest.mark.parametrize("tokens,e,topk,hidden,inter", [(150, 8, 2, 512, 1024), (700, 8, 2, 512, 512), (257, 4, 1, 1024, 512), (331, 16, 3, 512, 1536)])
@pytest.mark.parametrize("block", [64, 128])
def test_tile_experts(monkeypatch, dtype, layout, tokens, e, topk, hidden, inter, block):
    from aphrodite_engine_amd import moe as M
    experts, a, b = experts_of(e, hidden, inter, dtype, layout, tokens + e)
    g = torch.Generator(device=DEV).manual_seed(tokens)
    x = torch.randn(tokens, hidden + 8, generator=g, device=DEV).to(dtype)[:, :hidden]
    logits = torch.randn(tokens, e, generator=g, device=DEV).to(dtype)
    logits[:, e - 1] = -30.0                             # an expert without a token
    logits[: tokens // 2, 0] += 6.0                      # ... and one with many
    monkeypatch.setattr(M, "MOE_TILE_ROWS", 1)
    monkeypatch.setattr(M, "MOE_TILE_WIDE", 0 if block == 128 else 1 << 30)
    assert M.moe_tile_block(tokens * topk, experts, dtype) == block
    got = M.fused_wna16_moe(x, experts, logits, topk, True)
    deferred = M.fused_wna16_moe(x, experts, logits, topk, True, defer_combine=True)
    assert torch.equal(deferred.combine(), got)
    monkeypatch.setattr(M, "MOE_TILE_ROWS", 1 << 30)
    small = M.fused_wna16_moe(x, experts, logits, topk, True)
    p = torch.softmax(logits.double(), -1)
    w, ids = p.topk(topk, -1)
    w = w / w.sum(-1, keepdim=True)
    want = torch.zeros(tokens, hidden, dtype=torch.float64, device=DEV)
    for i in range(e):
        row, place = torch.where(ids == i)
        if row.numel():
            gate, up = (x[row].double() @ dense(a[i], layout)).chunk(2, -1)
            want[row] += (torch.nn.functional.silu(gate) * up) @ dense(b[i], layout) * w[row, place][:, None]

    def off(y):
        return float((y.double() - want).norm() / want.norm())
    # gate, up, silu, activation and the weighted result are rounded to 16 bits on the way: a few half-ulps; no worse than the decode path
    assert off(got) < (1.5e-3 if dtype == torch.float16 else 1.2e-2)
    assert off(got) < 1.05 * off(small) + 1e-6


@pytest.mark.parametrize("tokens,e,topk,block", [(1, 8, 2, 64), (255, 8, 2, 128), (256, 16, 8, 64), (257, 3, 3, 128), (2047, 8, 2, 128)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
def test_route_align_blocks_is_route_align(tokens, e, topk, block, dtype):
    from aphrodite_engine_amd import _custom_ops as ops
    g = torch.Generator(device=DEV).manual_seed(tokens * e)
    logits = (torch.randn(tokens, e + 1, generator=g, device=DEV) * 2).round().to(dtype)[:, 1:]      # (ties among them)
    for renorm in (True, False):
        a = ops.moe_route_align_blocks(logits, topk, renorm, e, block)
        b = ops.moe_route_align(logits, topk, renorm, e, block, True)
        for x, y in zip(a, b):
            assert torch.equal(x, y)


@pytest.mark.parametrize("e,topk,block", [(8, 2, 64), (16, 8, 128), (3, 3, 64)])
def test_routing_places_every_slot_of_rows_that_are_not_finite(e, topk, block):
    """A row with a NaN, a +inf, or of -inf only names expert 0 with every choice: in several waves and workgroups, first and last."""
    from aphrodite_engine_amd import _custom_ops as ops
    tokens = 700
    logits = torch.randn(tokens, e, device=DEV)
    for i, t in enumerate((0, 1, 63, 64, 100, 255, 256, 400, 401, 699)):
        logits[t] = (float("nan"), -float("inf"))[i % 2]
        if i % 3 == 0:
            logits[t] = 0.5
            logits[t, i % e] = (float("inf"), float("nan"))[i % 2]
    a = ops.moe_route_align_blocks(logits, topk, True, e, block)
    b = ops.moe_route_align(logits, topk, True, e, block, True)
    for x, y in zip(a, b):
        assert torch.equal(x.nan_to_num(-1.0), y.nan_to_num(-1.0))
    order = a[2][: int(a[4])].tolist()
    assert sorted(i for i in order if i < tokens * topk) == list(range(tokens * topk))
    assert all(order[p] == i for i, p in enumerate(a[5].tolist()))


def test_a_token_without_a_finite_logit_leaves_the_others(monkeypatch):
    """The prompt-sized experts with such tokens in the batch: everyone else's output is what it is without them."""
    from aphrodite_engine_amd import moe as M
    experts, _, _ = experts_of(8, 512, 512, torch.float16, "gptq", 11)
    monkeypatch.setattr(M, "MOE_TILE_ROWS", 1)
    x, logits = torch.randn(300, 512, device=DEV).half(), torch.randn(300, 8, device=DEV).half()
    want = M.fused_wna16_moe(x, experts, logits, 2, True)
    assert M.moe_tile_block(600, experts, torch.float16)
    logits[17], logits[64, 5], logits[299] = float("nan"), float("inf"), -float("inf")
    got = M.fused_wna16_moe(x, experts, logits, 2, True)
    rest = [t for t in range(300) if t not in (17, 64, 299)]
    assert torch.equal(got[rest], want[rest])


def test_route_align_blocks_many_tokens():
    """More slots than the one-workgroup form holds: against the separate ops."""
    from aphrodite_engine_amd import _custom_ops as ops
    from aphrodite_engine_amd import moe as M
    logits = torch.randn(9001, 8, device=DEV)
    w, ids, s, x, n, inv = ops.moe_route_align_blocks(logits, 2, True, 8, 128)
    w2, ids2 = M.fused_topk(logits, logits, 2, True)
    s2, x2, n2, inv2 = M.moe_align_block_size(ids2, 128, 8, want_inverse=True)
    assert torch.equal(ids, ids2) and torch.equal(s, s2) and torch.equal(x, x2) and torch.equal(n, n2) and torch.equal(inv, inv2)
    assert torch.allclose(w, w2, rtol=1e-6)
