"""The expert tile GEMM at the edges of its 32-row pieces, of the groups it holds at a time and of quantisation groups longer than its step: against the
experts' products in 64 bits and the decode-sized path, rows aligned in blocks of 64 and of 128."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _experts(e, hidden, inter, group, seed):
    from aphrodite_engine_amd.moe import Wna16Experts
    g = torch.Generator(device=DEV).manual_seed(seed)

    def one(k, n):
        w = [torch.randint(-2 ** 31, 2 ** 31 - 1, s, generator=g, device=DEV, dtype=torch.int64).to(torch.int32) for s in ((k // 8, n), (k // group, n // 8))]
        return w[0], w[1], ((torch.rand(k // group, n, generator=g, device=DEV) * 0.5 + 0.75) / (6.7 * k ** 0.5)).half()
    a, b = [one(hidden, 2 * inter) for _ in range(e)], [one(inter, hidden) for _ in range(e)]
    return Wna16Experts(a, b, zero_offset=1, layout="gptq"), a, b


def _dense(t, group):
    qw, qz, sc = t
    q = torch.stack([(qw >> (4 * i)) & 15 for i in range(8)], 1).flatten(0, 1)
    z = torch.stack([(qz >> (4 * i)) & 15 for i in range(8)], 2).flatten(1, 2) + 1
    rows = torch.arange(q.shape[0], device=DEV) // group
    return (q - z[rows]).double() * sc.double()[rows]


@pytest.mark.parametrize("block", [64, 128])
@pytest.mark.parametrize("counts,hidden,inter,group", [
    ((1, 31, 32, 33), 512, 512, 128), ((64, 65, 96, 97, 0, 63), 512, 768, 128), ((128, 0, 129, 160, 191), 768, 512, 128),
    ((40, 70, 5), 1024, 512, 256), ((100, 33), 12544, 512, 128), ((20, 120), 512, 12416, 128)])
def test_pieces_of_a_tile(monkeypatch, counts, hidden, inter, group, block):
    from aphrodite_engine_amd import moe as M
    e = len(counts)
    experts, a, b = _experts(e, hidden, inter, group, sum(counts))
    tokens = sum(counts)
    g = torch.Generator(device=DEV).manual_seed(tokens)
    ids = torch.repeat_interleave(torch.arange(e, device=DEV), torch.tensor(counts, device=DEV))[torch.randperm(tokens, generator=g, device=DEV)]
    x = torch.randn(tokens, hidden, generator=g, device=DEV).half()
    logits, w = torch.zeros(tokens, e, device=DEV).half(), torch.rand(tokens, 1, generator=g, device=DEV) + 0.5
    run = lambda: M.fused_wna16_moe(x, experts, logits, 1, True, w, ids[:, None].to(torch.int32))
    monkeypatch.setattr(M, "moe_tile_align", lambda *_: block)
    got = run()
    monkeypatch.setattr(M, "moe_tile_align", lambda *_: 0)
    small = run() if all(M.ops.wna16_grouped_ksplit(tokens + 16 * e, n, k, k // group) > 0 for k, n in ((hidden, 2 * inter), (inter, hidden))) else None
    want = torch.zeros(tokens, hidden, dtype=torch.float64, device=DEV)
    for i in range(e):
        rows = ids == i
        gate, up = (x[rows].double() @ _dense(a[i], group)).chunk(2, -1)
        want[rows] = (torch.nn.functional.silu(gate) * up) @ _dense(b[i], group) * w[rows].double()

    def off(y):
        return float((y.double() - want).norm() / want.norm())
    # gate, up, silu, activation and the weighted result are rounded to 16 bits on the way: a few half-ulps; no worse than the decode path
    assert off(got) < 1.5e-3 and (small is None or off(got) < 1.05 * off(small) + 1e-6)


def test_which_batches_are_aligned_how():
    from types import SimpleNamespace
    from aphrodite_engine_amd import moe as M
    w = lambda k, n: tuple(torch.empty(8, r, c, dtype=t, device="meta") for r, c, t in
                           ((k // 8, n, torch.int32), (k // 128, n // 8, torch.int32), (k // 128, n, torch.float16)))
    experts = SimpleNamespace(num_experts=8, hidden=4096, inter=14336, w13=w(4096, 28672), w2=w(14336, 4096))
    align = lambda slots: M.moe_tile_align(slots, experts, torch.float16)
    assert [align(s) for s in (127, 128, 479, 480, 8192)] == [0, 64, 64, 128, 128]


def test_batches_that_only_blocks_of_64_serve():
    """128 groups in front of the activation: blocks of 128 rows hold 102, and the largest batches of such experts take those of 64."""
    from types import SimpleNamespace
    from aphrodite_engine_amd import moe as M
    w = lambda k, n: tuple(torch.empty(8, r, c, dtype=t, device="meta") for r, c, t in
                           ((k // 8, n, torch.int32), (k // 128, n // 8, torch.int32), (k // 128, n, torch.float16)))
    experts = SimpleNamespace(num_experts=8, hidden=16384, inter=4096, w13=w(16384, 8192), w2=w(4096, 16384))
    align = lambda slots: M.moe_tile_align(slots, experts, torch.float16)
    assert [align(s) for s in (127, 128, 480, 767 * 8, 768 * 8, 20000)] == [0, 64, 64, 64, 64, 64]

    experts, a, b = _experts(2, 16384, 512, 128, 0)
    g = torch.Generator(device=DEV).manual_seed(0)
    tokens, ids = 1600, torch.randint(0, 2, (1600,), generator=g, device=DEV)
    assert M.moe_tile_align(tokens, experts, torch.float16) == 64
    x = torch.randn(tokens, 16384, generator=g, device=DEV).half()
    logits, weight = torch.zeros(tokens, 2, device=DEV).half(), torch.rand(tokens, 1, generator=g, device=DEV) + 0.5
    got = M.fused_wna16_moe(x, experts, logits, 1, True, weight, ids[:, None].to(torch.int32))
    want = torch.zeros(tokens, 16384, dtype=torch.float64, device=DEV)
    for i in range(2):
        rows = ids == i
        gate, up = (x[rows].double() @ _dense(a[i], 128)).chunk(2, -1)
        want[rows] = (torch.nn.functional.silu(gate) * up) @ _dense(b[i], 128) * weight[rows].double()
    assert float((got.double() - want).norm() / want.norm()) < 1.5e-3        # (as above)
