"""Routed weights and the sum over a token's choices (moe_combine): every number of slabs that has a kernel of its own and others, odd numbers of choices,
rows at the edges of a workgroup's columns -- the same bits as the sums in the order that the operation states."""
import pytest
import torch

from aphrodite_engine_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("tokens,topk,nslab,n", [(1, 1, 1, 4), (3, 2, 2, 1020), (32, 2, 4, 4096), (5, 3, 3, 1028), (2, 5, 4, 2052), (17, 8, 7, 260),
                                                 (65, 3, 1, 1024), (300, 2, 2, 512), (9, 1, 7, 512), (9, 2, 6, 512), (9, 1, 5, 516), (40, 6, 2, 512), (7, 5, 1, 2052)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_combine(tokens, topk, nslab, n, dtype):
    g = torch.Generator(device=DEV).manual_seed(tokens * n + nslab)
    rows = tokens * topk + 7
    slabs = torch.randn(nslab, rows, n, generator=g, device=DEV)
    inv = torch.randperm(rows, generator=g, device=DEV)[:tokens * topk].int()
    w = torch.rand(tokens, topk, generator=g, device=DEV)
    y = slabs[0]
    for s in range(1, nslab):
        y = y + slabs[s]
    acc = torch.zeros(tokens, n, device=DEV)
    for k in range(topk):
        acc = acc + (y[inv.view(tokens, topk)[:, k].long()] * w[:, k:k + 1]).to(dtype).float()
    assert torch.equal(ops.moe_combine(slabs, inv, w, dtype), acc.to(dtype))


def test_rows_of_more_workgroups_than_16_bits_count():
    n = 4 * 256 * 65536 + 4
    slabs = torch.arange(n, dtype=torch.float32, device=DEV).remainder_(2048).view(1, 1, n)
    out = ops.moe_combine(slabs, torch.zeros(1, dtype=torch.int32, device=DEV), torch.ones(1, 1, device=DEV), torch.float16)
    assert torch.equal(out, slabs[0].half())
