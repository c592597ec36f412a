"""What bench.py puts in the place of the framework's own functions takes their arguments."""
import inspect

import torch

import bench
from aphrodite_engine_amd import _custom_ops as ops


def test_library_attention_stands_in_for_the_prompt_kernel():
    ours, theirs = (inspect.signature(f).parameters for f in (ops.flash_attn_varlen, bench.sdpa_varlen))
    assert list(ours) == list(theirs) and all(ours[n].default == theirs[n].default for n in ours)
    g = torch.Generator().manual_seed(0)
    q, k, v = (torch.randn(9, h, 16, generator=g) for h in (4, 2, 2))
    cu = torch.tensor([0, 9], dtype=torch.int32)
    want = bench.sdpa_varlen(q, k, v, cu, 9, 0.25)
    s = torch.einsum("qhd,khd->hqk", q.double(), k.double().repeat_interleave(2, 1)) * 0.25
    s.masked_fill_(torch.ones(9, 9).triu(1).bool(), -torch.inf)
    exact = torch.einsum("hqk,khd->qhd", s.softmax(-1), v.double().repeat_interleave(2, 1))
    assert want.shape == q.shape and torch.allclose(want.double(), exact, atol=1e-5)
    out = torch.full((12, 4, 16), torch.nan)
    assert bench.sdpa_varlen(q, k, v, cu, 9, 0.25, out=out[:9]).data_ptr() == out.data_ptr()
    assert torch.equal(out[:9], want) and out[9:].isnan().all()
