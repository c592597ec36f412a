"""Rotation and cache write in the launch that sums a qkv projection's K slices: the bits of the product followed by rotary_embedding_and_cache, rows
and caches, for windows of 16 tokens and their remainders, both head sizes, both types, cache formats, both orders of the weights and slots that
run through a block, are shuffled and are padding; and None, with nothing written, for calls that sum no slices or a geometry it does not serve."""
import pytest
import torch

from test_rotary_cache_gpu import parts, setup
from test_wna16_add_norm_gpu import weights

pytestmark = pytest.mark.gpu
DEV = "cuda"


def call(ops, a, qw, qz, sc, strip, pos, heads, kv_heads, hd, cs, kc, vc, sm, kv):
    return ops.wna16_linear_rotary_cache(a, qw, qz, sc, 1, strip, pos, heads, kv_heads, hd, cs, kc, vc, sm, kv, 0.5, 2.0)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kv", ["auto", "fp8", "fp8_e5m2"])
@pytest.mark.parametrize("heads,kv_heads,hd,block,k", [(32, 8, 128, 16, 4096), (9, 3, 128, 32, 2048), (14, 5, 64, 16, 2048)])
@pytest.mark.parametrize("m,slots", [(65, "run"), (96, "shuffled"), (97, "padding"), (128, "offset"), (129, "shuffled"), (150, "padding"), (300, "run")])
def test_same_bits(dtype, kv, heads, kv_heads, hd, block, k, m, slots):
    from aphrodite_engine_amd import _custom_ops as ops
    _, kc, vc, cs, pos, sm = setup(m, heads, kv_heads, hd, block, dtype, kv, slots, seed=m)
    n = (heads + 2 * kv_heads) * hd
    qw, qz, sc, g = weights(k, n, 128, dtype, m + n)
    a = torch.randn(m, k + 8, generator=g, device=DEV).to(dtype)[:, :k]
    forms = [(qw, False)]
    if dtype == torch.float16 and ops.wna16_gemm_rowmajor_supported(32, n, k, k // 128, dtype):
        forms.append((ops.wna16_strip_relayout(qw, 32, k // 128), True))
    for words, strip in forms:
        kc1, vc1, kc2, vc2 = kc.clone(), vc.clone(), kc.clone(), vc.clone()
        got = call(ops, a, words, qz, sc, strip, pos, heads, kv_heads, hd, cs, kc1, vc1, sm, kv)
        served = ops.wna16_prefers_large(m, n, k, dtype, k // 128, strip=strip) and bool(
            ops._lib.lib().aphro_wna16_gemm_large_rotary_cache_supported(m, n, k, k // 128, ops._dt(a)))
        assert (got is not None) == served and (served or m not in (129, 150))       # (every head size, type and order of the weights)
        if got is None:                                     # (this order of the weights goes to other kernels)
            assert not kc1.any() and not vc1.any()
            continue
        want = ops.wna16_linear_strip(a, words, qz, sc, 1) if strip else ops.wna16_gemm(a, qw, qz, sc, None, 1)
        assert ops.rotary_embedding_and_cache(pos, *parts(want, heads, kv_heads, hd), hd, cs, True, kc2, vc2, sm, kv, 0.5, 2.0)
        assert torch.equal(got, want) and torch.equal(kc1, kc2) and torch.equal(vc1, vc2)


@pytest.mark.parametrize("m,change", [(64, None), (4096, None), (150, "heads"), (150, "positions"), (150, "interleaved cos"), (150, "aligned")])
def test_what_it_does_not_serve(m, change):
    from aphrodite_engine_amd import _custom_ops as ops
    _, kc, vc, cs, pos, sm = setup(m, 32, 8, 128, 16, torch.float16, "auto", "run")
    qw, qz, sc, g = weights(4096, 6144, 128, torch.float16, m)
    a = torch.randn(m, 4096, generator=g, device=DEV).half()
    heads, hd = 32, 128
    if change == "heads":
        heads = 31
    elif change == "positions":
        pos = pos.int()
    elif change == "interleaved cos":
        cs = cs[:, :64].contiguous()
    elif change == "aligned":
        cs = torch.cat([cs.flatten(), cs.flatten()[:8]])[1:64 * 128 + 1].view(64, 128)
    assert call(ops, a, qw, qz, sc, False, pos, heads, 8, hd, cs, kc, vc, sm, "auto") is None
    assert not kc.any() and not vc.any()


def test_a_captured_call_replays():
    from aphrodite_engine_amd import _custom_ops as ops
    _, kc, vc, cs, pos, sm = setup(150, 32, 8, 128, 16, torch.float16, "auto", "shuffled")
    qw, qz, sc, g = weights(4096, 6144, 128, torch.float16, 1)
    a = torch.randn(150, 4096, generator=g, device=DEV).half()
    args = (ops, a, qw, qz, sc, False, pos, 32, 8, 128, cs)
    want = call(*args, kc, vc, sm, "auto")
    kc2, vc2 = torch.zeros_like(kc), torch.zeros_like(vc)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = call(*args, kc2, vc2, sm, "auto")
    for _ in range(3):
        kc2.zero_(), vc2.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(kc2, kc) and torch.equal(vc2, vc)
