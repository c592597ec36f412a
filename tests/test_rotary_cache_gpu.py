"""Rotary embedding and cache write in one launch (csrc/paged_attention.hip, rotary_cache_kernel): the bits of the two ops it stands for, for
token counts around its 16-token windows, slots that run through a block, that begin inside one, that are shuffled and that are padding,
block sizes of one and two windows, head sizes, types, cache formats and scales; and what it does not serve."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def setup(T, heads, kv_heads, hd, block, dtype, kv, slots, seed=0):
    g = torch.Generator(device=DEV).manual_seed(seed)
    nb = (T + 40) // block + 3
    qkv = torch.randn(T, (heads + 2 * kv_heads) * hd + 16, generator=g, device=DEV).to(dtype)
    x, cdt = (8, dtype) if kv == "auto" else (16, torch.uint8)
    kc = torch.zeros(nb, kv_heads, hd // x, block, x, device=DEV, dtype=cdt)
    vc = torch.zeros(nb, kv_heads, hd, block, device=DEV, dtype=cdt)
    cs = torch.randn(64, hd, generator=g, device=DEV).to(dtype)
    pos = torch.randint(0, 64, (T, ), generator=g, device=DEV)
    if slots == "run":
        sm = torch.arange(T, device=DEV) + block
    elif slots == "offset":
        sm = torch.arange(T, device=DEV) + block + 5
    else:
        sm = torch.randperm(nb * block, generator=g, device=DEV)[:T]
    if slots == "padding":
        sm[::3] = -1
    return qkv, kc, vc, cs, pos, sm.contiguous()


def parts(qkv, heads, kv_heads, hd):
    a, b = heads * hd, (heads + kv_heads) * hd
    return qkv[:, :a], qkv[:, a:b], qkv[:, b:b + kv_heads * hd]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kv", ["auto", "fp8", "fp8_e5m2"])
@pytest.mark.parametrize("T", [1, 15, 16, 17, 80])
@pytest.mark.parametrize("heads,kv_heads,hd,block", [(32, 8, 128, 16), (5, 1, 64, 32), (3, 3, 128, 32), (6, 2, 64, 16)])
@pytest.mark.parametrize("slots", ["run", "offset", "shuffled", "padding"])
def test_same_bits_as_the_two_ops(dtype, kv, T, heads, kv_heads, hd, block, slots):
    from aphrodite_engine_amd import _custom_ops as ops
    qkv, kc, vc, cs, pos, sm = setup(T, heads, kv_heads, hd, block, dtype, kv, slots, seed=T + heads)
    want, kc2, vc2 = qkv.clone(), kc.clone(), vc.clone()
    q, k, v = parts(want, heads, kv_heads, hd)
    ops.rotary_embedding(pos, q, k, hd, cs, True)
    ops.reshape_and_cache(k.view(T, kv_heads, hd), v.view(T, kv_heads, hd), kc2, vc2, sm, kv, 0.5, 2.0)
    q, k, v = parts(qkv, heads, kv_heads, hd)
    assert ops.rotary_embedding_and_cache(pos, q, k, v, hd, cs, True, kc, vc, sm, kv, 0.5, 2.0)
    assert torch.equal(qkv, want) and torch.equal(kc, kc2) and torch.equal(vc, vc2)


def test_what_it_does_not_serve():
    from aphrodite_engine_amd import _custom_ops as ops
    qkv, kc, vc, cs, pos, sm = setup(20, 4, 2, 64, 16, torch.float16, "auto", "run")
    before = qkv.clone()
    q, k, v = parts(qkv, 4, 2, 64)
    go = lambda *a: ops.rotary_embedding_and_cache(*a, "auto", 1.0, 1.0)
    assert not go(pos, q, k, v, 64, cs, False, kc, vc, sm)                        # pairs of neighbours
    assert not go(pos, q, k, v, 64, cs[:, :32].contiguous(), True, kc, vc, sm)     # half of the head
    assert not go(pos.int(), q, k, v, 64, cs, True, kc, vc, sm)
    wide = torch.empty(20, 4 * 64 + 1, device=DEV, dtype=torch.float16)[:, 1:]
    assert not go(pos, wide, k, v, 64, cs, True, kc, vc, sm)                       # rows off 16 bytes
    qkv8, kc8, vc8, cs8, pos8, sm8 = setup(20, 4, 2, 80, 16, torch.float16, "auto", "run")
    assert not go(pos8, *parts(qkv8, 4, 2, 80), 80, cs8, True, kc8, vc8, sm8)       # heads of 80
    assert torch.equal(qkv, before) and not kc.any() and not vc.any()
