"""The 128-wide decode attention of the sequence mixers (csrc/mixers/biased_attention_fast.h, dba_decode128_kernel): single tokens against a
64-bit softmax where it can go wrong -- contexts around its 16-key tiles, windows and chunks that begin inside a tile, split key ranges,
block sizes of one tile and of several, slots without a key that hold NaN -- and, for blocks that are no multiples of a tile and unaligned
caches, the general kernel beside it."""
import pytest
import torch

from test_wide_attention_gpu import GROUPS, run

pytestmark = pytest.mark.gpu
CTXS = [0, 1, 14, 15, 16, 17, 62, 63, 64, 65, 127, 333]


@pytest.mark.parametrize("heads,kv_heads", GROUPS + [(1, 1), (5, 1), (8, 8), (16, 1)])
@pytest.mark.parametrize("block", [16, 32, 64, 8, 24])
def test_contexts_around_tiles(heads, kv_heads, block):
    run([1] * len(CTXS), CTXS, heads, kv_heads, block, seed=heads, fill=float("nan"))


@pytest.mark.parametrize("kw", [dict(bias=1), dict(bias=50, temp=0.1), dict(bias=4096, gate="heads"), dict(window=1), dict(window=40, bias=64), dict(chunk=48),
                                dict(softcap=5.0, bias=16, sink=True), dict(window=100, chunk=64, sink=True, gate="columns"), dict(gate="columns"),
                                dict(gate="columns", pad=1), dict(softcap=2.0, window=64, gate="heads", pad=3)])
@pytest.mark.parametrize("block", [16, 64])
def test_forms(kw, block):
    run([1] * len(CTXS), CTXS, 8, 2, block, seed=3, fill=float("nan"), **kw)


@pytest.mark.parametrize("kw", [dict(), dict(bias=300, temp=0.1), dict(window=700, sink=True), dict(window=513, softcap=9.0, gate="columns")])
@pytest.mark.parametrize("ctxs", [[512], [511, 40, 1300], [2047, 2048, 2049, 3], [4000, 15]])
@pytest.mark.parametrize("shift", [0, 4])
def test_split_key_ranges(kw, ctxs, shift):
    run([1] * len(ctxs), ctxs, 8, 2, 16, seed=len(ctxs), fill=float("nan"), shift=shift, **kw)
