"""Which form a decode batch takes: runs of keys shared by workgroups against one workgroup a (sequence, kv head) on both sides of the plan's
lines, and few-rows products whose weights take the non-temporal hint on both sides of theirs."""
import os

import pytest
import torch

from aphrodite_engine_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu


# (sequences, kv heads, longest): the last length without runs and the first with them for up to eight, four and two of them; more groups than
# half the CUs; the longest
@pytest.mark.parametrize("seqs,hkv,longest", [(1, 8, 352), (1, 8, 353), (1, 1, 600), (8, 8, 384), (8, 8, 385), (9, 8, 500), (16, 8, 864), (16, 8, 865),
                                              (17, 8, 1100), (3, 2, 5000)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_runs_of_keys(seqs, hkv, longest, dtype):
    g = torch.Generator(device="cuda").manual_seed(seqs * longest)
    D, BS, rep = 128, 16, 4
    bps = (longest + BS - 1) // BS
    q = torch.randn(seqs, hkv * rep, D, generator=g, device="cuda").to(dtype)
    kc = torch.randn(seqs * bps + 2, hkv, D // 8, BS, 8, generator=g, device="cuda").to(dtype)
    vc = torch.randn(seqs * bps + 2, hkv, D, BS, generator=g, device="cuda").to(dtype)
    table = torch.randperm(seqs * bps + 2, generator=g, device="cuda")[:seqs * bps].int().view(seqs, bps)
    lens = torch.randint(1, longest + 1, (seqs,), generator=g, device="cuda").int()
    lens[seqs - 1] = longest

    def run():
        out = torch.full_like(q, float("nan"))
        ops.paged_attention_v1(out, q, kc, vc, hkv, D ** -0.5, table, lens, BS, longest, None, "auto", 1.0, 1.0)
        return out

    got, again = run(), run()
    old = os.environ.get("APHRO_PA_SPLITS")
    try:
        os.environ["APHRO_PA_SPLITS"] = "1"
        ops.reload_env()
        want = run().double()
    finally:
        if old is None:
            del os.environ["APHRO_PA_SPLITS"]
        else:
            os.environ["APHRO_PA_SPLITS"] = old
        ops.reload_env()
    # a probability is rounded to the type against another maximum in each form (u of the largest value each), and so is the result
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    assert bool(((got.double() - want).abs() <= 2 * u * (float(vc.abs().max()) + want.abs())).all())
    assert torch.equal(got, again)


# 48 / 49 and 128 / 129 rows; 39 and 40 steps of 64 k in one piece, in slices of 40, and in short ones
@pytest.mark.parametrize("m", [16, 48, 49, 64, 65, 96, 97, 128, 129])
@pytest.mark.parametrize("n,k", [(20488, 2496), (20488, 2560), (6152, 10240), (4104, 2048)])
def test_streamed_weights(m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, k, generator=g, device="cuda").half()
    w = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).half()
    want = x.double() @ w.double().t()
    got = ops.dense_rows(x, w)
    # one rounding to the type, and fp32 sums of k products whose terms' sizes add up to about sqrt(k) times the result's
    assert bool(((got.double() - want).abs() <= 2.0 ** -11 * want.abs() + k * 2.0 ** -24 * 4.0).all())


# 256 rows of w a workgroup, two rounds of them: every height of x's tile, its first and last row, a ragged last tile; one row past it, a round less
# full and K below the line, which go the other way
@pytest.mark.parametrize("m,n,k", [(65, 124936, 2560), (96, 124936, 2560), (97, 131072, 2560), (128, 124936, 2560), (129, 124936, 2560), (160, 124936, 2560),
                                   (161, 124936, 2560), (96, 110000, 2560), (96, 124936, 2496)])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_wide_heads(m, n, k, dtype):
    g = torch.Generator(device="cuda").manual_seed(m)
    x = torch.randn(m, k, generator=g, device="cuda").to(dtype)
    w = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).to(dtype)
    bias = torch.randn(n, generator=g, device="cuda").to(dtype)
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    got, biased, wide = ops.dense_rows(x, w), ops.dense_rows(x, w, bias), ops.dense_rows(x, w, f32=True)
    assert torch.equal(wide, got.float())
    for part in range(0, n, 32768):                      # one rounding to the type, and fp32 sums of k products
        want = x.double() @ w[part:part + 32768].double().t()
        for out, off in ((got, 0.0), (biased, bias[part:part + 32768].double())):
            assert bool(((out[:, part:part + 32768].double() - (want + off)).abs() <= u * (want + off).abs() + k * 2.0 ** -24 * 4.0).all())


def test_marked_weights_give_the_same_results():
    """Every kernel that takes the hint, with it, without it and by the weight's size."""
    g = torch.Generator(device="cuda").manual_seed(0)
    f8 = lambda *s: (torch.randn(*s, generator=g, device="cuda") * 0.1).to(torch.float8_e4m3fn)

    def same(weight, call):
        outs = []
        for mark in (None, True, False):
            if mark is None:
                weight.__dict__.pop("streamed", None)
            else:
                weight.streamed = mark
            outs.append(call(weight))
        assert outs[0].isfinite().all() and outs[0].any() and torch.equal(outs[0], outs[1]) and torch.equal(outs[0], outs[2])

    for m in (1, 16, 40, 64, 100, 150):
        x = torch.randn(m, 2560, generator=g, device="cuda").half()
        same((torch.randn(20488, 2560, generator=g, device="cuda") * 0.02).half(), lambda w: ops.dense_rows(x, w))
    x = torch.randn(20, 2048, generator=g, device="cuda").bfloat16()
    same(torch.randn(32008, 2048, generator=g, device="cuda").bfloat16(), lambda w: ops.lm_head_argmax(x, w))
    sb, one = torch.rand(16384, generator=g, device="cuda") + 0.5, torch.ones(1, device="cuda")
    for m in (7, 32, 64, 128, 192):                          # (the stream kernel up to 32 rows, the few-rows one from 33 on)
        a, sa = f8(m, 1024), torch.rand(m, 1, generator=g, device="cuda") + 0.5
        w = f8(16384, 1024).t()
        same(w, lambda w: ops.cutlass_scaled_mm(a, w, sa, sb, torch.float16))
        same(w, lambda w: ops.scaled_mm_fp8_slabs(a, w))
        if m <= 32:
            assert ops.fp8_gemm_silu_quant_supported(m, 16384, 1024)
            same(w, lambda w: ops.fp8_gemm_silu_quant(a, w, sa, sb, one, torch.float16).float())
