"""Decode attention whose runs of keys are dealt out by the lengths that the launch finds: batches of one length, ragged ones, one long sequence among
short ones, empty ones, more sequences than a wave has lanes -- against the same launch without runs; in the fused forms, where one run writes the new
token, too; and captured once for lengths that differ from replay to replay."""
import contextlib
import os

import pytest
import torch

from aphrodite_engine_amd import _custom_ops as ops, _lib

pytestmark = pytest.mark.gpu
DEV, D = "cuda", 128


@contextlib.contextmanager
def unsplit():
    old = os.environ.get("APHRO_PA_SPLITS")
    try:
        os.environ["APHRO_PA_SPLITS"] = "1"
        ops.reload_env()
        yield
    finally:
        os.environ.pop("APHRO_PA_SPLITS", None) if old is None else os.environ.update(APHRO_PA_SPLITS=old)
        ops.reload_env()


def _lens(kind, n, longest):
    g = torch.Generator().manual_seed(n * longest)
    if kind == "one long":
        lens = torch.full((n,), 300)
    elif kind == "even":
        lens = torch.full((n,), longest)
    elif kind == "short":                                    # (none worth a run, whatever the longest length given)
        lens = torch.randint(1, 480, (n,), generator=g)
    else:
        lens = torch.randint(1, longest + 1, (n,), generator=g)
    if kind == "empty":
        lens[::5] = 0
    if kind != "short":
        lens[n // 2 + 1] = longest
    return lens.int().to(DEV)


def _caches(n, hkv, longest, bs, kv, dtype, g):
    bps = (longest + bs - 1) // bs
    blocks = n * bps + 2
    if kv == "auto":
        kc = torch.randn(blocks, hkv, D // 8, bs, 8, generator=g, device=DEV).to(dtype)
        vc = torch.randn(blocks, hkv, D, bs, generator=g, device=DEV).to(dtype)
    else:
        f8 = torch.float8_e4m3fn if kv == "fp8" else torch.float8_e5m2
        kc = torch.randn(blocks, hkv, D // 16, bs, 16, generator=g, device=DEV).to(f8).view(torch.uint8)
        vc = torch.randn(blocks, hkv, D, bs, generator=g, device=DEV).to(f8).view(torch.uint8)
    return kc, vc, torch.randperm(blocks, generator=g, device=DEV)[:n * bps].int().view(n, bps)


# numbers of about 1: a probability is rounded to the type against another maximum in each form (u of the largest value each), and so is the result
def _bound(want, dtype, top):
    return 2 * (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8) * (top + want.abs())


CASES = [("one long", 24, 8, 4, 4100, 16), ("one long", 31, 8, 4, 3000, 16), ("one long", 9, 8, 1, 2017, 32), ("ragged", 12, 8, 4, 5000, 16), ("ragged", 17, 8, 4, 2600, 32),
         ("ragged", 63, 4, 2, 2100, 16), ("even", 9, 8, 4, 2048, 16), ("even", 16, 8, 16, 2048, 16), ("even", 30, 8, 4, 2050, 16), ("short", 20, 8, 4, 2600, 16),
         ("empty", 21, 8, 4, 2300, 16), ("ragged", 200, 1, 8, 2100, 16), ("one long", 255, 1, 4, 2500, 16), ("one long", 65, 2, 4, 4000, 16)]


@pytest.mark.parametrize("kind,n,hkv,rep,longest,bs", CASES)
@pytest.mark.parametrize("dtype,kv", [(torch.float16, "auto"), (torch.bfloat16, "auto"), (torch.float16, "fp8"), (torch.bfloat16, "fp8_e5m2")])
def test_runs_by_length(kind, n, hkv, rep, longest, bs, dtype, kv):
    g = torch.Generator(device=DEV).manual_seed(n * longest)
    assert _lib.lib().aphro_paged_attention_runs(n, hkv * rep, hkv, D, bs, longest) == 8
    q = torch.randn(n, hkv * rep, D, generator=g, device=DEV).to(dtype)
    kc, vc, table = _caches(n, hkv, longest, bs, kv, dtype, g)
    lens = _lens(kind, n, longest)

    def run():
        out = torch.full_like(q, float("nan"))
        ops.paged_attention_v1(out, q, kc, vc, hkv, D ** -0.5, table, lens, bs, longest, None, kv, 1.0, 1.0)
        return out[lens > 0]

    got, again = run(), run()
    with unsplit():
        want = run().double()
    assert bool(((got.double() - want).abs() <= _bound(want, dtype, 6.0)).all())
    assert torch.equal(got, again)


@pytest.mark.parametrize("kind,n,longest", [("one long", 24, 4100), ("ragged", 12, 2600), ("even", 16, 2048), ("empty", 20, 2300)])
@pytest.mark.parametrize("kv", ["auto", "fp8"])
@pytest.mark.parametrize("form", ["packed", "scaled", "absmax", "q8"])
def test_the_fused_forms(kind, n, longest, kv, form):
    hkv, heads, bs, dtype = 8, 32, 16, torch.float16
    g = torch.Generator(device=DEV).manual_seed(n + longest)
    kc, vc, table = _caches(n, hkv, longest, bs, kv, dtype, g)
    lens = _lens(kind, n, longest).clamp(min=1)
    last = (lens - 1).long()
    slots = table.long().gather(1, (last // bs)[:, None])[:, 0] * bs + last % bs
    slabs = torch.randn(2, n, (heads + 2 * hkv) * D, generator=g, device=DEV) * 0.4
    cs = torch.randn(longest + 1, D, generator=g, device=DEV).to(dtype)
    cols, rows = torch.rand(slabs.shape[2], generator=g, device=DEV) + 0.5, torch.rand(n, generator=g, device=DEV) + 0.5
    scale = torch.tensor([0.02], device=DEV)

    def run():
        k, v = kc.clone(), vc.clone()
        tail = (k, v, heads, hkv, 0.09, table, lens, bs, longest, None, kv, 1.0, 1.0)
        if form == "packed":
            res = ops.paged_attention_rope_packed(slabs, last, cs, slots, *tail, want_out=True)[1]
        else:
            res = ops.paged_attention_rope_scaled(slabs, rows, cols, last, cs, slots, *tail, out_q8_scale=scale if form == "q8" else None,
                                                  want_absmax=form == "absmax")
        return res if isinstance(res, tuple) else (res,), k, v

    (got, k1, v1), (again, _, _) = run(), run()
    with unsplit():
        want, k2, v2 = run()
    assert torch.equal(k1, k2) and torch.equal(v1, v2)       # the run that holds the new token wrote it
    assert bool(((got[0].double() - want[0].double()).abs() <= _bound(want[0].double(), dtype, 6.0)).all())
    if form == "absmax":
        assert torch.equal(got[1], got[0].float().view(n, hkv, -1).abs().amax(-1))
    if form == "q8":
        assert torch.equal(got[1].view(torch.uint8), ops.scaled_fp8_quant(got[0].view(n, -1), scale)[0].view(torch.uint8))
    assert all(torch.equal(a.view(torch.uint8) if a.dtype == torch.float8_e4m3fn else a, b.view(torch.uint8) if b.dtype == torch.float8_e4m3fn else b)
               for a, b in zip(got, again))


def test_a_captured_launch_deals_anew():
    n, hkv, longest, bs, dtype = 24, 8, 4096, 16, torch.float16
    g = torch.Generator(device=DEV).manual_seed(3)
    q = torch.randn(n, 32, D, generator=g, device=DEV).to(dtype)
    kc, vc, table = _caches(n, hkv, longest, bs, "auto", dtype, g)
    lens = _lens("even", n, longest)
    out = torch.empty_like(q)
    run = lambda: ops.paged_attention_v1(out, q, kc, vc, hkv, D ** -0.5, table, lens, bs, longest, None, "auto", 1.0, 1.0)
    run()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for kind in ("one long", "even", "short", "ragged", "one long", "ragged"):
        lens.copy_(_lens(kind, n, longest))
        out.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        got = out.clone()
        run()
        assert torch.equal(out, got)
        with unsplit():
            run()
        assert bool(((got.double() - out.double()).abs() <= _bound(out.double(), dtype, 6.0)).all())
