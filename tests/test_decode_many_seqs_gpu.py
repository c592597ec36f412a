"""Decode attention of more (sequence, kv head) pairs than CUs: workgroups of four waves or eight, the sequences in order or from the longest to the shortest, on
both sides of where each is taken -- against attention in fp32 over the gathered pages."""
import pytest
import torch

from aphrodite_engine_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu
DEV, BS = "cuda", 16


def _lens(kind, n, longest):
    g = torch.Generator().manual_seed(n * longest)
    lens = torch.full((n,), longest) if kind == "even" else torch.randint(1, longest + 1, (n,), generator=g)
    if kind == "empty":
        lens[::7] = 0
    if kind == "tied":                                       # many of one number of 32-token pairs, of different lengths
        lens = 32 * (lens // 100) + 1 + lens % 32
    lens[n - 1] = longest
    return lens.int().to(DEV)


def _cache(x, width):                                        # [n, pages, hkv, BS, d] -> keys [pages, hkv, d / width, BS, width]
    n, pages, hkv, _, d = x.shape
    return x.view(n * pages, hkv, BS, d // width, width).transpose(2, 3).contiguous()


@pytest.mark.parametrize("kind,n,hkv,rep,d,longest", [
    ("ragged", 97, 8, 4, 128, 700), ("ragged", 256, 3, 8, 128, 333), ("empty", 130, 8, 4, 128, 290), ("tied", 200, 4, 2, 64, 500),
    ("even", 96, 8, 4, 128, 257), ("ragged", 257, 4, 1, 128, 300), ("ragged", 100, 8, 2, 256, 400), ("tied", 65, 12, 20, 128, 300),
    ("ragged", 256, 3, 8, 128, 533), ("empty", 130, 8, 4, 128, 590), ("tied", 200, 4, 2, 64, 700), ("even", 96, 8, 4, 128, 513), ("ragged", 100, 8, 2, 256, 600),
    ("empty", 48, 8, 4, 128, 1100), ("ragged", 39, 8, 1, 128, 700), ("ragged", 40, 8, 2, 64, 600), ("ragged", 41, 8, 4, 128, 1023)])
@pytest.mark.parametrize("dtype,kv", [(torch.float16, "auto"), (torch.bfloat16, "auto"), (torch.float16, "fp8")])
def test_longest_first(kind, n, hkv, rep, d, longest, dtype, kv):
    g = torch.Generator(device=DEV).manual_seed(n + longest)
    pages = (longest + BS - 1) // BS
    q = torch.randn(n, hkv * rep, d, generator=g, device=DEV).to(dtype)
    k, v = (torch.randn(n, pages, hkv, BS, d, generator=g, device=DEV).to(dtype) for _ in range(2))
    if kv == "fp8":
        k, v = (x.to(torch.float8_e4m3fn) for x in (k, v))
    lens = _lens(kind, n, longest)
    order = torch.randperm(n * pages, generator=g, device=DEV)
    width = 16 // k.element_size()
    kc, vc = _cache(k, width), v.view(n * pages, hkv, BS, d).transpose(2, 3).contiguous()
    if kv == "fp8":
        kc, vc = kc.view(torch.uint8), vc.view(torch.uint8)
    kc[order], vc[order] = kc.clone(), vc.clone()
    table = order.int().view(n, pages)
    out = torch.full_like(q, float("nan"))
    ops.paged_attention_v1(out, q, kc, vc, hkv, d ** -0.5, table, lens, BS, longest, None, kv, 1.0, 1.0)
    kf, vf = (x.float().permute(0, 2, 1, 3, 4).reshape(n, hkv, pages * BS, d) for x in (k, v))
    s = torch.matmul(q.float().view(n, hkv, rep, d) * d ** -0.5, kf.transpose(2, 3).contiguous())
    s.masked_fill_(torch.arange(pages * BS, device=DEV) >= lens.view(n, 1, 1, 1), float("-inf"))
    want = torch.matmul(torch.softmax(s, -1), vf).view(n, hkv * rep, d)
    some = lens > 0
    # probabilities are rounded to the type (u of the largest value, which weights that sum to one average) and so is the result
    u = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    top = vf.abs().amax()
    assert ((out.float() - want).abs()[some] <= 2 * u * (top + want.abs()[some])).all()
    assert out[~some].isnan().all()
