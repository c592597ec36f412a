"""Norms over groups that lie within a wave and the embedding's 16-byte form (csrc/mixers/norm_act.hip: group_rms_norm_vec8_kernel,
embed_scale_vec8_kernel): against 64-bit math for every group size, row counts that leave a workgroup partly empty, strided rows, with and
without weight and gate, both activations; sizes beside them that take the general kernels."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV, F64 = "cuda", torch.float64
# one rounding to the result's type and fp32 math before it
TOL = {torch.bfloat16: 2.0 ** -8, torch.float32: 2e-6}


def close(got, want, dtype):
    err = (got.to(F64) - want).abs()
    assert bool((err <= TOL[dtype] * want.abs() + 1e-9).all()), float((err / (want.abs() + 1e-9)).max())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("group", [8, 16, 32, 64, 128, 256, 512, 1024, 24, 36])
@pytest.mark.parametrize("rows,groups", [(1, 1), (3, 5), (37, 3)])
def test_group_rms_norm(dtype, group, rows, groups):
    from aphrodite_engine_amd import mixer_ops as mops
    g = torch.Generator(device=DEV).manual_seed(group + rows)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    n = group * groups
    x, w, gt = rnd(rows, n), rnd(n).to(dtype), rnd(rows, n + 8).to(dtype)[:, 8:]
    norm = lambda y: y / torch.sqrt((y * y).mean(-1, keepdim=True) + 1e-5)
    base = norm(x.to(F64).view(rows, groups, group))
    for weight, gate in ((w, gt), (None, gt), (w, None), (None, None)):
        out = torch.full((rows, n + 16), 7.0, device=DEV).to(dtype)
        mops.gated_group_rms_norm(out[:, 8:8 + n], x, weight, gate, group, 1e-5, out_scale=0.7)
        want = base.reshape(rows, n) * 0.7 * (weight.to(F64) if weight is not None else 1) * (torch.sigmoid(gate.to(F64)) if gate is not None else 1)
        close(out[:, 8:8 + n], want, dtype)
        assert bool((out[:, :8] == 7).all()) and bool((out[:, 8 + n:] == 7).all())
    for act in (0, 1):
        out = torch.empty(rows, n, device=DEV, dtype=dtype)
        mops.gated_head_rms_norm(out, x, w[:group].contiguous(), gt, groups, 1e-5, act)
        s = torch.sigmoid(gt.to(F64))
        close(out, (base * w[:group].to(F64)).reshape(rows, n) * (s * gt.to(F64) if act else s), dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("width", [8, 64, 2048, 2056, 4104, 36])
def test_embedding_rows(dtype, width):
    from aphrodite_engine_amd import mixer_ops as mops
    table = torch.randn(50, width, device=DEV).to(dtype)
    ids = torch.tensor([49, 0, 7, 7, 13], device=DEV)
    copy = torch.empty(5, width, device=DEV, dtype=dtype)
    got = mops.embed_scale(table, ids, 1.5, copy=copy)
    assert torch.equal(got, table[ids].float() * 1.5) and torch.equal(copy, got.to(dtype))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d,e,shift", [(128, 128, 0), (8, 24, 0), (20, 4, 0), (4, 6, 0), (64, 32, 1)])
def test_paged_kv_write(dtype, d, e, shift):
    """paged_kv_write in 16-byte pieces and, where rows are none, number by number: every slot gets its row, padding and slots outside none."""
    from aphrodite_engine_amd import mixer_ops as mops
    T, G, nb, bs = 37, 2, 9, 8
    k, v = (torch.randn(T, G * n + 8 + shift, device=DEV).to(dtype)[:, shift:shift + G * n] for n in (d, e))
    kc, vc = (torch.full((nb, bs, G, n), 7.0, device=DEV, dtype=dtype) for n in (d, e))
    slots = torch.randperm(nb * bs, device=DEV)[:T].contiguous()
    slots[5], slots[6] = -1, nb * bs
    want_k, want_v = kc.view(-1, G * d).clone(), vc.view(-1, G * e).clone()
    ok = [i for i in range(T) if i not in (5, 6)]
    want_k[slots[ok]], want_v[slots[ok]] = k[ok], v[ok]
    mops.paged_kv_write(kc, vc, k, v, slots)
    assert torch.equal(kc.view(-1, G * d), want_k) and torch.equal(vc.view(-1, G * e), want_v)
