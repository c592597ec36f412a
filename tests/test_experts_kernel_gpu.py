"""The grouped int4 product of workgroups that stay (more units than one a workgroup) against the one of a workgroup a unit, tile by tile: the same bits,
for every length of a wave's chain and every result, rows and experts that are not there, shares that do not divide."""
import pytest
import torch

from aphrodite_engine_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _weights(e, k, n, group, dtype, g):
    qw = torch.randint(-2 ** 31, 2 ** 31 - 1, (e, k // 8, n), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    qz = torch.randint(-2 ** 31, 2 ** 31 - 1, (e, k // group, n // 8), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    return qw, qz, ((torch.rand(e, k // group, n, generator=g, device=DEV) * 0.5 + 0.75) / (6.7 * k ** 0.5)).to(dtype)


def _call(x, rows, ids, there, w, mode):
    m_pad = 16 * len(ids)
    post = torch.tensor([there], dtype=torch.int32, device=DEV)
    packed = ops.moe_gather_pack(x, rows, torch.tensor([m_pad], dtype=torch.int32, device=DEV), m_pad, 1)
    return ops.wna16_gemm_grouped(packed, m_pad, x.shape[1], *w, torch.tensor(ids, dtype=torch.int32, device=DEV), post, 1, mode)


def _call_into(out, mode, x, rows, ids, there, w):
    """The same into a result that is there: packed activations, slabs or rows."""
    m_pad, k, n, groups = 16 * len(ids), x.shape[1], w[0].shape[2], w[2].shape[1]
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device=DEV)
    packed, post, ids = ops.moe_gather_pack(x, rows, i32([m_pad]), m_pad, 1), i32([there]), i32(ids)
    c, slabs, act = (out if mode == "out" else None), (out if mode == "slabs" else None), (out if mode == "silu_pack" else None)
    p = lambda t: None if t is None else t.data_ptr()
    ops.check(ops._lib.lib().aphro_wna16_gemm_grouped(packed.data_ptr(), *(t.data_ptr() for t in w), ids.data_ptr(), post.data_ptr(), p(c), p(slabs),
                                                      0 if slabs is None else slabs.numel() * 4, p(act), m_pad, n, k, groups, 1, ops._dt(w[2]), ops._stream()), "grouped")


def _tiles_of(out, mode, tiles, n):
    """[tile, ...]: what belongs to each tile of 16 rows."""
    if mode == "silu_pack":
        return out.view(n // 256, 4, tiles, 64 * 8).permute(2, 0, 1, 3)
    if mode == "slabs":
        return out[0].view(out[1], tiles, 16, n).transpose(0, 1)
    return out.view(tiles, 16, n)


@pytest.mark.parametrize("k,n,group,tiles,there,mode,dtype", [
    (4096, 4096, 128, 40, 640, "silu_pack", torch.float16), (4096, 4096, 128, 40, 601, "slabs", torch.bfloat16), (2048, 8192, 128, 37, 592, "out", torch.float16),
    (2048, 8192, 256, 20, 320, "silu_pack", torch.bfloat16), (3584, 8192, 128, 19, 300, "slabs", torch.float16), (14336, 4096, 128, 12, 16, "slabs", torch.float16),
    (14336, 4096, 512, 9, 144, "slabs", torch.bfloat16)])
def test_same_bits_as_a_workgroup_a_unit(k, n, group, tiles, there, mode, dtype):
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    ks = ops.wna16_grouped_ksplit(16 * tiles, n, k, k // group)
    assert tiles * ks * (n // 64) > 2 * cus
    g = torch.Generator(device=DEV).manual_seed(k + n + tiles)
    w = _weights(3, k, n, group, dtype, g)
    x = torch.randn(16 * tiles, k, generator=g, device=DEV).to(dtype)
    rows = torch.arange(16 * tiles, dtype=torch.int32, device=DEV)
    ids = [(t * 7 + t // 5) % 4 - 1 for t in range(tiles)]                 # (-1: an expert that lies elsewhere)
    got = _tiles_of(_call(x, rows, ids, there, w, mode), mode, tiles, n)
    few = 2 * cus // (ks * (n // 64))
    seen = 0
    for t in range(tiles):
        if ids[t] < 0 or 16 * t >= there:
            continue
        assert few >= 1 and ops.wna16_grouped_ksplit(16, n, k, k // group) >= ks
        if ops.wna16_grouped_ksplit(16 * few, n, k, k // group) != ks:
            pytest.skip("no call of few tiles cuts K alike")
        pad = [ids[t]] + [-1] * (few - 1)
        alone = _call(x, torch.cat([rows[16 * t:16 * t + 16], rows[:16 * (few - 1)]]), pad, 16, w, mode)
        assert torch.equal(got[t], _tiles_of(alone, mode, few, n)[0])
        seen += 1
    assert seen == sum(1 for t in range(tiles) if ids[t] >= 0 and 16 * t < there)


@pytest.mark.parametrize("k,n,tiles,there,mode,dtype", [
    (4096, 8192, 17, 0, "slabs", torch.float16), (4096, 8192, 17, 0, "out", torch.bfloat16), (4096, 4096, 40, 0, "silu_pack", torch.float16),
    (4096, 4096, 40, 601, "silu_pack", torch.bfloat16), (14336, 4096, 12, 100, "slabs", torch.float16), (2048, 8192, 37, 320, "out", torch.float16)])
def test_tiles_that_are_not_there_stay(k, n, tiles, there, mode, dtype):
    """Tiles past the rows that are there, and those of experts that lie elsewhere, keep what was in their place; the others lose all of it."""
    ks = ops.wna16_grouped_ksplit(16 * tiles, n, k, k // 128)
    assert tiles * ks * (n // 64) > 2 * torch.cuda.get_device_properties(0).multi_processor_count
    g = torch.Generator(device=DEV).manual_seed(k + tiles)
    w, x = _weights(3, k, n, 128, dtype, g), torch.randn(16 * tiles, k, generator=g, device=DEV).to(dtype)
    ids = [(t * 7 + t // 5) % 4 - 1 for t in range(tiles)]
    if mode == "slabs":
        out = torch.full((ks, 16 * tiles, n), -12345.0, device=DEV)
    elif mode == "out":
        assert ks == 1
        out = torch.full((16 * tiles, n), -12345.0, device=DEV).to(dtype)
    else:
        out = torch.full((16 * tiles * (n // 2), ), -12345.0, dtype=torch.float16, device=DEV)
    before = out.flatten()[0].item()
    _call_into(out, mode, x, torch.arange(16 * tiles, dtype=torch.int32, device=DEV), ids, there, w)
    got = _tiles_of((out, ks) if mode == "slabs" else out, mode, tiles, n)
    for t in range(tiles):
        stays = (got[t] == before)
        assert stays.all() if ids[t] < 0 or 16 * t >= there else not stays.any(), t
