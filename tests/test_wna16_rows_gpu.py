"""The int4 GEMM for 65 rows and more with tile heights that fit the batch (csrc/wna16_gemm_rows.hip): against 64-bit products at the
edges of tiles, row blocks, K slices and groups, on the packed and the strip-major weights, with and without SiluAndMul."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def weights(k, n, group, dtype, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    words = lambda *s: torch.randint(-2 ** 31, 2 ** 31 - 1, s, generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    sc = (torch.rand(k // group, n, generator=g, device=DEV) * 0.5 + 0.75) / (6.7 * k ** 0.5)
    return words(k // 8, n), words(k // group, n // 8), sc.to(dtype), g


def dense(qw, qz, sc, zero_offset):
    """float64 [K, N] of exllama words: nibble i of a word is k = (0, 2, 4, 6, 1, 3, 5, 7)[i]"""
    q = torch.empty(qw.shape[0], 8, qw.shape[1], dtype=torch.int32, device=DEV)
    for i, k in enumerate((0, 2, 4, 6, 1, 3, 5, 7)):
        q[:, k] = (qw >> (4 * i)) & 15
    z = torch.stack([(qz >> (4 * i)) & 15 for i in range(8)], 2).flatten(1) + zero_offset
    q = q.flatten(0, 1)
    rows = torch.arange(q.shape[0], device=DEV) // (q.shape[0] // sc.shape[0])
    return (q - z[rows]).double() * sc.double()[rows]


# A weight is rounded to float16 once and the result once: each half an ulp at most, 2^-11 / sqrt(3) on the root mean square of a relative
# error (2^-8 for a bfloat16 result); fp32 sums in between.
BOUND = {torch.float16: 2 ** 0.5 * 2 ** -11 / 3 ** 0.5 * 1.1, torch.bfloat16: 2 ** -8 / 3 ** 0.5 * 1.1}


@pytest.mark.parametrize("dtype,group", [(torch.float16, 128), (torch.float16, 64), (torch.bfloat16, 128), (torch.float16, 0)])
@pytest.mark.parametrize("m", [65, 96, 97, 128, 129, 160, 161, 300, 1025])
@pytest.mark.parametrize("k,n", [(128, 128), (640, 384), (1536, 2048), (4224, 256), (512, 28672)])
def test_rows_gemm(dtype, group, m, k, n):
    from aphrodite_engine_amd import _custom_ops as ops
    group = group or k
    qw, qz, sc, g = weights(k, n, group, dtype, m + k + n)
    a = torch.randn(m, k + 8, generator=g, device=DEV).to(dtype)[:, :k]              # rows further apart than they are long
    want = a.double() @ dense(qw, qz, sc, 1)
    got = ops._wna16_large(a, qw, qz, sc, None, 1)
    assert float((got.double() - want).norm() / want.norm()) < BOUND[dtype]
    for _ in range(3):
        assert torch.equal(ops._wna16_large(a, qw, qz, sc, None, 1), got)
    assert torch.equal(ops.gptq_gemm(a, qw, qz, sc, torch.empty(0, dtype=torch.int32, device=DEV), True, 4), got) \
        or not ops.wna16_prefers_large(m, n, k)
    if ops.wna16_gemm_large_silu_supported(m, n, k, k // group):
        act = ops.wna16_gemm_large_silu(a, qw, qz, sc, 1)
        gate, up = got[:, 0::2].contiguous(), got[:, 1::2].contiguous()
        out = torch.empty_like(gate)
        ops.silu_and_mul(out, torch.cat([gate, up], 1))
        assert torch.equal(act, out)
    if group == 128 and ops.wna16_resident_ksplit(32, n, k, k // 128) > 0:
        strip = ops.wna16_strip_relayout(qw, 32, k // 128)
        assert torch.equal(ops.wna16_gemm_large_strip(a, strip, qz, sc, 1), got)
        if m > 128 or ops.wna16_prefers_large(m, n, k):
            assert torch.equal(ops.wna16_linear_strip(a, strip, qz, sc, 1), got)


@pytest.mark.parametrize("m", [65, 96, 97, 128])
@pytest.mark.parametrize("k,n", [(4096, 4096), (4096, 6144), (2048, 4096)])
def test_small_projections_do_not_round_their_weights(m, k, n):
    """float16, 65 to 128 rows, by the public entries: no further from 64 bits than the rounding of the exact result is (the fp32 sums add
    a hundredth of it; weights rounded to float16 as well add four tenths)."""
    from aphrodite_engine_amd import _custom_ops as ops
    qw, qz, sc, g = weights(k, n, 128, torch.float16, m + n)
    a = torch.randn(m, k, generator=g, device=DEV).half()
    want = a.double() @ dense(qw, qz, sc, 1)
    bound = 1.02 * float((want.half().double() - want).norm())
    got = [ops.gptq_gemm(a, qw, qz, sc, torch.empty(0, dtype=torch.int32, device=DEV), True, 4)]
    if ops.wna16_resident_ksplit(32, n, k, k // 128) > 0:
        got.append(ops.wna16_linear_strip(a, ops.wna16_strip_relayout(qw, 32, k // 128), qz, sc, 1))
    assert all(float((x.double() - want).norm()) < bound for x in got)


@pytest.mark.parametrize("m", [65, 97, 128])
@pytest.mark.parametrize("k,n,group", [(128, 128, 128), (640, 384, 64), (4224, 256, 128), (1536, 2048, 192), (8192, 1024, 64), (16384, 512, 64), (4096, 1024, 4096)])
def test_tiles_that_round_no_weight(m, k, n, group):
    """The form for 65 to 128 float16 rows: groups inside, across and beside K tiles, more of them than one slice's scales fit."""
    from aphrodite_engine_amd import _custom_ops as ops, _lib
    assert _lib.lib().aphro_wna16_rows_exact_tiles(m, n, k, k // group) > 0
    qw, qz, sc, g = weights(k, n, group, torch.float16, m + n)
    a = torch.randn(m, k + 8, generator=g, device=DEV).half()[:, :k]
    want = a.double() @ dense(qw, qz, sc, 0)
    got = ops._wna16_large(a, qw, qz, sc, None, 0)
    assert float((got.double() - want).norm()) < 1.02 * float((want.half().double() - want).norm())
    assert torch.equal(ops._wna16_large(a, qw, qz, sc, None, 0), got)


@pytest.mark.parametrize("m,k,n", [(65, 576, 256), (150, 4160, 4096), (300, 4160, 1024), (513, 2112, 8192)])
def test_k_that_the_row_tile_does_not_take(m, k, n):
    """K = 64 (mod 128): the few-tile plans of csrc/wna16_gemm_large.hip, K slices of whole groups among them."""
    from aphrodite_engine_amd import _custom_ops as ops
    qw, qz, sc, g = weights(k, n, 64, torch.float16, m + k + n)
    a = torch.randn(m, k, generator=g, device=DEV).half()
    want, got = a.double() @ dense(qw, qz, sc, 1), ops._wna16_large(a, qw, qz, sc, None, 1)
    assert float((got.double() - want).norm() / want.norm()) < BOUND[torch.float16]
    assert torch.equal(ops._wna16_large(a, qw, qz, sc, None, 1), got)


def test_rows_gemm_keeps_a_row_s_infinities_and_nans_to_itself():
    from aphrodite_engine_amd import _custom_ops as ops
    qw, qz, sc, g = weights(1024, 512, 128, torch.float16, 3)
    a = torch.randn(150, 1024, generator=g, device=DEV).half()
    want = ops._wna16_large(a, qw, qz, sc, None, 1)
    b = a.clone()
    b[7, 100], b[149, 1023] = float("inf"), float("nan")
    got = ops._wna16_large(b, qw, qz, sc, None, 1)
    rows = [r for r in range(150) if r not in (7, 149)]
    assert torch.equal(got[rows], want[rows])
    assert not torch.isfinite(got[7]).any() and torch.isnan(got[149]).all()


def test_rows_gemm_in_a_graph():
    from aphrodite_engine_amd import _custom_ops as ops
    qw, qz, sc, g = weights(4096, 4096, 128, torch.float16, 5)
    a = torch.randn(150, 4096, generator=g, device=DEV).half()
    ops._wna16_large(a, qw, qz, sc, None, 1)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops._wna16_large(a, qw, qz, sc, None, 1)
    for i in range(4):
        a.copy_(torch.randn(150, 4096, generator=g, device=DEV).half())
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, ops._wna16_large(a, qw, qz, sc, None, 1))
