"""The norm in the launch that sums a GEMM's K slices (csrc/wna16_gemm_rows.hip): the bits of the GEMM followed by fused_add_rms_norm, product,
residual and normed rows, for every height of the tile, the form that rounds no weight, both types, both orders of the weights, ragged last
tiles and rows of one and of two vectors a thread; and None for calls that sum no slices."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def weights(k, n, group, dtype, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    word = lambda *s: torch.randint(-2 ** 31, 2 ** 31, s, generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    return word(k // 8, n), word(k // group, n // 8), (torch.rand(k // group, n, generator=g, device=DEV) * 0.01).to(dtype), g


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("k,n,group", [(4096, 4096, 128), (14336, 4096, 128), (2048, 8192, 64), (4096, 10240, 128), (11008, 4096, 128)])
@pytest.mark.parametrize("m", [65, 96, 97, 128, 129, 150, 161, 300])
def test_same_bits(dtype, k, n, group, m):
    from aphrodite_engine_amd import _custom_ops as ops
    qw, qz, sc, g = weights(k, n, group, dtype, m + n)
    a = torch.randn(m, k + 8, generator=g, device=DEV).to(dtype)[:, :k]
    res = torch.randn(m, n, generator=g, device=DEV).to(dtype)
    w = torch.rand(n, generator=g, device=DEV).to(dtype)
    strips = [None]
    if dtype == torch.float16 and ops.wna16_gemm_rowmajor_supported(32, n, k, k // group, dtype):
        strips.append(ops.wna16_strip_relayout(qw, 32, k // group))
    served = False
    for strip in strips:
        mine = res.clone()
        got = ops.wna16_linear_add_norm(a, qw if strip is None else strip, qz, sc, 1, strip is not None, mine, w, 1e-5)
        if got is None:
            assert torch.equal(mine, res)
            continue
        want = ops.wna16_gemm(a, qw, qz, sc, None, 1) if strip is None else ops.wna16_linear_strip(a, strip, qz, sc, 1)
        ops.fused_add_rms_norm(want, res_want := res.clone(), w, 1e-5)
        assert torch.equal(mine, res_want) and torch.equal(got, want)
        served = True
    assert served or (k, n) != (14336, 4096)


def test_a_captured_call_replays():
    from aphrodite_engine_amd import _custom_ops as ops
    qw, qz, sc, g = weights(4096, 4096, 128, torch.float16, 1)
    a, res, w = (torch.randn(*s, generator=g, device=DEV).half() for s in ((150, 4096), (150, 4096), (4096,)))
    mine = res.clone()
    want = ops.wna16_linear_add_norm(a, qw, qz, sc, 1, False, mine, w, 1e-5)
    graph, again = torch.cuda.CUDAGraph(), res.clone()
    with torch.cuda.graph(graph):
        got = ops.wna16_linear_add_norm(a, qw, qz, sc, 1, False, again, w, 1e-5)
    for _ in range(3):
        again.copy_(res)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(again, mine)


@pytest.mark.parametrize("m", [1, 32, 64, 4096])
def test_calls_without_summed_slices(m):
    from aphrodite_engine_amd import _custom_ops as ops
    qw, qz, sc, g = weights(4096, 4096, 128, torch.float16, m)
    a, res, w = (torch.randn(*s, generator=g, device=DEV).half() for s in ((m, 4096), (m, 4096), (4096,)))
    kept = res.clone()
    assert ops.wna16_linear_add_norm(a, qw, qz, sc, 1, False, res, w, 1e-5) is None and torch.equal(res, kept)
