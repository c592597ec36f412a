"""The stream-K GEMMs, whose workgroups wait for one another's flags, replayed from a graph among eager calls of the same kernels: flags left
from the last replay would let a workgroup take the last replay's sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("kind", ["int4", "fp8"])
def test_streamk_gemms_replay(kind):
    from aphrodite_engine_amd import _custom_ops as ops
    m, k, n = 2048, 4096, 6144
    tiles, cus = m // 256 * (n // 256), torch.cuda.get_device_properties(0).multi_processor_count
    assert tiles >= 128 and tiles % cus != 0                 # a persistent grid whose workgroups share tiles
    g = torch.Generator(device=DEV).manual_seed(1)
    if kind == "int4":
        words = lambda *s: torch.randint(-2 ** 31, 2 ** 31 - 1, s, generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
        qw, qz, sc = words(k // 8, n), words(k // 128, n // 8), torch.rand(k // 128, n, generator=g, device=DEV).half() * 0.01
        fresh = lambda: torch.randn(m, k, generator=g, device=DEV).half()

        def gemm(x):
            with ops.knob("APHRO_WNA16_LARGE_8PHASE", 1):    # (the stream-K kernel also where the row tile would be as good)
                return ops._wna16_large(x, qw, qz, sc, None, 1)
    else:
        w = torch.randn(n, k, generator=g, device=DEV).to(torch.float8_e4m3fn)
        one = torch.ones(1, device=DEV)
        fresh = lambda: torch.randn(m, k, generator=g, device=DEV).to(torch.float8_e4m3fn)
        gemm = lambda x: ops.cutlass_scaled_mm(x, w.t(), one, one, torch.bfloat16)
    a = fresh()
    gemm(a)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = gemm(a)
    for _ in range(5):
        a.copy_(fresh())
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, gemm(a))
