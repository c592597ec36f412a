"""The forms of the FP8 prompt product, on whole numbers whose sums are exact in fp32, so that every form and every order of slices gives the same
bits: tiles that fill the CUs, tiles left over in one to four slices, few tiles, K slices, stream-K ranges, short K, ragged rows and columns."""
import pytest
import torch

from aphrodite_engine_amd import _custom_ops as ops, _lib

pytestmark = pytest.mark.gpu


# (rows, columns, k)
SIZES = [(260, 28672, 2048), (1100, 28672, 2048), (1340, 8192, 2176), (2100, 8192, 4096), (520, 4096, 14336), (700, 4096, 14336), (1340, 4096, 14336),
         (5000, 4096, 2048), (520, 6144, 4096), (900, 6144, 4096), (3000, 6144, 4096), (430, 4096, 4096), (193, 4096, 4096), (1100, 4096, 4096), (200, 1152, 4096),
         (4096, 8192, 1024), (2500, 8192, 512), (1500, 28672, 1024), (8192, 1024, 512), (700, 384, 2048),
         # fewer K tiles than workgroups, a K of one tile, one tile in all
         (4096, 1024, 128), (2048, 1024, 256), (4096, 512, 384), (1024, 4096, 256), (256, 256, 2048), (7, 128, 128), (300, 512, 2048)]


@pytest.mark.parametrize("m,n,k", SIZES)
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_exact_sums(m, n, k, dtype):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-2, 3, (m, k), generator=g, device="cuda").to(torch.float8_e4m3fn)
    b = torch.randint(-2, 3, (n, k), generator=g, device="cuda").to(torch.float8_e4m3fn)
    sa = torch.rand(m, generator=g, device="cuda") + 0.5
    sb = torch.rand(n, generator=g, device="cuda") + 0.5
    lib = _lib.lib()
    out = torch.empty(m, n, dtype=dtype, device="cuda")
    ws = torch.empty(lib.aphro_scaled_mm_fp8_large_workspace_bytes(m, n, k) + 16, dtype=torch.uint8, device="cuda")
    want = (sa[:, None] * (sb[None, :] * (a.float() @ b.float().t()))).to(dtype)      # (sums below 4 k < 2^24: exact in any order)
    for _ in range(2):
        out.fill_(float("nan"))
        ws.fill_(0x7f)
        _lib.check(lib.aphro_scaled_mm_fp8_large(out.data_ptr(), a.data_ptr(), b.data_ptr(), sa.data_ptr(), sb.data_ptr(), None, ws.data_ptr(), ws.numel(), m, n, k,
                                                 1, 1, _lib.BF16 if dtype == torch.bfloat16 else _lib.F16, torch.cuda.current_stream().cuda_stream))
        assert torch.equal(out, want)


def test_captured_slices_replay():
    g = torch.Generator(device="cuda").manual_seed(1)
    a = torch.randint(-2, 3, (520, 14336), generator=g, device="cuda").to(torch.float8_e4m3fn)
    b = torch.randint(-2, 3, (4096, 14336), generator=g, device="cuda").to(torch.float8_e4m3fn)
    one = torch.ones(1, device="cuda")
    run = lambda: ops.cutlass_scaled_mm(a, b.t(), one, one, torch.bfloat16)
    want = run()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = run()
    for _ in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want) and torch.equal(run(), want)


# (rows that the workspace is sized for, rows, columns, k): the form of the most rows needs less than that of the fewer, or nothing
@pytest.mark.parametrize("most,m,n,k", [(2048, 430, 4096, 4096), (2688, 1281, 6144, 4096), (640, 257, 22016, 4096), (895, 300, 4096, 4096),
                                        (1552, 1300, 4224, 8192), (5392, 3000, 4224, 4096)])
def test_a_workspace_for_many_rows_serves_fewer(most, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = torch.randint(-2, 3, (m, k), generator=g, device="cuda").to(torch.float8_e4m3fn)
    b = torch.randint(-2, 3, (n, k), generator=g, device="cuda").to(torch.float8_e4m3fn)
    one = torch.ones(1, device="cuda")
    lib = _lib.lib()
    out = torch.empty(m, n, dtype=torch.bfloat16, device="cuda")
    ws = torch.full((lib.aphro_scaled_mm_fp8_large_workspace_bytes(most, n, k),), 0x7f, dtype=torch.uint8, device="cuda")
    _lib.check(lib.aphro_scaled_mm_fp8_large(out.data_ptr(), a.data_ptr(), b.data_ptr(), one.data_ptr(), one.data_ptr(), None, ws.data_ptr(), ws.numel(), m, n, k,
                                             0, 0, _lib.BF16, torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out, (a.float() @ b.float().t()).to(torch.bfloat16))
