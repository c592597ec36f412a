"""Prompt GEMMs whose tiles the workgroups divide evenly (no tile is cut, no flag is cleared or read) beside ones that cut tiles: whole numbers,
equal to the product, in a scratch that holds any words, and again when a captured graph is replayed."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"
# rows, columns, K: 256 and 512 tiles of 256 x 256 (the last rows whole or ragged), then tiles that are cut
SHAPES = [(4096, 4096, 512), (4000, 4096, 2048), (8192, 4096, 2048), (4096, 4352, 2048), (3000, 4096, 512)]


def replayed(call, out, ws):
    """The eager result, then three replays of its graph, the scratch filled with ones (as floats and flags) before each."""
    ws.fill_(1)
    call()
    got = [out.clone()]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for _ in range(3):
        ws.fill_(1)
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got.append(out.clone())
    return got


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_fp8(m, n, k):
    from aphrodite_engine_amd import _lib
    lib = _lib.lib()
    g = torch.Generator(device=DEV).manual_seed(m + n)
    a, b = (torch.randint(-1, 2, (r, k), generator=g, device=DEV).half() for r in (m, n))
    one = torch.ones(1, device=DEV)
    a8, b8 = a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn)
    want = a @ b.t()                                     # sums below 2048: whole numbers in either type
    out = torch.empty(m, n, dtype=torch.float16, device=DEV)
    ws = torch.empty(lib.aphro_scaled_mm_fp8_large_workspace_bytes(m, n, k) // 4, dtype=torch.int32, device=DEV)

    def call():
        _lib.check(lib.aphro_scaled_mm_fp8_large(out.data_ptr(), a8.data_ptr(), b8.data_ptr(), one.data_ptr(), one.data_ptr(), None, ws.data_ptr(),
                                                 4 * ws.numel(), m, n, k, 0, 0, _lib.F16, torch.cuda.current_stream().cuda_stream), "gemm")

    for got in replayed(call, out, ws):
        assert torch.equal(got, want)


@pytest.mark.parametrize("m,n,k", [(5120, 4096 * 4, 512), (8192, 4096, 2048), (5120, 4096, 2048), (6145, 4096, 512)])
def test_int4(m, n, k):
    from aphrodite_engine_amd import _lib
    lib = _lib.lib()
    g = torch.Generator(device=DEV).manual_seed(m + k)
    a = torch.randint(-1, 2, (m, k), generator=g, device=DEV).half()
    w8 = torch.randint(7, 10, (k // 8, n), generator=g, device=DEV)       # eight rows alike, whatever their order in the word
    qw = (w8 * 0x11111111).to(torch.int32)            # (wraps: the top nibble may be 8 or 9)
    qz = torch.full((k // 128, n // 8), 0x77777777, dtype=torch.int32, device=DEV)      # zero points of 7, stored less one
    sc = torch.ones(k // 128, n, dtype=torch.float16, device=DEV)
    want = a @ (w8 - 8).repeat_interleave(8, 0).half()
    out = torch.empty(m, n, dtype=torch.float16, device=DEV)
    ws = torch.empty(lib.aphro_wna16_gemm_large_workspace_bytes(m, n, k, k // 128, _lib.F16) // 4 + 1, dtype=torch.int32, device=DEV)

    def call():
        _lib.check(lib.aphro_wna16_gemm_large(a.data_ptr(), qw.data_ptr(), qz.data_ptr(), sc.data_ptr(), out.data_ptr(), ws.data_ptr(), 4 * ws.numel(),
                                              m, n, k, k // 128, k, 1, _lib.F16, torch.cuda.current_stream().cuda_stream), "gemm")

    for got in replayed(call, out, ws):
        assert torch.equal(got, want)
