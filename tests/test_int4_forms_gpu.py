"""The forms of the int4 prompt product and of the W8A16 one beside them, on whole numbers whose sums are exact, in a scratch that holds any words: tiles
that fill the CUs, tiles left over in one to four slices, in one pass and in two, the tile of fewer rows, equal ranges, ragged last rows; again when
a captured graph is replayed."""
import pytest
import torch

from aphrodite_engine_amd import _custom_ops as ops, _lib
from test_whole_tile_gemm_gpu import replayed

pytestmark = pytest.mark.gpu
DEV = "cuda"


def weights(n, k, g):
    w8 = torch.randint(7, 10, (k // 8, n), generator=g, device=DEV)       # eight rows alike, whatever their order in the word
    return (w8 * 0x11111111).to(torch.int32), (w8 - 8).repeat_interleave(8, 0).half()


# rows, columns, k; passes: None the plan's, else forced
@pytest.mark.parametrize("m,n,k,passes", [(520, 28672, 2048, None), (1600, 28672, 2048, 0), (1600, 28672, 2048, 1), (2048, 16384, 2048, 0), (5000, 4096, 2048, None),
                                          (5000, 4096, 2048, 0), (6500, 4096, 2176, None), (3072, 6144, 2048, None), (3071, 6144, 2048, None), (3000, 4096, 2048, 0),
                                          (1340, 6144, 2048, 0), (4100, 4096, 2048, 1), (900, 8192, 2048, None), (4096, 4096, 512, 0), (1100, 28672, 512, None)])
def test_int4(m, n, k, passes):
    lib = _lib.lib()
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a = torch.randint(-1, 2, (m, k), generator=g, device=DEV).half()
    qw, w = weights(n, k, g)
    qz = torch.full((k // 128, n // 8), 0x77777777, dtype=torch.int32, device=DEV)      # zero points of 7, stored less one
    sc = torch.ones(k // 128, n, dtype=torch.float16, device=DEV)
    want = a @ w                                            # sums within 2176: rounded once in either
    out = torch.empty(m, n, dtype=torch.float16, device=DEV)

    def run():
        ws = torch.empty(lib.aphro_wna16_gemm_large_workspace_bytes(m, n, k, k // 128, _lib.F16) // 4 + 1, dtype=torch.int32, device=DEV)

        def call():
            _lib.check(lib.aphro_wna16_gemm_large(a.data_ptr(), qw.data_ptr(), qz.data_ptr(), sc.data_ptr(), out.data_ptr(), ws.data_ptr(), 4 * ws.numel(),
                                                  m, n, k, k // 128, k, 1, _lib.F16, torch.cuda.current_stream().cuda_stream), "gemm")
        for got in replayed(call, out, ws):
            assert torch.equal(got, want)
    if passes is None:
        run()
    else:
        with ops.knob("APHRO_WNA16_LARGE_TWO_PASS", passes):
            run()


@pytest.mark.parametrize("m,n,k", [(900, 12288, 2048), (2100, 4096, 2048), (4096, 4096, 2048)])
def test_w8a16_clears_its_flags(m, n, k):
    lib = _lib.lib()
    g = torch.Generator(device=DEV).manual_seed(m)
    a, b = (torch.randint(-1, 2, (r, k), generator=g, device=DEV).half() for r in (m, n))
    b8, one = b.to(torch.float8_e4m3fn), torch.ones(1, device=DEV)
    want = a @ b.t()
    out = torch.empty(m, n, dtype=torch.float16, device=DEV)
    ws = torch.empty(lib.aphro_fp8_w8a16_gemm_large_workspace_bytes(m, n, k, _lib.F16) // 4 + 1, dtype=torch.int32, device=DEV)

    def call():
        _lib.check(lib.aphro_fp8_w8a16_gemm_large(out.data_ptr(), a.data_ptr(), b8.data_ptr(), one.data_ptr(), None, ws.data_ptr(), 4 * ws.numel(), m, n, k, k, 0,
                                                  _lib.F16, torch.cuda.current_stream().cuda_stream), "gemm")
    for got in replayed(call, out, ws):
        assert torch.equal(got, want)


# (rows that the workspace is sized for, rows, columns, k, groups): the most rows ask for fewer slabs than the fewer, or none; 65 to 128 float16 rows
# keep their own form
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("most,m,n,k,groups", [(200, 65, 6144, 4096, 1), (256, 128, 6144, 4096, 1), (300, 150, 4096, 4096, 1), (300, 257, 4096, 4096, 1), (257, 129, 4096, 11008, 86),
                                               (257, 100, 4096, 11008, 86), (1024, 200, 6144, 4096, 32)])
def test_a_workspace_for_other_rows_serves_with_fewer_slices(most, m, n, k, groups, dtype):
    lib, dt = _lib.lib(), _lib.F16 if dtype == torch.float16 else _lib.BF16
    g = torch.Generator(device=DEV).manual_seed(m + n + k)
    a = torch.randint(-1, 2, (m, k), generator=g, device=DEV).to(dtype)
    qw, w = weights(n, k, g)
    qz = torch.full((groups, n // 8), 0x77777777, dtype=torch.int32, device=DEV)
    sc = torch.ones(groups, n, dtype=dtype, device=DEV)
    size = lambda rows: lib.aphro_wna16_gemm_large_workspace_bytes(rows, n, k, groups, dt)
    assert size(most) < size(m)
    ws = torch.full((size(most) + 256,), 0x7f, dtype=torch.uint8, device=DEV)        # (256 bytes that no call may write)
    out = torch.empty(m, n, dtype=dtype, device=DEV)
    _lib.check(lib.aphro_wna16_gemm_large(a.data_ptr(), qw.data_ptr(), qz.data_ptr(), sc.data_ptr(), out.data_ptr(), ws.data_ptr(), ws.numel() - 256, m, n, k,
                                          groups, k, 1, dt, torch.cuda.current_stream().cuda_stream), "gemm")
    assert torch.equal(out, (a.float() @ w.float()).to(dtype)) and bool((ws[-256:] == 0x7f).all())
