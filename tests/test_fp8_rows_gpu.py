"""The FP8 product of 33 to 192 rows: its row and column tiles and their remainders, K in one piece and split, scalar and vector scales,
bias; raw slabs add up to the same bits.  Operands are eighths up to 15 / 8: their products' sums fit fp32 without a rounding, so that results
are compared bit by bit."""
import pytest
import torch

from aphrodite_engine_amd import _custom_ops as ops
from aphrodite_engine_amd import _lib

pytestmark = pytest.mark.gpu

SHAPES = [(33, 16, 128), (48, 6144, 4096), (49, 4096, 14336), (64, 28672, 512), (65, 1040, 2048), (96, 10304, 1024), (97, 4096, 4096),
          (128, 20496, 256), (150, 6144, 4096), (160, 4096, 14336), (161, 28672, 384), (192, 528, 8192), (192, 65552, 128),
          # one workgroup a CU from 129 rows on; few long slices of 128 columns; more 128-column tiles than CUs
          (129, 6144, 4096), (150, 18960, 256), (140, 8336, 1024), (100, 10256, 4096), (100, 37904, 128), (180, 37904, 256)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("vector", [False, True])
def test_rows(m, n, k, dtype, vector):
    g = torch.Generator(device="cuda").manual_seed(m + n + k)
    a = (torch.randint(-15, 16, (m, k), generator=g, device="cuda") / 8).to(torch.float8_e4m3fn)
    w = (torch.randint(-15, 16, (n, k), generator=g, device="cuda") / 8).to(torch.float8_e4m3fn)
    sa = torch.rand(m if vector else 1, 1, generator=g, device="cuda") * 0.02 + 0.01
    sb = torch.rand(n if vector else 1, generator=g, device="cuda") * 0.02 + 0.01
    bias = torch.randn(n, generator=g, device="cuda").to(dtype) if vector else None
    assert ops.fp8_gemm_ksplit(m, n, k) == _lib.lib().aphro_fp8_gemm_rows_ksplit(m, n, k) > 0
    got = torch.empty(m, n, dtype=dtype, device="cuda")
    split = ops.fp8_gemm_ksplit(m, n, k)
    ws = torch.empty(split * m * n, dtype=torch.float32, device="cuda")
    rc = _lib.lib().aphro_scaled_mm_fp8(got.data_ptr(), a.data_ptr(), w.data_ptr(), sa.data_ptr(), sb.data_ptr(), None if bias is None else bias.data_ptr(),
                                        ws.data_ptr(), ws.numel() * 4, m, n, k, int(vector), int(vector), _lib.F16 if dtype == torch.float16 else _lib.BF16,
                                        torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    exact = (a.double() @ w.double().t()).float()
    scaled = sa * (sb * exact)
    want = (scaled if bias is None else scaled + bias.float()).to(dtype)
    assert torch.equal(got, want)
    slabs = ops.scaled_mm_fp8_slabs(a, w.t())
    assert slabs.shape == (split, m, n) and torch.equal(slabs.sum(0), exact)
    assert torch.equal(got, ops.cutlass_scaled_mm(a, w.t(), sa, sb, dtype, bias)) or not (m <= 64 or _lib.lib().aphro_fp8_gemm_rows_preferred(m, n, k))


def test_not_served():
    for m, n, k in ((32, 4096, 4096), (193, 4096, 4096), (64, 4096, 4032), (64, 4104, 4096)):
        assert _lib.lib().aphro_fp8_gemm_rows_ksplit(m, n, k) == 0


@pytest.mark.parametrize("kv", ["auto", "fp8"])
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("nslab,rows", [(1, True), (5, True), (9, False)])
def test_rope_cache_of_scaled_slabs(kv, dtype, nslab, rows):
    """Scales over raw slabs: the bits of the scaled sums handed over in 16 bits."""
    g = torch.Generator(device="cuda").manual_seed(nslab)
    T, H, G, d, block = 37, 8, 2, 128, 16
    n = (H + 2 * G) * d
    slabs = torch.randn(nslab, T, n, generator=g, device="cuda") * 20
    sa = torch.rand(T, 1, generator=g, device="cuda") * 0.1 if rows else None
    sb = torch.rand(n, generator=g, device="cuda") * 0.1
    total = slabs[0].clone()
    for s in slabs[1:]:
        total += s
    qkv = ((sb * total) if sa is None else sa * (sb * total)).to(dtype)
    cos_sin = torch.randn(T, d, generator=g, device="cuda").to(dtype)
    slots = torch.randperm(64, generator=g, device="cuda")[:T]
    results = []
    for args in ((None, slabs, dict(row_scale=sa, col_scale=sb)), (qkv, None, {})):
        kind, x = (torch.uint8, 16) if kv == "fp8" else (dtype, 8)
        k = torch.zeros(4, G, d // x, block, x, dtype=kind, device="cuda")
        v = torch.zeros(4, G, d, block, dtype=kind, device="cuda")
        q = ops.rope_cache(args[0], args[1], None, cos_sin, True, k, v, slots, H, G, d, kv, 1.0, 1.0, **args[2])
        results.append((q, k, v))
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("m", [65, 100, 192, 300])
def test_scales_of_another_length_are_refused(m):
    a, w = torch.zeros(m, 256, device="cuda").to(torch.float8_e4m3fn), torch.zeros(512, 256, device="cuda").to(torch.float8_e4m3fn)
    one = lambda n: torch.ones(n, device="cuda")
    for sa, sb in ((one(m - 1), one(512)), (one(m + 1), one(1)), (one(2), one(1)), (one(m), one(511)), (one(1), one(2))):
        with pytest.raises(RuntimeError, match="scale_a must have 1 or M elements"):
            ops.cutlass_scaled_mm(a, w.t(), sa, sb, torch.bfloat16)
    assert not ops.cutlass_scaled_mm(a, w.t(), one(m), one(512), torch.bfloat16).any()
