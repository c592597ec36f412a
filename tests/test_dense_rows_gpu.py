"""The few-rows 16-bit product against torch in 64 bits: row tiles and their remainders, ragged and narrow column counts, K in one piece
and split, bias, fp32 results, gated activations, strided operands; what it does not serve goes to torch."""
import pytest
import torch
from torch.nn import functional as F

from aphrodite_engine_amd import _custom_ops as ops

pytestmark = pytest.mark.gpu
U = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}      # half a unit in the last place, relative


def _operands(m, n, k, dtype, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(m, k, generator=g, device="cuda").to(dtype)
    w = (torch.randn(n, k, generator=g, device="cuda") * k ** -0.5).to(dtype)
    return x, w


def _close(got, want, dtype, k):
    # one rounding to the type, and fp32 sums of k products whose terms' sizes add up to about sqrt(k) times the result's
    bound = U[dtype] * want.abs() + k * 2.0 ** -24 * 4.0
    assert bool(((got.double() - want).abs() <= bound).all())


# (rows, columns, k): every row tile, its first and last row; tiles of 64 and 128 columns with remainders; K split and not, uneven slices
SHAPES = [(1, 8, 64), (1, 4096, 11008), (16, 2048, 5632), (17, 2056, 832), (32, 6144, 4096), (33, 72, 1024), (48, 11264, 512), (49, 20552, 256),
          (64, 30736, 320), (65, 1000, 4096), (96, 11272, 256), (97, 4104, 11008), (128, 22016, 256), (129, 2048, 7680), (160, 65544, 128),
          (177, 22024, 192), (192, 520, 2112), (192, 65536, 64),
          # one workgroup a CU from 129 rows on; few long slices of 128 columns; more 128-column tiles than CUs
          (150, 18952, 192), (140, 8328, 1024), (70, 10248, 1280), (100, 10248, 2048), (100, 37896, 64), (180, 37896, 128), (65, 62008, 64)]


@pytest.mark.parametrize("m,n,k", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_product(m, n, k, dtype):
    x, w = _operands(m, n, k, dtype)
    want = x.double() @ w.double().t()
    got = ops.dense_rows(x, w)
    assert got is not None and got.dtype == dtype
    _close(got, want, dtype, k)
    wide = ops.dense_rows(x, w, f32=True)
    assert wide.dtype == torch.float32 and torch.equal(wide, got.float())
    assert torch.equal(got, ops.dense_rows(x, w))                # slices are added in order


@pytest.mark.parametrize("m,ff,k", [(1, 8, 64), (20, 5632, 2048), (31, 56, 640), (50, 11008, 256), (64, 1032, 4096), (100, 344, 2048), (192, 11008, 192)])
@pytest.mark.parametrize("act", [0, 1])
def test_gated(m, ff, k, act):
    x, w = _operands(m, 2 * ff, k, torch.bfloat16, 1)
    y = x.double() @ w.double().t()
    a = F.silu(y[:, :ff]) if act == 0 else F.gelu(y[:, :ff], approximate="tanh")
    want = a * y[:, ff:]
    buf = torch.full((m, ff + 24), 7.0, dtype=torch.bfloat16, device="cuda")
    got = ops.dense_rows(x, w, act=act, out=buf[:, 8:8 + ff])
    assert got is not None and got.data_ptr() == buf[:, 8:].data_ptr()
    # the sums' error (4 k 2^-24, as above) passes each factor; the activations' slopes stay below 1.2
    bound = U[torch.bfloat16] * want.abs() + k * 2.0 ** -22 * (1.2 * y[:, ff:].abs() + a.abs()) + 1e-6 * (1 + y[:, ff:].abs())
    assert bool(((got.double() - want).abs() <= bound).all())
    assert bool((buf[:, :8] == 7).all()) and bool((buf[:, 8 + ff:] == 7).all())


@pytest.mark.parametrize("m,n,k", [(5, 2048, 2048), (40, 11264, 256), (70, 65536, 64)])
def test_bias_and_strides(m, n, k):
    x, w = _operands(m, n, k, torch.bfloat16, 2)
    bias = torch.randn(n, device="cuda").to(torch.bfloat16)
    wide_x = torch.full((m, k + 72), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide_x[:, 64:64 + k] = x
    wide_w = torch.full((n + 1, k + 8), float("nan"), dtype=torch.bfloat16, device="cuda")
    wide_w[:n, :k] = w
    got = ops.dense_rows(wide_x[:, 64:64 + k], wide_w[:n, :k], bias)
    assert got is not None
    _close(got, x.double() @ w.double().t() + bias.double(), torch.bfloat16, k)


def test_graph_replays():
    x, w = _operands(24, 2048, 5632, torch.bfloat16, 3)
    want = ops.dense_rows(x, w).clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.dense_rows(x, w)
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, want)


def test_other_forms_go_to_torch():
    x, w = _operands(8, 128, 128, torch.bfloat16, 4)
    assert ops.dense_rows(x.float(), w.float()) is None
    assert ops.dense_rows(x.repeat(25, 1), w) is None            # 200 rows
    assert ops.dense_rows(x[:, 1:65], w[:, 1:65]) is None        # not 16-byte aligned
    assert ops.dense_rows(x[:, :100], w[:, :100]) is None        # K not a multiple of 64
    assert ops.dense_rows(x, w[:100]) is None                    # N not a multiple of 8
    assert ops.dense_rows(x[:1].expand(8, -1), w) is None        # rows on top of one another
    assert ops.dense_rows(x.t().contiguous().t(), w) is None
    assert ops.dense_rows(x.clone().requires_grad_(), w) is None
    assert ops.dense_rows(x.cpu(), w.cpu()) is None
    for a, b in ((x[:, :100], w[:, :100]), (x.float(), w.float()), (x.view(2, 4, 128), w), (x.cpu(), w.cpu())):
        assert torch.equal(ops.dense_linear(a, b), F.linear(a, b))
    y = torch.func.vmap(lambda r: ops.dense_linear(r, w))(x.view(4, 2, 128))
    assert torch.allclose(y.reshape(8, 128).float(), F.linear(x, w).float(), rtol=2e-2, atol=2e-2)


def test_forward_mode_keeps_its_tangent():
    x, w = _operands(8, 128, 128, torch.bfloat16, 5)
    tx, tw = _operands(8, 128, 128, torch.bfloat16, 6)
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual
        unpack = torch.autograd.forward_ad.unpack_dual
        for f in (ops.dense_linear, ops.dense_logits):
            assert torch.equal(unpack(f(dual(x, tx), w)).tangent.float(), F.linear(tx, w).float())
            assert torch.equal(unpack(f(x, dual(w, tw))).tangent.float(), F.linear(x, tw).float())
    assert ops.dense_rows(x, w) is not None


def test_autocast_chooses_the_type():
    x, w = _operands(8, 128, 128, torch.bfloat16, 7)
    with torch.autocast("cuda", dtype=torch.float16):
        got = ops.dense_linear(x, w)
        assert got.dtype == torch.float16 and torch.equal(got, F.linear(x, w))
        with torch.autocast("cuda", enabled=False):
            assert ops.dense_linear(x, w).dtype == torch.bfloat16


@pytest.mark.parametrize("m,n,k", [(100, 28672, 4096), (70, 12288, 4096)])
def test_wide_weights_go_to_torch(m, n, k):
    x, w = _operands(m, n, k, torch.bfloat16, 8)
    assert torch.equal(ops.dense_linear(x, w), F.linear(x, w))
    assert torch.equal(ops.dense_linear(x[:40], w), ops.dense_rows(x[:40], w))
