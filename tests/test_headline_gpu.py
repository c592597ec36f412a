"""BASELINE.json configs[1] (Llama-3-8B GPTQ 4-bit g128, bs 32) at its REAL shapes against the ORACLE.

VERDICT r1 ("What's weak" #1): the kernel instantiations the bench times -- wna16_gemm_kernel<Half,4,2,{8,7,4,2}>,
the packed-activation / split-K-slab / SiluAndMul-epilogue entry points, the fused decode layer -- were checked at
full size only against this repo's own dequant kernel.  Here every one of them is compared with oracle.quant (pinned
by the reference's own CUDA kernels, tests/test_oracle_golden.py::test_gptq_*reference*) on the four projection
shapes at M = 1 and M = 32, and a 2-layer Llama-3-8B-geometry decode step through forward_decode_fused is compared
with a layer composed from oracle functions only."""
import dataclasses

import numpy as np
import pytest
import torch

from oracle import attention as oa
from oracle import quant as oq

pytestmark = pytest.mark.gpu
DEV = "cuda"

SHAPES = [(4096, 6144), (4096, 4096), (4096, 28672), (14336, 4096)]     # qkv, o, gate_up, down (tests/benchmarks/kernels/weight_shapes.py:11-48)


@pytest.fixture(scope="module")
def ops():
    if not torch.cuda.is_available():
        pytest.fail("GPU tests need a visible MI355X (torch.cuda.is_available() is False)")
    from aphrodite_engine_amd import _custom_ops, _lib
    _lib.lib()
    return _custom_ops


def t(x, dtype=None):
    out = torch.from_numpy(np.ascontiguousarray(x)).to(DEV)
    return out.to(dtype) if dtype is not None else out


def unpack_a(packed, M, K):
    """numpy inverse of the fragment-major layout (include/aphrodite_mi355x.h)."""
    mt = (M + 15) // 16
    p = packed.cpu().numpy().view(np.uint16)[: (K // 128) * 4 * mt * 64 * 8].reshape(K // 128, 4, mt, 4, 16, 8)
    return p.transpose(2, 4, 0, 3, 1, 5).reshape(mt * 16, K)[:M]


_CASES = {}


def case(K, N):
    """Random AutoGPTQ-v1 tensors of the shape, their exllama-shuffled form, activations and the fp64 oracle result."""
    if (K, N) not in _CASES:
        rng = np.random.default_rng(K * 7 + N)
        G = K // 128
        qweight = rng.integers(0, 2 ** 32, size=(K // 8, N), dtype=np.uint32).view(np.int32)
        qzeros = rng.integers(0, 2 ** 32, size=(G, N // 8), dtype=np.uint32).view(np.int32)
        scales = (rng.uniform(0.75, 1.25, size=(G, N)) / (4.6 * np.sqrt(K))).astype(np.float16)
        a = rng.standard_normal((32, K)).astype(np.float16)
        shuf = oq.gptq_shuffle(qweight)
        ref = oq.gptq_gemm(a, shuf, qzeros, scales, None, True)           # fp64 [32, N]
        _CASES[(K, N)] = (shuf, qzeros, scales, a, ref)
    return _CASES[(K, N)]


@pytest.mark.parametrize("M", [1, 32])
@pytest.mark.parametrize("K,N", SHAPES)
def test_config1_gptq_gemm_vs_oracle(ops, K, N, M):
    """ops.gptq_gemm (the schema-level op: pack + fast kernel + split-K reduce) at the bench's shapes."""
    shuf, qzeros, scales, a, ref = case(K, N)
    ref = ref[:M]
    empty = torch.empty(0, dtype=torch.int32, device=DEV)
    got = ops.gptq_gemm(t(a[:M]), t(shuf), t(qzeros), t(scales), empty, True, 4)
    g = got.float().cpu().numpy()
    assert np.abs(g - ref).mean() / np.abs(ref).mean() < 0.04            # the reference's Marlin-family bar
    np.testing.assert_allclose(g, ref, rtol=2e-3, atol=2e-3 * np.abs(ref).max())
    assert torch.equal(got, ops.gptq_gemm(t(a[:M]), t(shuf), t(qzeros), t(scales), empty, True, 4))   # no atomics


@pytest.mark.parametrize("M", [1, 32])
@pytest.mark.parametrize("K,N", SHAPES)
def test_config1_packed_and_slab_entry_points_vs_oracle(ops, K, N, M):
    """The entry points the decode fast path (and bench.py's roofline leg) launches: fragment-major activations,
    f16 output and raw fp32 split-K slabs for a fused consumer."""
    shuf, qzeros, scales, a, ref = case(K, N)
    ref = ref[:M]
    pk = ops.wna16_pack_a(t(a[:M]))
    np.testing.assert_array_equal(unpack_a(pk, M, K), a[:M].view(np.uint16))
    y = ops.wna16_gemm_packed(pk, M, K, t(shuf), t(qzeros), t(scales), 1, partials=False)
    np.testing.assert_allclose(y.float().cpu().numpy(), ref, rtol=2e-3, atol=2e-3 * np.abs(ref).max())
    slabs, ks = ops.wna16_gemm_packed(pk, M, K, t(shuf), t(qzeros), t(scales), 1, partials=True)
    assert slabs.shape == (ks, M, N) and ks == ops.wna16_ksplit(M, N, K, K // 128) and ks >= 1
    s = slabs.double().sum(0).cpu().numpy()
    np.testing.assert_allclose(s, ref, rtol=1e-4, atol=2e-5 * np.abs(ref).max())     # fp32 accumulate vs fp64
    # the f16 output is the rounded slab sum (same kernel, same order)
    assert torch.equal(y, slabs.sum(0).to(torch.float16)) or ks > 2   # (a + b) + c order of torch.sum may differ beyond 2 slabs


@pytest.mark.parametrize("M", [1, 32])
def test_config1_gate_up_silu_epilogue_vs_oracle(ops, M):
    """gate_up with interleaved (gate_j, up_j) columns + SiluAndMul + pack in the GEMM epilogue, against
    silu_and_mul(round16(oracle GEMM)) (activation_kernels.cu:12-60 on the fp16-rounded projection)."""
    K, N = 4096, 28672
    shuf, qzeros, scales, a, ref = case(K, N)
    qw_i, qz_i, sc_i = ops.interleave_gate_up(t(shuf), t(qzeros), t(scales))
    act = ops.wna16_gemm_silu_pack(ops.wna16_pack_a(t(a[:M])), M, K, qw_i, qz_i, sc_i, 1)
    got = unpack_a(act, M, N // 2).view(np.float16).astype(np.float64)
    gu = ref[:M].astype(np.float16)                                       # the kernel rounds the projection first
    d = N // 2
    gate = gu[:, :d].astype(np.float64)
    silu = (gate / (1.0 + np.exp(-gate))).astype(np.float16).astype(np.float64)   # silu is rounded, then multiplied
    want = (silu * gu[:, d:].astype(np.float64)).astype(np.float16).astype(np.float64)
    np.testing.assert_allclose(got, want, rtol=4e-3, atol=4e-3 * np.abs(want).max())
    # and the oracle's own (unrounded) silu_and_mul is within fp16 rounding of it
    np.testing.assert_allclose(got, oa.silu_and_mul(ref[:M]), rtol=6e-3, atol=6e-3 * np.abs(want).max())


_DEQ = {}


def dequant32(K, N):
    """fp32 dequantised weight of case(K, N), cached (oracle.quant.gptq_dequant: (q - (z + 1)) * s, exact in fp32)."""
    if (K, N) not in _DEQ:
        shuf, qzeros, scales, _, _ = case(K, N)
        _DEQ[(K, N)] = oq.gptq_dequant(shuf, qzeros, scales, None, shuffled=True)
    return _DEQ[(K, N)]


@pytest.mark.parametrize("M", [65, 256, 2048, 8192])
@pytest.mark.parametrize("K,N", SHAPES)
def test_config1_prefill_sized_gemm_vs_oracle(ops, K, N, M):
    """Prefill-sized M: ops.gptq_gemm dispatches to the hand-written MFMA kernel (csrc/wna16_gemm_large.hip: dequant in
    registers, 32x32x16 MFMA, direct-to-LDS activation tiles, split-K slabs for small grids).
    The whole [M, N] result is produced on the device; 160 rows of it (tile edges, first / last, random) are compared
    with the oracle: every output row depends on its own activation row only."""
    assert ops.wna16_large_ok(M, N, K, K // 128)
    shuf, qzeros, scales, _, _ = case(K, N)
    rng = np.random.default_rng(M + K + N)
    a = rng.standard_normal((M, K)).astype(np.float16)
    empty = torch.empty(0, dtype=torch.int32, device=DEV)
    got = ops.gptq_gemm(t(a), t(shuf), t(qzeros), t(scales), empty, True, 4)
    assert got.shape == (M, N) and got.dtype == torch.float16
    rows = sorted(set([0, 1, 31, 32, 63, 64, 127, 128, 255, 256, 257, M // 2, M - 2, M - 1]) & set(range(M))
                  | set(rng.integers(0, M, size=146).tolist()))
    w = dequant32(K, N)
    ref = a[rows].astype(np.float32) @ w                                  # fp32 BLAS on exact fp32 weights
    g = got[torch.tensor(rows, device=DEV)].float().cpu().numpy()
    assert np.isfinite(g).all()
    assert np.abs(g - ref).mean() / np.abs(ref).mean() < 0.04              # tests/kernels/test_marlin_gemm.py:57-59
    np.testing.assert_allclose(g, ref, rtol=2e-3, atol=2e-3 * np.abs(ref).max())
    # deterministic (fixed-order split-K reduction, no atomics)
    assert torch.equal(got, ops.gptq_gemm(t(a), t(shuf), t(qzeros), t(scales), empty, True, 4))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("K,N", SHAPES)
def test_config1_prefill_two_pass_form_is_the_fused_form_bit_for_bit(ops, K, N, dtype):
    """Round 6: from 6144 rows the W4A16 prefill GEMM dequantises the weights ONCE per call (f16 W^T, the numerics of the in-loop
    dequantisation) and runs the eight-phase schedule with the weights by LDS-DMA (csrc/wna16_gemm_large.hip, WDMA) -- same tile
    order, same MFMA order, same operands: the bits of the fused kernel (which the test above holds against the oracle), at
    8192 rows (default dispatch) and, forced, at a ragged 1000 rows; also the SiluAndMul-epilogue entry point on gate_up."""
    g = torch.Generator(device=DEV).manual_seed(K * 7 + N)
    qw = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 8, N), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    qz = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 128, N // 8), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
    sc = (torch.rand(K // 128, N, generator=g, device=DEV) * 0.01 + 0.005).to(dtype)
    for M in (8192, 1000):
        a = torch.randn(M, K, device=DEV, dtype=dtype, generator=g)
        with ops.knob("APHRO_WNA16_LARGE_TWO_PASS", 0):
            fused = ops._wna16_large(a, qw, qz, sc, None, 1)
        with ops.knob("APHRO_WNA16_LARGE_TWO_PASS", 1):
            two = ops._wna16_large(a, qw, qz, sc, None, 1)
        assert torch.equal(fused.view(torch.int16), two.view(torch.int16)), (M, K, N)
        if M == 8192:
            assert torch.equal(ops._wna16_large(a, qw, qz, sc, None, 1).view(torch.int16), two.view(torch.int16))      # default dispatch
        if N == 28672 and ops.wna16_gemm_large_silu_supported(M, N, K, K // 128):
            with ops.knob("APHRO_WNA16_LARGE_TWO_PASS", 0):
                act_f = ops.wna16_gemm_large_silu(a, qw, qz, sc, 1)
            with ops.knob("APHRO_WNA16_LARGE_TWO_PASS", 1):
                act_t = ops.wna16_gemm_large_silu(a, qw, qz, sc, 1)
            assert torch.equal(act_f.view(torch.int16), act_t.view(torch.int16))


def test_prefill_sized_gemm_bf16_act_order_and_odd_rows(ops):
    """bf16 activations / scales (widened to f16 with saturation), act-order gather, M not a multiple of any tile,
    group size 64, against the oracle."""
    rng = np.random.default_rng(77)
    K, N, G, M = 1024, 384, 64, 333
    w_ = (rng.standard_normal((K, N)) * 0.02).astype(np.float16)
    _, q, s, zp = oq.quantize_weights(w_, 4, G, zero_points=True)
    perm = rng.permutation(K)
    g_idx = (np.arange(K) // G).astype(np.int32)[perm]                      # row -> group of the SHUFFLED checkpoint rows
    qweight = oq.gptq_pack(q[perm])
    qzeros = oq.gptq_pack_zeros(zp)
    sort = np.argsort(g_idx, kind="stable").astype(np.int32)              # gptq.py:219-221: g_idx becomes the permutation
    shuf = oq.gptq_shuffle(qweight, sort)
    a = (rng.standard_normal((M, K)) * 2).astype(np.float32)
    at = t(a, torch.bfloat16)
    sc = t(s.astype(np.float32), torch.bfloat16)
    got = ops.gptq_gemm(at, t(shuf), t(qzeros), sc, t(sort), True, 4)
    ref = oq.gptq_gemm(at.float().cpu().numpy(), shuf, qzeros, sc.float().cpu().numpy(), sort, True)
    assert got.dtype == torch.bfloat16
    np.testing.assert_allclose(got.float().cpu().numpy(), ref, rtol=1.6e-2, atol=1.6e-2 * np.abs(ref).max())


@pytest.mark.parametrize("M,per_token,per_channel,dtype,with_bias", [
    (65, True, True, torch.bfloat16, False),       # one ragged row tile, K slices (small grid)
    (1000, True, True, torch.float16, True),       # 96 tiles: one workgroup per tile
    (2100, True, True, torch.bfloat16, True),      # 216 tiles: persistent stream-K grid, tiles cut between workgroups
    (2100, False, False, torch.float16, False),    # per-tensor scales
    (8192, True, False, torch.bfloat16, False),    # configs[2] prefill length
])
@pytest.mark.parametrize("K,N", [(4096, 6144), (14336, 4096)])
def test_config2_prefill_sized_fp8_scaled_mm_vs_oracle(ops, K, N, M, per_token, per_channel, dtype, with_bias):
    """configs[2] (FP8 W8A8) at prefill-sized M: cutlass_scaled_mm runs the hand-written MFMA kernel
    (csrc/fp8_gemm_large.hip: v_mfma_scale_f32_32x32x64_f8f6f4, stream-K) instead of torch._scaled_mm
    missing #1.  The result is compared with the oracle (fp64 on the decoded e4m3 values, test_cutlass.py:36-47) on
    160 rows; the whole output must be finite, and a second call must give the same bits (fixed-order fix-up)."""
    from oracle import fp8 as of8
    rng = np.random.default_rng(M + K + N)
    a = t((rng.standard_normal((M, K)) * 2).astype(np.float32)).to(torch.float8_e4m3fn)
    w = t((rng.standard_normal((N, K)) * 2).astype(np.float32)).to(torch.float8_e4m3fn)
    sa = t((rng.random((M, 1) if per_token else (1, )) * 0.1 + 0.01).astype(np.float32))
    sb = t((rng.random((N, 1) if per_channel else (1, )) * 0.1 + 0.01).astype(np.float32))
    bias = t(rng.standard_normal(N).astype(np.float32), dtype) if with_bias else None
    got = ops.cutlass_scaled_mm(a, w.t(), sa, sb, dtype, bias)
    assert got.shape == (M, N) and got.dtype == dtype and torch.isfinite(got.float()).all()
    rows = sorted(set([0, 1, 31, 32, 63, 64, 127, 128, 255, 256, 257, M // 2, M - 2, M - 1]) & set(range(M))
                  | set(rng.integers(0, M, size=146).tolist()))
    ridx = torch.tensor(rows, device=DEV)
    ref = of8.scaled_mm(a[ridx].view(torch.uint8).cpu().numpy(), w.view(torch.uint8).cpu().numpy().T,
                        sa[ridx].cpu().numpy() if per_token else sa.cpu().numpy(), sb.cpu().numpy().reshape(-1),
                        None if bias is None else bias.float().cpu().numpy())
    g = got[ridx].float().cpu().numpy()
    tol = 2e-3 if dtype == torch.float16 else 1.6e-2            # one rounding of the fp32 result to the output type
    np.testing.assert_allclose(g, ref, rtol=tol, atol=tol * np.abs(ref).max())
    assert torch.equal(got, ops.cutlass_scaled_mm(a, w.t(), sa, sb, dtype, bias))


def test_prefill_sized_fp8_scaled_mm_under_graph_capture(ops):
    """The stream-K form clears its flag words with a kernel of its own in front: capture it, replay it twice."""
    g_ = torch.Generator(device=DEV).manual_seed(3)
    M, K, N = 2304, 1024, 6144
    a = torch.randn(M, K, generator=g_, device=DEV).to(torch.float8_e4m3fn)
    w = torch.randn(N, K, generator=g_, device=DEV).to(torch.float8_e4m3fn)
    sa = torch.rand(M, 1, generator=g_, device=DEV) * 0.1 + 0.01
    sb = torch.rand(N, generator=g_, device=DEV) * 0.1 + 0.01
    out = torch.empty(M, N, device=DEV, dtype=torch.bfloat16)
    eager = ops.cutlass_scaled_mm(a, w.t(), sa, sb, torch.bfloat16)
    torch.cuda.synchronize()
    gr = torch.cuda.CUDAGraph()
    with torch.cuda.graph(gr):
        ops.cutlass_scaled_mm(a, w.t(), sa, sb, torch.bfloat16, out=out)
    for _ in range(2):
        out.zero_()
        gr.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,K,N,per_channel,with_bias", [(65, 4096, 6144, True, False), (1000, 14336, 4096, True, True),
                                                          (2100, 4096, 6144, False, False), (8192, 4096, 4096, True, False)])
def test_prefill_sized_fp8_w8a16_vs_oracle(ops, dtype, M, K, N, per_channel, with_bias):
    """W8A16 (fp8_marlin_gemm role) at prefill-sized M: e4m3 weights widened to f16 in registers on the int4 kernel's tile
    machine, scale + bias in the epilogue; 160 rows vs the oracle, whole output finite, bit-identical across calls."""
    from oracle import fp8 as of8
    rng = np.random.default_rng(M + K + N)
    a = t(rng.standard_normal((M, K)).astype(np.float32), dtype)
    w = t((rng.standard_normal((N, K)) * 2).astype(np.float32)).to(torch.float8_e4m3fn)
    sb = t((rng.random(N if per_channel else 1) * 0.1 + 0.01).astype(np.float32))
    bias = t(rng.standard_normal(N).astype(np.float32), dtype) if with_bias else None
    got = ops.fp8_marlin_gemm(a, w, sb, None, 8, M, N, K, bias)
    assert got.shape == (M, N) and got.dtype == dtype and torch.isfinite(got.float()).all()
    rows = sorted(set([0, 1, 31, 32, 63, 64, 127, 128, 255, 256, 257, M // 2, M - 2, M - 1]) & set(range(M))
                  | set(rng.integers(0, M, size=146).tolist()))
    ridx = torch.tensor(rows, device=DEV)
    ref = of8.fp8_w8a16_gemm(a[ridx].float().cpu().numpy(), w.view(torch.uint8).cpu().numpy().T, sb.cpu().numpy())
    if bias is not None:
        ref = ref + bias.float().cpu().numpy()
    tol = 2e-3 if dtype == torch.float16 else 1.6e-2
    np.testing.assert_allclose(got[ridx].float().cpu().numpy(), ref, rtol=tol, atol=tol * np.abs(ref).max())
    assert torch.equal(got, ops.fp8_marlin_gemm(a, w, sb, None, 8, M, N, K, bias))


def _lin_np(lin):
    fp = lin.fast_params()
    assert fp is not None and fp[3] == 1
    return tuple(x.cpu().numpy() for x in fp[:3])


def test_config1_fused_decode_layers_vs_oracle(ops):
    """A decode step through TWO decoder layers of Llama-3-8B geometry (hidden 4096, 32/8 heads, inter 14336, GPTQ
    g128) on the fused fast path -- norm+pack, qkv slabs, rope+cache+attention in one launch, o_proj slabs,
    norm+pack, gate_up with the SiluAndMul epilogue, down slabs -- against the same step composed from ORACLE
    functions only (fp64 math, rounded to fp16 where the reference's kernels store fp16)."""
    _config1_fused_layers_vs_oracle([5, 17, 33, 64], 512)


def test_config1_bs32_ctx1024_fused_decode_layers_vs_oracle(ops):
    """The same composition AT THE BENCHED POINT: batch 32 -- the resident / strip-major GEMM
    forms, the 8-wave attention form -- with contexts around 1024: a ragged mix randint(1, 1100), one sequence exactly
    on a 16-token block edge (1024), its neighbours (1023, 1025), a one-token sequence, and the longest at 1100.
    Tolerances: the reference's own bars for these ops (tests/kernels/test_attention.py:318-326 atol 1e-3 on the
    attention output, test_marlin_gemm.py:57-59 4 % mean relative on the GEMMs); the composed step is held to the
    same end-to-end bound as the small case above."""
    rng = np.random.default_rng(1024)
    lens = [1024, 1023, 1025, 1, 1100, 16, 17] + [int(x) for x in rng.integers(1, 1101, size=25)]
    _config1_fused_layers_vs_oracle(lens, 2048)


def _config1_fused_layers_vs_oracle(lens, max_pos):
    from aphrodite_engine_amd import model as M
    from aphrodite_engine_amd.quantization.gptq import GPTQConfig
    cfg = dataclasses.replace(M.LLAMA3_8B, num_hidden_layers=2, vocab_size=2048, max_position_embeddings=max_pos)
    bs, block = len(lens), 16
    f16 = lambda x: np.asarray(x).astype(np.float16)
    with torch.no_grad():
        m = M.LlamaForCausalLM(cfg, GPTQConfig(4, 128, False), torch.float16)
        m.init_synthetic(torch.device(DEV))
        assert all(l.enable_fused_silu(bs) for l in m.layers)
        meta, pos, nblocks = M.make_decode_metadata(bs, lens, block, DEV)
        ids = torch.randint(0, cfg.vocab_size, (bs, ), device=DEV, generator=torch.Generator(device=DEV).manual_seed(5))
        caches = M.make_kv_caches(cfg, nblocks, block, torch.float16, "auto", DEV, seed=3)
        caches0 = [c.cpu().numpy().copy() for c in caches]
        m.use_fused_decode = True
        assert all(l.fused_decode_ok(bs) for l in m.layers)
        got = m(ids, pos, caches, meta).float().cpu().numpy()

        # ---- the same step from oracle functions ---------------------------------------------------------------
        hkv, hd, hq = cfg.num_key_value_heads, cfg.head_dim, cfg.num_attention_heads
        positions = pos.cpu().numpy()
        slots = meta.slot_mapping.cpu().numpy()
        bt = meta.block_tables.cpu().numpy()
        cos_sin = m.cos_sin.cpu().numpy()
        hidden = f16(m.embed_tokens[ids].cpu().numpy())
        residual = None
        for li, layer in enumerate(m.layers):
            ln1 = layer.input_layernorm.cpu().numpy()
            ln2 = layer.post_attention_layernorm.cpu().numpy()
            if residual is None:
                residual = hidden
                x = f16(oa.rms_norm(hidden, ln1, cfg.rms_norm_eps))
            else:
                x, r = oa.fused_add_rms_norm(hidden, residual, ln1, cfg.rms_norm_eps)
                residual = f16(r)
                x = f16(oa.rms_norm(residual, ln1, cfg.rms_norm_eps))
            qw, qz, sc = _lin_np(layer.qkv_proj)
            qkv = f16(oq.gptq_gemm(x, qw, qz, sc, None, True))
            q, k, v = qkv[:, :hq * hd], qkv[:, hq * hd:(hq + hkv) * hd], qkv[:, (hq + hkv) * hd:]
            q, k = oa.rotary_embedding_neox(positions, q, k, hd, cos_sin)
            q, k = f16(q), f16(k)
            kc_shape, vc_shape = oa.split_kv_cache_shapes(nblocks, hkv, hd, block, 2)
            kc = caches0[li][0].reshape(kc_shape)
            vc = caches0[li][1].reshape(vc_shape)
            oa.reshape_and_cache(k.reshape(bs, hkv, hd), v.reshape(bs, hkv, hd), kc, vc, slots)
            attn = f16(oa.paged_attention_decode(q.reshape(bs, hq, hd), kc, vc, bt, lens, hd ** -0.5)).reshape(bs, hq * hd)
            # the device wrote the same K / V bits into the same slots
            dev_cache = caches[li].cpu().numpy()
            # (rotary differences cancel: the error is a few fp16 ulps of the INPUT magnitude, not of the result)
            kmax = float(np.abs(k.astype(np.float32)).max())
            np.testing.assert_allclose(dev_cache[0].reshape(kc_shape).astype(np.float32), kc.astype(np.float32), atol=4e-3 * kmax, rtol=2e-3)
            np.testing.assert_allclose(dev_cache[1].reshape(vc_shape).astype(np.float32), vc.astype(np.float32), atol=4e-3 * kmax, rtol=2e-3)
            qw, qz, sc = _lin_np(layer.o_proj)
            o = f16(oq.gptq_gemm(attn, qw, qz, sc, None, True))
            x2, r = oa.fused_add_rms_norm(o, residual, ln2, cfg.rms_norm_eps)
            residual = f16(r)
            x2 = f16(oa.rms_norm(residual, ln2, cfg.rms_norm_eps))
            qw, qz, sc = _lin_np(layer.gate_up_proj)
            gu = f16(oq.gptq_gemm(x2, qw, qz, sc, None, True))
            act = f16(oa.silu_and_mul(gu))
            qw, qz, sc = _lin_np(layer.down_proj)
            hidden = f16(oq.gptq_gemm(act, qw, qz, sc, None, True))
        _, r = oa.fused_add_rms_norm(hidden, residual, m.norm.cpu().numpy(), cfg.rms_norm_eps)
        want = oa.rms_norm(f16(r), m.norm.cpu().numpy(), cfg.rms_norm_eps)
    np.testing.assert_allclose(got, want, atol=2e-2, rtol=2e-2)
    assert np.abs(got - want).mean() / np.abs(want).mean() < 4e-3


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M", [33, 48, 64])
def test_decode_fast_path_mid_kernel_forms(ops, M, dtype):
    """33..64 rows on the decode fast path (csrc/wna16_gemm_mid.hip reading the decode kernel's fragment-major
    activations): the gate_up form (SiluAndMul + pack in the epilogue) against the decode kernel's own fused epilogue --
    same packed layout, compared element by element over the valid rows -- and the slab form on the down_proj shape
    against the decode kernel's slabs.  Tolerance: the two kernels round the dequantised weight differently (f16
    (q - z) * s vs exact integers + fp32 scale), ~3e-4 relative."""
    g = torch.Generator(device=DEV).manual_seed(1000 + M)

    def weights(K, N):
        qw = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 8, N), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
        qz = torch.randint(-2 ** 31, 2 ** 31 - 1, (K // 128, N // 8), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)
        sc = (torch.rand(K // 128, N, generator=g, device=DEV) * 0.01 + 0.005).to(dtype)
        return qw, qz, sc

    K, N = 4096, 28672
    qw, qz, sc = weights(K, N)
    a = (torch.randn(M, K, generator=g, device=DEV) * 0.5).to(dtype)
    packed = ops.wna16_pack_a(a)
    assert ops.wna16_gemm_mid_ksplit(M, N, K, K // 128) == 1
    ref = ops.wna16_gemm_silu_pack(packed, M, K, qw, qz, sc, 1).float()
    got = ops.wna16_gemm_mid_silu_pack(packed, M, K, qw, qz, sc, 1).float()
    valid = ops.wna16_pack_a(torch.ones(M, N // 2, device=DEV, dtype=torch.float16)) != 0   # rows < M of the packed layout
    assert valid.sum().item() == M * (N // 2)
    scale = ref[valid].abs().max().item()
    assert scale > 1.0
    assert (got - ref)[valid].abs().max().item() <= (6e-3 if dtype == torch.float16 else 2.5e-2) * scale
    assert (got - ref)[valid].abs().mean().item() <= 4e-4 * scale if dtype == torch.float16 else True

    K2, N2 = 14336, 4096
    qw2, qz2, sc2 = weights(K2, N2)
    a2 = (torch.randn(M, K2, generator=g, device=DEV) * 0.5).to(dtype)
    packed2 = ops.wna16_pack_a(a2)
    ref2 = ops.wna16_gemm_packed(packed2, M, K2, qw2, qz2, sc2, 1, partials=True)[0].sum(0)
    slabs, ks = ops.wna16_gemm_mid_packed(packed2, M, K2, qw2, qz2, sc2, 1, partials=True)
    assert ks == slabs.shape[0] == ops.wna16_gemm_mid_ksplit(M, N2, K2, K2 // 128) and slabs.shape[1:] == (M, N2)
    got2 = slabs.sum(0)
    torch.testing.assert_close(got2, ref2, rtol=0, atol=2e-3 * ref2.abs().max().item())
    again, _ = ops.wna16_gemm_mid_packed(packed2, M, K2, qw2, qz2, sc2, 1, partials=True)
    assert torch.equal(again, slabs)


# ---------------------------------------------------------------------------------------------------------------------
# the 33..64-row decode fast path and the FP8 fused path against the ORACLE (not against
# another HIP kernel)
# ---------------------------------------------------------------------------------------------------------------------
def _oracle_gemm64(K, N, M, seed):
    """64 fresh activation rows and their fp64 oracle product with case(K, N)'s weights (column blocks keep the fp64
    intermediate small)."""
    w32 = dequant32(K, N)
    rng = np.random.default_rng(seed)
    a = (rng.standard_normal((M, K)) * 0.5).astype(np.float16)
    a64 = a.astype(np.float64)
    ref = np.concatenate([a64 @ w32[:, j:j + 2048].astype(np.float64) for j in range(0, N, 2048)], axis=1)
    return a, ref


@pytest.mark.parametrize("M", [33, 48, 64])
def test_config1_fused_forms_vs_oracle_33_to_64_rows(ops, M):
    """configs[3] lives at bs 64: at 33..64 rows the decode step's MLP runs wna16_gemm_mid_kernel's fused forms (gate_up:
    SiluAndMul + pack epilogue, down: fp32 slabs) and, when that is switched off, the decode kernel's own fused forms in
    two 32-row passes.  Both against oracle.quant.gptq_gemm / oracle.attention.silu_and_mul on the REAL gate_up / down
    shapes of configs[1]."""
    K, N = 4096, 28672
    shuf, qzeros, scales, _, _ = case(K, N)
    a, ref = _oracle_gemm64(K, N, M, 4000 + M)
    qw_i, qz_i, sc_i = ops.interleave_gate_up(t(shuf), t(qzeros), t(scales))
    pk = ops.wna16_pack_a(t(a))
    gu = ref.astype(np.float16)                                           # the kernels round the projection first
    d = N // 2
    gate = gu[:, :d].astype(np.float64)
    silu = (gate / (1.0 + np.exp(-gate))).astype(np.float16).astype(np.float64)
    want = (silu * gu[:, d:].astype(np.float64)).astype(np.float16).astype(np.float64)
    assert ops.wna16_gemm_mid_ksplit(M, N, K, K // 128) == 1
    for name, fn in (("mid", ops.wna16_gemm_mid_silu_pack), ("decode", ops.wna16_gemm_silu_pack)):
        act = fn(pk, M, K, qw_i, qz_i, sc_i, 1)
        got = unpack_a(act, M, d).view(np.float16).astype(np.float64)
        np.testing.assert_allclose(got, want, rtol=4e-3, atol=4e-3 * np.abs(want).max(), err_msg=name)
        np.testing.assert_allclose(got, oa.silu_and_mul(ref), rtol=6e-3, atol=6e-3 * np.abs(want).max(), err_msg=name)

    K2, N2 = 14336, 4096
    shuf2, qzeros2, scales2, _, _ = case(K2, N2)
    a2, ref2 = _oracle_gemm64(K2, N2, M, 5000 + M)
    pk2 = ops.wna16_pack_a(t(a2))
    slabs, ks = ops.wna16_gemm_mid_packed(pk2, M, K2, t(shuf2), t(qzeros2), t(scales2), 1, partials=True)
    assert ks == ops.wna16_gemm_mid_ksplit(M, N2, K2, K2 // 128) >= 1 and slabs.shape == (ks, M, N2)
    # the 33..64-row kernel multiplies f16-rounded (q - z) * s weights (the reference's own numerics, q_gemm.cu:1394-1434)
    np.testing.assert_allclose(slabs.double().sum(0).cpu().numpy(), ref2, rtol=2e-3, atol=1e-3 * np.abs(ref2).max())
    slabs_d, ksd = ops.wna16_gemm_packed(pk2, M, K2, t(shuf2), t(qzeros2), t(scales2), 1, partials=True)
    assert slabs_d.shape == (ksd, M, N2)
    # the decode kernel keeps exact integer weights and scales in fp32
    np.testing.assert_allclose(slabs_d.double().sum(0).cpu().numpy(), ref2, rtol=1e-4, atol=2e-5 * np.abs(ref2).max())


class _OracleLinears:
    """fp32 dequantised weights of a model's W4A16 linears, cached per (layer, name); products in fp64."""

    def __init__(self):
        self.w = {}

    def __call__(self, key, lin, x):
        if key not in self.w:
            qw, qz, sc = _lin_np(lin)
            self.w[key] = oq.gptq_dequant(qw, qz, sc, None, shuffled=True)
        w = self.w[key]
        x64 = np.asarray(x).astype(np.float64)
        return np.concatenate([x64 @ w[:, j:j + 2048].astype(np.float64) for j in range(0, w.shape[1], 2048)], axis=1)


def test_config3_batch64_fused_decode_layers_vs_oracle(ops):
    """bs = 64 (configs[3]'s batch) through TWO decoder layers of Llama-3-8B geometry on the fused fast path -- at 33..64 rows
    gate_up and down run wna16_gemm_mid_kernel's fused forms -- against the same step composed from ORACLE functions."""
    from aphrodite_engine_amd import model as M
    from aphrodite_engine_amd.quantization.gptq import GPTQConfig
    cfg = dataclasses.replace(M.LLAMA3_8B, num_hidden_layers=2, vocab_size=2048, max_position_embeddings=512)
    bs, block = 64, 16
    rng = np.random.default_rng(64)
    lens = [int(x) for x in rng.integers(1, 97, size=bs)]
    f16 = lambda x: np.asarray(x).astype(np.float16)
    lin = _OracleLinears()
    with torch.no_grad():
        m = M.LlamaForCausalLM(cfg, GPTQConfig(4, 128, False), torch.float16)
        m.init_synthetic(torch.device(DEV))
        assert all(l.enable_fused_silu(bs) for l in m.layers)
        meta, pos, nblocks = M.make_decode_metadata(bs, lens, block, DEV)
        ids = torch.randint(0, cfg.vocab_size, (bs, ), device=DEV, generator=torch.Generator(device=DEV).manual_seed(6))
        caches = M.make_kv_caches(cfg, nblocks, block, torch.float16, "auto", DEV, seed=4)
        caches0 = [c.cpu().numpy().copy() for c in caches]
        m.use_fused_decode = True
        assert all(l.fused_decode_ok(bs) for l in m.layers)
        l0 = m.layers[0]
        assert ops.wna16_gemm_mid_ksplit(bs, l0.gate_up_proj.out_features, cfg.hidden_size, cfg.hidden_size // 128) == 1
        got = m(ids, pos, caches, meta).float().cpu().numpy()

        hkv, hd, hq = cfg.num_key_value_heads, cfg.head_dim, cfg.num_attention_heads
        positions = pos.cpu().numpy()
        slots = meta.slot_mapping.cpu().numpy()
        bt = meta.block_tables.cpu().numpy()
        cos_sin = m.cos_sin.cpu().numpy()
        hidden = f16(m.embed_tokens[ids].cpu().numpy())
        residual = None
        for li, layer in enumerate(m.layers):
            ln1 = layer.input_layernorm.cpu().numpy()
            ln2 = layer.post_attention_layernorm.cpu().numpy()
            if residual is None:
                residual = hidden
            else:
                _, r = oa.fused_add_rms_norm(hidden, residual, ln1, cfg.rms_norm_eps)
                residual = f16(r)
            x = f16(oa.rms_norm(residual, ln1, cfg.rms_norm_eps))
            qkv = f16(lin((li, "qkv"), layer.qkv_proj, x))
            q, k, v = qkv[:, :hq * hd], qkv[:, hq * hd:(hq + hkv) * hd], qkv[:, (hq + hkv) * hd:]
            q, k = oa.rotary_embedding_neox(positions, q, k, hd, cos_sin)
            q, k = f16(q), f16(k)
            kc_shape, vc_shape = oa.split_kv_cache_shapes(nblocks, hkv, hd, block, 2)
            kc = caches0[li][0].reshape(kc_shape)
            vc = caches0[li][1].reshape(vc_shape)
            oa.reshape_and_cache(k.reshape(bs, hkv, hd), v.reshape(bs, hkv, hd), kc, vc, slots)
            attn = f16(oa.paged_attention_decode(q.reshape(bs, hq, hd), kc, vc, bt, lens, hd ** -0.5)).reshape(bs, hq * hd)
            o = f16(lin((li, "o"), layer.o_proj, attn))
            _, r = oa.fused_add_rms_norm(o, residual, ln2, cfg.rms_norm_eps)
            residual = f16(r)
            x2 = f16(oa.rms_norm(residual, ln2, cfg.rms_norm_eps))
            gu = f16(lin((li, "gate_up"), layer.gate_up_proj, x2))
            act = f16(oa.silu_and_mul(gu))
            hidden = f16(lin((li, "down"), layer.down_proj, act))
        _, r = oa.fused_add_rms_norm(hidden, residual, m.norm.cpu().numpy(), cfg.rms_norm_eps)
        want = oa.rms_norm(f16(r), m.norm.cpu().numpy(), cfg.rms_norm_eps)
    np.testing.assert_allclose(got, want, atol=2e-2, rtol=2e-2)
    assert np.abs(got - want).mean() / np.abs(want).mean() < 4e-3


@pytest.mark.parametrize("strips", [False, True])
@pytest.mark.parametrize("scheme", ["dynamic", "static"])
@pytest.mark.parametrize("kv_cache_dtype", ["fp8", "auto"])
def test_config2_fused_fp8_decode_layers_vs_oracle(ops, kv_cache_dtype, scheme, strips):
    """configs[2] (compressed-tensors FP8 W8A8, per-token dynamic activations x per-channel weights, FP8-E4M3 KV cache)
    through TWO decoder layers of Llama-3-8B geometry on forward_decode_fused_fp8 -- every activation quantisation fused
    into its producer, raw fp32 slabs between the GEMMs and their consumers, rotary + cache write inside the attention
    launch -- against the op sequence of the reference (compressed_tensors_w8a8_fp8.py:116-130 -> apply_fp8_linear,
    w8a8_utils.py:104-183; attention/layer.py) composed from ORACLE functions.  Activation quantisation is a step
    function: a half-ulp difference upstream moves a token's scale and with it many elements by one fp8 step (6 %), which the
    K-long dot products only average out -- hence a bound on the MEAN error, calibrated in the test itself against the
    oracle's own sensitivity to one omitted bf16 rounding, plus a loose element-wise one.
    scheme "static": the checkpoint carries one input_scale per projection (compressed_tensors_w8a8_fp8.py:98-113) and
    every quantisation is static_scaled_fp8_quant (x * (1 / scale)) -- the same fused launches with the scale handed in.
    strips: the strip-major decode copies of the benched path (``enable_fp8_strips``: the resident W8A8 kernel; round 6: 7
    launches per layer -- the o_proj / down GEMMs quantise the producers' 16-bit activations on load, SiluAndMul rides in the
    gate_up epilogue)."""
    _config2_fused_fp8_layers_vs_oracle(kv_cache_dtype, scheme, [5, 17, 33, 64], 2, 512, strips)


def test_config2_bs32_ctx8192_fused_fp8_decode_layer_vs_oracle(ops):
    """configs[2] AT ITS BENCHED POINT: batch 32, FP8 weights + FP8-E4M3 KV cache, contexts up to
    8192 -- the longest exactly 8192, a 16-token block edge, ragged others -- through ONE decoder layer on the fused
    FP8 path against the oracle-composed layer (same error model as the small case: mean error against the oracle's own
    sensitivity to one omitted bf16 rounding)."""
    rng = np.random.default_rng(8192)
    lens = [8192, 8191, 4096, 4097, 1, 16] + [int(x) for x in rng.integers(1, 8193, size=10)] + \
        [int(x) for x in rng.integers(1, 1025, size=16)]
    _config2_fused_fp8_layers_vs_oracle("fp8", "dynamic", lens, 1, 8448, True)


def _config2_fused_fp8_layers_vs_oracle(kv_cache_dtype, scheme, lens, nlayers, max_pos, strips=False):
    from oracle import fp8 as of8
    from aphrodite_engine_amd import model as M
    from aphrodite_engine_amd.quantization.fp8 import CompressedTensorsW8A8Fp8Config
    cfg = dataclasses.replace(M.LLAMA3_8B, num_hidden_layers=nlayers, vocab_size=2048, max_position_embeddings=max_pos)
    bs, block = len(lens), 16
    dtype = torch.bfloat16
    to_dt = lambda x: torch.from_numpy(np.asarray(x, dtype=np.float32)).to(dtype).float().numpy()     # round to bf16
    kind = "fp8_e4m3" if kv_cache_dtype == "fp8" else "auto"
    with torch.no_grad():
        m = M.LlamaForCausalLM(cfg, CompressedTensorsW8A8Fp8Config("channel", is_static_input_scheme=scheme == "static"),
                               dtype, kv_cache_dtype)
        m.init_synthetic(torch.device(DEV))
        if scheme == "static":          # distinct scales per projection, some rows saturating
            for li, layer in enumerate(m.layers):
                for j, lin_ in enumerate(layer.linears()):
                    lin_.input_scale.fill_((3.0 + j + 0.5 * li) / 448.0)
        meta, pos, nblocks = M.make_decode_metadata(bs, lens, block, DEV)
        ids = torch.randint(0, cfg.vocab_size, (bs, ), device=DEV, generator=torch.Generator(device=DEV).manual_seed(7))
        caches = M.make_kv_caches(cfg, nblocks, block, dtype, kv_cache_dtype, DEV, seed=5)
        caches0 = [c.view(torch.uint8).cpu().numpy().copy() if kv_cache_dtype != "auto" else c.float().cpu().numpy().copy()
                   for c in caches]
        m.use_fused_decode = True
        assert all(l.fused_decode_fp8_ok(bs) for l in m.layers)
        if strips:
            for l in m.layers:
                l.enable_fp8_strips(bs)
            assert m.layers[0].fp8_gate_up_il is not None and "down_proj" in m.layers[0].fp8_strip
        got = m(ids, pos, caches, meta).float().cpu().numpy()

        def linear(lin_, x):
            """dynamic per-token quant + scaled_mm, output rounded to the activation dtype (w8a8_utils.py:143-183)."""
            if lin_.input_scale is not None:
                sx = np.float32(lin_.input_scale.item())
                qx = of8.static_scaled_fp8_quant(x, sx)
            else:
                qx, sx = of8.dynamic_per_token_scaled_fp8_quant(x)
            w = lin_.weight.view(torch.uint8).cpu().numpy()                 # [K, N] view of the [N, K] checkpoint tensor
            return to_dt(of8.scaled_mm(qx, w, sx, lin_.weight_scale.float().cpu().numpy()))

        hkv, hd, hq = cfg.num_key_value_heads, cfg.head_dim, cfg.num_attention_heads
        positions = pos.cpu().numpy()
        slots = meta.slot_mapping.cpu().numpy()
        bt = meta.block_tables.cpu().numpy()
        cos_sin = m.cos_sin.float().cpu().numpy()

        def oracle_step(skip_one_rounding):
            hidden = m.embed_tokens[ids].float().cpu().numpy()
            residual = None
            for li, layer in enumerate(m.layers):
                ln1 = layer.input_layernorm.float().cpu().numpy()
                ln2 = layer.post_attention_layernorm.float().cpu().numpy()
                if residual is None:
                    residual = hidden
                else:
                    _, r = oa.fused_add_rms_norm(hidden, residual, ln1, cfg.rms_norm_eps)
                    residual = to_dt(r)
                x = oa.rms_norm(residual, ln1, cfg.rms_norm_eps)
                if not (skip_one_rounding and li == 0):
                    x = to_dt(x)
                qkv = linear(layer.qkv_proj, x)
                q, k, v = qkv[:, :hq * hd], qkv[:, hq * hd:(hq + hkv) * hd], qkv[:, (hq + hkv) * hd:]
                q, k = oa.rotary_embedding_neox(positions, q, k, hd, cos_sin)
                q, k = to_dt(q), to_dt(k)
                esz = 1 if kv_cache_dtype != "auto" else 2
                kc_shape, vc_shape = oa.split_kv_cache_shapes(nblocks, hkv, hd, block, esz)
                kc = caches0[li][0].copy().reshape(kc_shape)
                vc = caches0[li][1].copy().reshape(vc_shape)
                oa.reshape_and_cache(k.reshape(bs, hkv, hd), v.reshape(bs, hkv, hd), kc, vc, slots, kind, layer.k_scale, layer.v_scale)
                attn = to_dt(oa.paged_attention_decode(q.reshape(bs, hq, hd), kc, vc, bt, lens, hd ** -0.5, None, kind,
                                                       layer.k_scale, layer.v_scale)).reshape(bs, hq * hd)
                o = linear(layer.o_proj, attn)
                _, r = oa.fused_add_rms_norm(o, residual, ln2, cfg.rms_norm_eps)
                residual = to_dt(r)
                x2 = to_dt(oa.rms_norm(residual, ln2, cfg.rms_norm_eps))
                gu = linear(layer.gate_up_proj, x2)
                act = to_dt(oa.silu_and_mul(gu))
                hidden = linear(layer.down_proj, act)
            _, r = oa.fused_add_rms_norm(hidden, residual, m.norm.float().cpu().numpy(), cfg.rms_norm_eps)
            return oa.rms_norm(to_dt(r), m.norm.float().cpu().numpy(), cfg.rms_norm_eps)

        want = oracle_step(False)
        # the yardstick: the SAME oracle with ONE bf16 rounding left out (the first layer's normed input) -- how far the step
        # function of four activation quantisations per layer carries a half-ulp difference through two layers
        yard = np.abs(oracle_step(True) - want).mean() / np.abs(want).mean()
    assert np.isfinite(got).all()
    err = np.abs(got - want).mean() / np.abs(want).mean()
    assert err < max(2e-2, 2.5 * yard), (err, yard)
    np.testing.assert_allclose(got, want, atol=0.25 * np.abs(want).max(), rtol=0.1)
