"""Whole FP8 steps of more rows than one decode launch serves, against the same step op by op: decoded rows from 33 to 192, prompts beside
decoded rows, both activation schemes, 16-bit and FP8 caches.  The fused step does the same operations in fewer launches, so that every bit of
the hidden rows and of the caches is the same."""
import dataclasses
import functools

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@functools.lru_cache(1)
def _model(scheme, kv, dtype):
    from aphrodite_engine_amd import model as M
    from aphrodite_engine_amd.quantization.fp8 import CompressedTensorsW8A8Fp8Config
    cfg = dataclasses.replace(M.LLAMA3_8B, num_hidden_layers=2, vocab_size=512, max_position_embeddings=512, intermediate_size=3584)
    m = M.LlamaForCausalLM(cfg, CompressedTensorsW8A8Fp8Config("channel", is_static_input_scheme=scheme == "static"), dtype, kv)
    m.init_synthetic(torch.device(DEV))
    if scheme == "static":
        for i, layer in enumerate(m.layers):
            for j, lin in enumerate(layer.linears()):
                lin.input_scale.fill_((3.0 + j + 0.5 * i) / 448.0)
    for layer in m.layers:
        layer.enable_fp8_strips(32)
    return M, cfg, m


def _same(M, cfg, m, ids, pos, meta, blocks, kv, dtype, monkeypatch):
    results = []
    for fused in (True, False):
        m.use_fused_decode = fused
        if not fused:
            monkeypatch.setenv("APHRO_PREFILL_NO_FUSED_FP8", "1")
        calls = []
        hook = None if fused else m.layers[0].register_forward_hook(lambda *args: calls.append(1))
        caches = M.make_kv_caches(cfg, blocks, 16, dtype, kv, DEV, seed=3)
        hidden = m(ids, pos, caches, meta)
        if hook is not None:
            hook.remove()
            assert calls                                     # (op by op indeed)
        results.append((hidden.clone(), caches))
    monkeypatch.delenv("APHRO_PREFILL_NO_FUSED_FP8")
    (a, ca), (b, cb) = results
    assert torch.isfinite(a.float()).all() and a.float().norm() > 0
    assert torch.equal(a.view(torch.int16), b.view(torch.int16))
    for x, y in zip(ca, cb):
        assert torch.equal(x.view(torch.uint8), y.view(torch.uint8))


@pytest.mark.parametrize("rows", [33, 64, 65, 128, 129, 192, 193])
@pytest.mark.parametrize("scheme,kv,dtype", [("dynamic", "fp8", torch.bfloat16), ("dynamic", "auto", torch.float16), ("static", "fp8", torch.float16),
                                             ("static", "auto", torch.bfloat16)])
def test_decoded_rows(scheme, kv, dtype, rows, monkeypatch):
    with torch.no_grad():
        M, cfg, m = _model(scheme, kv, dtype)
        assert m.layers[0].fused_decode_fp8_rows_ok(rows) == (rows <= 192)
        meta, pos, blocks = M.make_decode_metadata(rows, [1 + (37 * i) % 300 for i in range(rows)], 16, DEV)
        ids = torch.randint(0, cfg.vocab_size, (rows, ), device=DEV, generator=torch.Generator(device=DEV).manual_seed(rows))
        _same(M, cfg, m, ids, pos, meta, blocks, kv, dtype, monkeypatch)


@pytest.mark.parametrize("prompts,decoded", [([(40, 0), (25, 0)], [30, 7]), ([(50, 33), (1, 0), (17, 160)], [1, 16, 17, 200]), ([(300, 0)], [20] * 40)])
@pytest.mark.parametrize("scheme,kv,dtype", [("dynamic", "fp8", torch.bfloat16), ("static", "auto", torch.float16)])
def test_prompts_beside_decoded_rows(scheme, kv, dtype, prompts, decoded, monkeypatch):
    from aphrodite_engine_amd.attention.backend import MI355XAttentionMetadata
    with torch.no_grad():
        M, cfg, m = _model(scheme, kv, dtype)
        segments = [(n, c) for n, c in prompts] + [(1, c) for c in decoded]      # new tokens, tokens before them
        lens = [n + c for n, c in segments]
        wide = max((n + 15) // 16 for n in lens)
        tables = torch.randperm(len(segments) * wide, generator=torch.Generator().manual_seed(1)).view(len(segments), wide).tolist()
        dev = lambda x, t=torch.int32: torch.tensor(x, dtype=t, device=DEV)
        pos = [c + i for n, c in segments for i in range(n)]
        slots = [t[p // 16] * 16 + p % 16 for (n, c), t in zip(segments, tables) for p in range(c, c + n)]
        news, k = [n for n, _ in prompts], len(prompts)
        starts = lambda x: dev([sum(x[:i]) for i in range(len(x) + 1)])
        meta = MI355XAttentionMetadata(
            num_prefills=k, num_prefill_tokens=sum(news), num_decode_tokens=len(decoded), slot_mapping=dev(slots, torch.int64), seq_lens=lens,
            seq_lens_tensor=dev(lens), max_query_len=max(news), max_prefill_seq_len=max(lens[:k]), max_decode_seq_len=max(lens[k:]),
            query_start_loc=starts(news), seq_start_loc=starts(lens[:k]), context_lens_tensor=dev([c for _, c in segments]),
            block_tables=dev(tables), use_cuda_graph=False, max_context_len=max(c for _, c in prompts))
        ids = torch.randint(0, cfg.vocab_size, (len(pos), ), device=DEV, generator=torch.Generator(device=DEV).manual_seed(2))
        _same(M, cfg, m, ids, dev(pos, torch.int64), meta, len(segments) * wide, kv, dtype, monkeypatch)
