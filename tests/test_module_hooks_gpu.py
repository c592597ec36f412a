"""Hooks on a projection see its calls, and change what they return, also where a kernel of its own does the projection's work with what follows."""
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rows", [1, 40, 192, 200])
def test_gate_and_up(rows):
    from aphrodite_engine_amd import mixer_ops as mops
    from aphrodite_engine_amd.mixers import GatedMLP
    with torch.device(DEV):
        mlp = GatedMLP(256, 512, mops.ACT_SILU, torch.bfloat16)
    g = torch.Generator(device=DEV).manual_seed(rows)
    for lin in (mlp.gate_up, mlp.down):
        lin.weight.data.copy_(torch.randn(lin.weight.shape, generator=g, device=DEV) * 0.1)
    h = torch.randn(rows, 256, generator=g, device=DEV).to(torch.bfloat16)
    with torch.no_grad():
        plain, seen = mlp(h), []
        assert plain.abs().max() > 0
        handle = mlp.gate_up.register_forward_hook(lambda module, args, out: (seen.append(out.shape), out.zero_())[1])
        assert not mlp(h).any() and seen == [(rows, 1024)]
        handle.remove()
        handle = mlp.gate_up.register_forward_pre_hook(lambda module, args: (torch.zeros_like(args[0]), ))
        assert not mlp(h).any()
        handle.remove()
        handle = torch.nn.modules.module.register_module_forward_hook(lambda module, args, out: seen.append(module))
        mlp(h)
        handle.remove()
        assert mlp.gate_up in seen
        assert torch.equal(mlp(h), plain)
        mlp.gate_up.bias = torch.nn.Parameter(torch.full((1024, ), -50.0, dtype=torch.bfloat16, device=DEV))       # (shuts every gate)
        assert mlp(h).abs().max() < 1e-6


def _llama(quant, layers=2, kv="auto", dtype=torch.float16):
    import dataclasses
    from aphrodite_engine_amd import model as M
    cfg = dataclasses.replace(M.LLAMA3_8B, num_hidden_layers=layers, vocab_size=512, max_position_embeddings=512)
    model = M.LlamaForCausalLM(cfg, quant, dtype, kv)
    model.init_synthetic(torch.device(DEV))
    return M, cfg, model


def _decode(M, cfg, model, rows, kv="auto", dtype=torch.float16):
    meta, pos, blocks = M.make_decode_metadata(rows, [5 + i % 40 for i in range(rows)], 16, DEV)
    caches = M.make_kv_caches(cfg, blocks, 16, dtype, kv, DEV, seed=5)
    ids = torch.arange(rows, device=DEV)
    return lambda: model(ids, pos, caches, meta)


@pytest.mark.parametrize("rows", [70, 150])
def test_int4_output_projections(rows):
    from aphrodite_engine_amd.quantization.gptq import GPTQConfig
    with torch.no_grad():
        M, cfg, model = _llama(GPTQConfig(4, 128, False))
        step, seen = _decode(M, cfg, model, rows), []
        plain = step()
        handles = [getattr(layer, name).register_forward_hook(lambda module, args, out: seen.append(module))
                   for layer in model.layers for name in ("o_proj", "down_proj")]
        assert torch.equal(step(), plain) and seen == [lin for layer in model.layers for lin in (layer.o_proj, layer.down_proj)]
        for h in handles:
            h.remove()
        handle = model.layers[0].o_proj.register_forward_hook(lambda module, args, out: out * 2)
        assert not torch.equal(step(), plain)
        handle.remove()
        assert torch.equal(step(), plain)


@pytest.mark.parametrize("rows", [70, 150])
def test_layers(rows):
    """A hook on a layer, and a class of its own in a layer's place, see rows that no norm has touched."""
    from aphrodite_engine_amd import _custom_ops as ops
    from aphrodite_engine_amd.quantization.gptq import GPTQConfig
    with torch.no_grad():
        M, cfg, model = _llama(GPTQConfig(4, 128, False))
        step, seen = _decode(M, cfg, model, rows), []
        plain = step()
        handle = model.layers[1].register_forward_hook(lambda module, args, out: seen.append([t.clone() for t in out]))
        assert torch.equal(step(), plain)
        handle.remove()
        (hidden, residual), = seen
        ops.fused_add_rms_norm(hidden, residual, model.norm, cfg.rms_norm_eps)
        assert torch.equal(hidden, plain)

        class Counted(M.LlamaDecoderLayer):
            calls = 0

            def forward(self, positions, hidden, residual, kv_cache, attn_metadata, cos_sin):
                Counted.calls += 1
                return super().forward(positions, hidden, residual, kv_cache, attn_metadata, cos_sin)

        model.layers[0].__class__ = Counted
        assert torch.equal(step(), plain) and Counted.calls == 1


@pytest.mark.parametrize("rows", [100, 200])
def test_fp8_steps_of_many_decoded_rows(rows):
    from aphrodite_engine_amd.quantization.fp8 import CompressedTensorsW8A8Fp8Config
    with torch.no_grad():
        M, cfg, model = _llama(CompressedTensorsW8A8Fp8Config("channel", is_static_input_scheme=False), dtype=torch.bfloat16)
        step, seen = _decode(M, cfg, model, rows, dtype=torch.bfloat16), []
        plain = step()
        for module in (model.layers[1], model.layers[0].o_proj):
            handle = module.register_forward_hook(lambda module, args, out: seen.append(module))
            assert torch.equal(step(), plain) and seen.pop() is module and not seen
            handle.remove()


@pytest.mark.parametrize("rows", [70, 150])
@pytest.mark.parametrize("name", ["qkv_proj", "o_proj", "gate_up_proj", "down_proj"])
def test_a_projection_of_ones_own(rows, name):
    """A class, or a forward, in a projection's place is called: its result counts."""
    from aphrodite_engine_amd.quantization.gptq import GPTQConfig
    with torch.no_grad():
        M, cfg, model = _llama(GPTQConfig(4, 128, False))
        if name == "gate_up_proj":                          # (the form whose columns are interleaved for the product's own SiluAndMul)
            assert model.layers[0].enable_fused_silu(32, keep_original=False)
        step, calls = _decode(M, cfg, model, rows), []
        plain, lin = step(), getattr(model.layers[0], name)

        class Own(M.QuantLinear):
            scale = 1

            def forward(self, x, add_bias=True):
                calls.append(x.shape[0])
                return super().forward(x, add_bias) * self.scale

        lin.__class__ = Own
        assert torch.equal(step(), plain) and calls == [rows]
        Own.scale = 2
        assert not torch.equal(step(), plain) and calls == [rows] * 2
        lin.__class__ = M.QuantLinear
        lin.forward = lambda x, add_bias=True: (calls.append("instance"), M.QuantLinear.forward(lin, x, add_bias))[1]
        assert torch.equal(step(), plain) and calls[2:] == ["instance"]


@pytest.mark.parametrize("rows", [100, 190])
def test_an_fp8_projection_of_ones_own(rows):
    from aphrodite_engine_amd.quantization.fp8 import CompressedTensorsW8A8Fp8Config
    with torch.no_grad():
        M, cfg, model = _llama(CompressedTensorsW8A8Fp8Config("channel", is_static_input_scheme=False), dtype=torch.bfloat16)
        step, calls = _decode(M, cfg, model, rows, dtype=torch.bfloat16), []
        step()

        class Own(M.QuantLinear):
            def forward(self, x, add_bias=True):
                calls.append(x.shape[0])
                return super().forward(x, add_bias)

        model.layers[1].qkv_proj.__class__ = Own
        step()
        assert calls == [rows]
