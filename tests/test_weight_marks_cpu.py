"""What a model says of its weights: whether they come from memory at every step or stay in the last-level cache; and what a call passes on."""
import dataclasses

import torch

from aphrodite_engine_amd import _custom_ops as ops, _lib, model as M


def _model(vocab, hidden):
    cfg = dataclasses.replace(M.LLAMA3_8B, num_hidden_layers=1, vocab_size=vocab, hidden_size=hidden, intermediate_size=2 * hidden, num_attention_heads=hidden // 128,
                              num_key_value_heads=hidden // 128)
    return M.LlamaForCausalLM(cfg, None, torch.float16, "auto").process_weights_after_loading()


def test_models_and_weights():
    small, large = _model(32000, 512), _model(70000, 2048)
    assert {w.streamed for w in small.parameters()} == {False} and {w.streamed for w in large.parameters()} == {True}
    assert ops._weight_flags(small.lm_head) == _lib.WEIGHTS_CACHED and ops._weight_flags(large.layers[0].o_proj.weight) == _lib.WEIGHTS_STREAMED
    assert ops._weight_flags(torch.empty(4, 4)) == 0         # (by its size)
    between = _model(100000, 1024)                           # 205 MB of head and as much of embedding, of which a step reads a few rows
    assert {w.streamed for w in between.parameters()} == {False}
    small.lm_head.streamed = True                            # whoever knows better says so
    assert ops._weight_flags(small.lm_head) == _lib.WEIGHTS_STREAMED


def test_flags_that_are_none_are_refused():
    assert _lib.lib().aphro_scaled_mm_fp8_slabs_flags(None, None, None, 0, 1, 16, 128, 1, None) == -1
