"""A prompt alone and beside others.  How a launch cuts its work goes by all of it -- one or two groups of waves a row tile in prompt attention, one to eight
chunks a workgroup in the memories -- and sums that are cut otherwise round otherwise.  What a prompt gets may differ by that much from batch to batch
and no more; the same batch gets the same bits."""
import pytest
import torch

from aphrodite_engine_amd import _custom_ops as ops
from aphrodite_engine_amd import mixer_ops as mo

pytestmark = pytest.mark.gpu
DEV, D = "cuda", 128


def _i32(x):
    return torch.tensor(x, dtype=torch.int32, device=DEV)


def _near(run, lens, rel):
    """``run(lens)`` -> rows of the first prompt."""
    alone, beside = run(lens[:1]), run(lens)
    assert torch.equal(beside, run(lens)) and torch.equal(alone, run(lens[:1]))
    assert float((alone.double() - beside.double()).norm() / alone.double().norm()) <= rel


# Attention's probabilities and results are bf16: either cut is within 1.2 x 2^-8 of 64 bits (as the tests of the kernels ask), two within twice that.
@pytest.mark.parametrize("lens", [[700, 700, 700], [300, 2500], [2000, 40]])
def test_attention(lens):
    g = torch.Generator(device=DEV).manual_seed(sum(lens))
    q, k, v = (torch.randn(sum(lens), h, D, generator=g, device=DEV).bfloat16() for h in (32, 8, 8))

    def run(lens):
        n = sum(lens)
        return ops.flash_attn_varlen(q[:n], k[:n], v[:n], _i32([sum(lens[:i]) for i in range(len(lens) + 1)]), max(lens), D ** -0.5)[:lens[0]]
    _near(run, lens, 2.4 * 2.0 ** -8)


@pytest.mark.parametrize("lens", [[700, 700, 700], [300, 2500], [2000, 40]])
def test_paged_attention_of_the_mixers(lens):
    g = torch.Generator(device=DEV).manual_seed(sum(lens))
    blocks = [(n + 15) // 16 for n in lens]
    q = torch.randn(sum(lens), 32 * D, generator=g, device=DEV).bfloat16()
    kc, vc = (torch.randn(sum(blocks), 16, 8, D, generator=g, device=DEV).bfloat16() for _ in range(2))
    lut = torch.randn(32, 300, generator=g, device=DEV)

    def run(lens):
        b = blocks[:len(lens)]
        table = torch.zeros(len(lens), max(b), dtype=torch.int32, device=DEV)
        for i, n in enumerate(b):
            table[i, :n] = sum(b[:i]) + torch.arange(n, device=DEV)
        out = torch.empty(sum(lens), 32 * D, device=DEV, dtype=torch.bfloat16)
        seq = torch.repeat_interleave(torch.arange(len(lens), device=DEV), _i32(lens).long()).int()
        mo.distance_bias_attention(out, q[:sum(lens)], None, kc, vc, table, _i32([sum(lens[:i]) for i in range(len(lens))]), _i32(lens), _i32([0] * len(lens)), seq,
                                   (min(lens), max(lens)), 32, D ** -0.5, lut, max_kv_len=max(lens))
        return out[:lens[0]]
    _near(run, lens, 2.4 * 2.0 ** -8)


# The memories are fp32 throughout: either cut is some 1.2e-7 of the result from 64 bits.
@pytest.mark.parametrize("mode,heads,d,e,lens", [(mo.MEMORY_STATE_SPACE, 64, 128, 64, [520, 3000]), (mo.MEMORY_MLSTM, 4, 128, 256, [520, 5000])])
def test_memories(mode, heads, d, e, lens):
    g = torch.Generator(device=DEV).manual_seed(sum(lens))
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    T = sum(lens)
    q, k, v, gi, gf = (rnd(T, heads * n).bfloat16() for n in (d, d, e, 1, 1))
    kw = dict(gate_f=gf + 2, gate_cap=15.0, q_scale=d ** -0.5) if mode == mo.MEMORY_MLSTM else dict(qk_heads=heads, a_log=rnd(heads) * 0.3, dt_bias=rnd(heads) - 3, skip=rnd(heads))

    def run(lens):
        n, s = sum(lens), len(lens)
        state = tuple(torch.zeros(x, device=DEV) for x in mo.memory_state_shapes(s, heads, d, e, mode))
        part = {key: x[:n] if key == "gate_f" else x for key, x in kw.items()}
        out = mo.outer_memory_scan(q[:n], k[:n], v[:n], state, _i32(range(s)), _i32([sum(lens[:i]) for i in range(s)]), _i32(lens), _i32([0] * s), heads, mode,
                                   max_q_len=max(lens), gate_i=gi[:n], **part)
        return torch.cat([out[:lens[0]].flatten(), state[0][0].flatten()])
    _near(run, lens, 4e-7)
