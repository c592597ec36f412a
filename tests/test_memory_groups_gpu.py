"""Prompt portions of the mLSTM and state-space memories on bf16 inputs in groups of two, four and eight chunks to a workgroup
(csrc/mixers/outer_memory_chunked.hip, om_group_chunks): the recurrence in 64 bits at sizes of every group, with segments that end inside a group and
beside single tokens, and the same bits from a workspace of one group."""
import pytest
import torch

from test_memory_rows_gpu import DEV, run

pytestmark = pytest.mark.gpu

# (mode, heads, key heads, d, e): chunks * heads * blocks of 64 columns makes the group
CASES = [(2, 64, 8, 100, 64, [597]), (2, 96, 4, 64, 60, [449]), (1, 16, 0, 128, 256, [610]),                      # two
         (2, 64, 8, 128, 64, [1281, 1, 65, 33]), (2, 80, 1, 40, 130, [400, 2, 129]), (1, 24, 0, 72, 200, [513, 256, 1]),    # four
         (2, 64, 2, 128, 256, [1089]), (2, 64, 8, 64, 250, [513, 512, 40]), (1, 64, 0, 64, 256, [577, 1, 450]),      # eight
         (2, 12, 1, 64, 64, [700]), (2, 27, 3, 64, 40, [130, 70])]                                               # few key heads: a pair's heads over the XCDs


@pytest.mark.parametrize("case", CASES)
def test_recurrence(case):
    mode, heads, groups, d, e, lens = case
    run(mode, lens, heads, d, e, groups, seed=heads + d)


@pytest.mark.parametrize("mode,heads,d,e,lens", [(2, 64, 128, 256, [700, 1, 500]), (1, 16, 128, 256, [700, 3, 100])])
def test_groups_in_spans(monkeypatch, mode, heads, d, e, lens):
    from aphrodite_engine_amd import mixer_ops as mops
    g = torch.Generator(device=DEV).manual_seed(3)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    T, n = sum(lens), len(lens)
    q, k, v = rnd(T, heads * d).bfloat16(), rnd(T, heads * d).bfloat16(), rnd(T, heads * e).bfloat16()
    kw = dict(gate_i=rnd(T, heads).bfloat16(), gate_f=(rnd(T, heads) + 2).bfloat16(), gate_cap=15.0) if mode == 1 else \
        dict(gate_i=rnd(T, heads).bfloat16(), qk_heads=heads, a_log=rnd(heads) * 0.3, dt_bias=rnd(heads) * 0.3, skip=rnd(heads))
    first = [rnd(*s) for s in mops.memory_state_shapes(n, heads, d, e, mode)]
    for s in first[1:]:
        s.copy_(s[:, :, :1].expand_as(s).clone())
    lib, name = mops._lib.mixers_lib(), "aphro_outer_memory_chunked_workspace"

    def go():
        state = tuple(s.clone() for s in first)
        starts = [sum(lens[:i]) for i in range(n)]
        return (mops.outer_memory_scan(q, k, v, state, i32(range(n)), i32(starts), i32(lens), i32([5] * n), heads, mode, max_q_len=max(lens), **kw), ) + state
    want, full = go(), getattr(lib, name)
    monkeypatch.setattr(lib, name, lambda *a: full(1, 64, *a[2:-1], 64) + (12 * heads * (T - 64) if mode == 1 else 0))
    for x, y in zip(go(), want):
        assert torch.equal(x, y)
