"""StepBatch.build against the same arrays made segment by segment."""
import dataclasses

import numpy as np
import pytest
import torch

from aphrodite_engine_amd.step_batch import StepBatch


@pytest.mark.parametrize("segs", [[(0, 1)], [(0, 17)], [(5, 33), (0, 2), (16, 1), (31, 1)], [(15, 1), (16, 1), (17, 1)], [(0, 1), (3, 1)]])
@pytest.mark.parametrize("block", [16, 5])
def test_build(segs, block):
    rng = np.random.default_rng(len(segs) * block)
    tokens = [rng.integers(0, 99, n).tolist() for _, n in segs]
    tables = [rng.permutation(200)[:(c + n + block - 1) // block + (i % 2)].tolist() for i, (c, n) in enumerate(segs)]
    slots = rng.permutation(9)[:len(segs)].tolist()
    b = StepBatch.build(tokens, [c for c, _ in segs], tables, slots, block, "cpu", rows=[0])
    row = 0
    for s, (c, n) in enumerate(segs):
        for i in range(n):
            p = c + i
            assert b.input_ids[row] == tokens[s][i] and b.positions[row] == p and b.seq_of_token[row] == s
            assert b.slot_mapping[row] == tables[s][p // block] * block + p % block
            row += 1
        assert b.block_tables[s, :len(tables[s])].tolist() == tables[s] and not b.block_tables[s, len(tables[s]):].any()
    assert row == b.num_tokens == b.input_ids.numel() and b.rows.tolist() == [0]
    assert b.q_start.tolist() == np.concatenate([[0], np.cumsum(b.q_lens)[:-1]]).tolist() and b.state_slots.tolist() == slots
    assert b.q_len.tolist() == [n for _, n in segs] and b.ctx_len.tolist() == [c for c, _ in segs]
    for t, kind in ((b.input_ids, torch.int64), (b.positions, torch.int64), (b.slot_mapping, torch.int64), (b.rows, torch.int64),
                    (b.q_start, torch.int32), (b.q_len, torch.int32), (b.ctx_len, torch.int32), (b.seq_of_token, torch.int32),
                    (b.block_tables, torch.int32), (b.state_slots, torch.int32)):
        assert t.dtype == kind and t.is_contiguous()
    m = b.attention_metadata()
    k = m.num_prefills
    assert m.seq_lens_tensor.tolist() == [c + n for c, n in segs] and m.num_prefill_tokens == sum(n for _, n in segs[:k])
    assert m.query_start_loc.tolist() == [0] + np.cumsum([n for _, n in segs[:k]]).tolist()
    assert m.seq_start_loc.tolist() == [0] + np.cumsum([c + n for c, n in segs[:k]]).tolist()
    by_hand = dataclasses.replace(b, rows=None, seq_lens_tensor=None, query_start_loc=None, seq_start_loc=None).attention_metadata()
    for name in ("seq_lens_tensor", "query_start_loc", "seq_start_loc"):
        assert torch.equal(getattr(by_hand, name), getattr(m, name)) and getattr(by_hand, name).dtype == torch.int32
    assert m.query_start_loc.dtype == m.seq_start_loc.dtype == m.seq_lens_tensor.dtype == torch.int32


def test_build_refuses():
    ok = dict(tokens=[[1, 2]], ctx_lens=[15], block_tables=[[3, 4]], state_slots=[0], block_size=16, device="cpu")
    StepBatch.build(**ok)
    for bad, what in ((dict(tokens=[]), "at least one"), (dict(tokens=[[]]), "at least one"), (dict(block_tables=[[3]]), "1 pages for 17 tokens"),
                      (dict(tokens=[[1], [2]], ctx_lens=[0, 0], block_tables=[[1], [2]], state_slots=[4, 4]), "share a state slot"),
                      (dict(tokens=[[1], [2]], ctx_lens=[0], block_tables=[[1], [2]], state_slots=[0, 1]), "1 contexts"),
                      (dict(tokens=[[1], [2]], ctx_lens=[0, 0], block_tables=[[1]], state_slots=[0, 1]), "1 page lists")):
        with pytest.raises(ValueError, match=what):
            StepBatch.build(**{**ok, **bad})
