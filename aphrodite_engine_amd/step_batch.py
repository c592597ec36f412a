"""What one engine step hands to a model: a batch of SEGMENTS.  Segment s is ``q_len[s]`` consecutive rows of the token
batch -- a portion of a prompt or a single decoded token -- that continue a sequence of which ``ctx_len[s]`` tokens were
processed by earlier steps; its keys live in the pages of ``block_tables[s]``, its recurrent state in slot
``state_slots[s]``.  The same structure serves paged attention (through ``attention_metadata()``, the fields of the
reference's AttentionMetadata, attention/backends/abstract.py:96-135) and the recurrent mixers."""
from dataclasses import dataclass, field
from typing import List, Optional, Sequence

import numpy as np
import torch


def _to_device(longs: List[np.ndarray], ints: List[np.ndarray], device, wait: bool) -> List[torch.Tensor]:
    """The int64 and int32 arrays (flat) on the device, as parts (16-byte aligned) of one buffer that one copy from pinned memory fills: a copy
    per array from pageable memory is ten round trips that wait for everything the stream still has to do."""
    if device.type == "cpu":
        return [torch.from_numpy(a) for a in longs + ints]
    sizes = [[x for a in part for x in (a.size, -a.size % unit)] for part, unit in ((longs, 2), (ints, 4))]
    split = sum(sizes[0])
    host = torch.empty(2 * split + sum(sizes[1]), dtype=torch.int32, pin_memory=True)
    image = host.numpy()
    for part, into in ((longs, image[:2 * split].view(np.int64)), (ints, image[2 * split:])):
        at = 0
        for a in part:
            into[at:at + a.size] = a
            at += a.size + -a.size % (16 // a.itemsize)
    buf = host.to(device, non_blocking=True)
    if wait:
        torch.cuda.current_stream(device).synchronize()
    return list(buf[:2 * split].view(torch.int64).split_with_sizes(sizes[0])[::2]) + list(buf[2 * split:].split_with_sizes(sizes[1])[::2])


@dataclass
class StepBatch:
    num_tokens: int
    num_seqs: int
    input_ids: torch.Tensor          # int64 [T]
    positions: torch.Tensor          # int64 [T]
    q_start: torch.Tensor            # int32 [S] first row of each segment
    q_len: torch.Tensor              # int32 [S]
    ctx_len: torch.Tensor            # int32 [S] tokens of the sequence before this step
    seq_of_token: torch.Tensor       # int32 [T]
    block_tables: torch.Tensor       # int32 [S, max_blocks]
    slot_mapping: torch.Tensor       # int64 [T] block * block_size + offset of each row's key / value
    state_slots: torch.Tensor        # int32 [S]
    block_size: int
    q_lens: List[int] = field(default_factory=list)      # host copies
    ctx_lens: List[int] = field(default_factory=list)
    rows: Optional[torch.Tensor] = None                  # int64, rows of the batch asked for
    seq_lens_tensor: Optional[torch.Tensor] = None       # int32 [S] ctx_len + q_len
    query_start_loc: Optional[torch.Tensor] = None       # int32, first rows of the leading prompt portions and their end
    seq_start_loc: Optional[torch.Tensor] = None         # int32, the same of their whole sequences

    @staticmethod
    def build(tokens: Sequence[Sequence[int]], ctx_lens: Sequence[int], block_tables: Sequence[Sequence[int]],
              state_slots: Sequence[int], block_size: int, device, rows: Optional[Sequence[int]] = None, wait: bool = True) -> "StepBatch":
        """From host lists, one entry per segment.  Every index the kernels will follow is checked here.  ``rows``: rows of the batch the
        caller will ask for (``StepBatch.rows``).  All arrays travel in one copy; ``wait`` False: without waiting for it -- for a caller who
        uses the batch on the current stream."""
        S = len(tokens)
        q_lens = [len(t) for t in tokens]
        if S == 0 or min(q_lens) <= 0:
            raise ValueError("a step batch needs at least one segment and no empty one")
        if min(len(ctx_lens), len(block_tables)) < S:
            raise ValueError(f"{S} segments, but {len(ctx_lens)} contexts and {len(block_tables)} page lists")
        ctx = [int(x) for x in ctx_lens[:S]]
        held = [len(b) for b in block_tables[:S]]
        for s in range(S):
            if held[s] * block_size < ctx[s] + q_lens[s]:
                raise ValueError(f"segment {s}: {held[s]} pages for {ctx[s] + q_lens[s]} tokens")
        if len(set(int(x) for x in state_slots)) != S:
            raise ValueError("two segments of one step share a state slot")
        n, c, i32 = np.array(q_lens, np.int64), np.array(ctx, np.int64), np.int32
        T = int(n.sum())
        ends = np.cumsum(n)
        starts = ends - n
        wide = max(1, max(held))
        bt = np.array([list(b) + [0] * (wide - len(b)) for b in block_tables[:S]], i32)
        if T == S:                                           # (decoded tokens: no segment to lay out)
            seq_of, pos, ids = np.arange(S, dtype=i32), c, np.array([t[0] for t in tokens], np.int64)
        else:
            seq_of = np.repeat(np.arange(S, dtype=i32), n)
            pos = np.arange(T) - (starts - c)[seq_of]
            ids = np.empty(T, np.int64)
            for t, a, z in zip(tokens, starts.tolist(), ends.tolist()):
                ids[a:z] = t
        page = pos // block_size
        slots = bt[seq_of, page].astype(np.int64) * block_size + (pos - page * block_size)
        # prompt portions lead (decode_split checks that): their rows and lengths, summed up
        seq_lens = c + n
        k = next((s for s in range(S) if q_lens[s] == 1 and ctx[s] > 0), S)
        loc = np.zeros((2, k + 1), i32)
        loc[0, 1:], loc[1, 1:] = ends[:k], np.cumsum(seq_lens[:k])
        wanted = np.array([] if rows is None else rows, np.int64)
        d = _to_device([ids, pos, slots, wanted], [starts.astype(i32), n.astype(i32), c.astype(i32), seq_of, bt.reshape(-1),
                                                   np.array(state_slots, i32).reshape(-1), seq_lens.astype(i32), loc[0], loc[1]], torch.device(device), wait)
        return StepBatch(num_tokens=T, num_seqs=S, input_ids=d[0], positions=d[1], q_start=d[4], q_len=d[5], ctx_len=d[6],
                         seq_of_token=d[7], block_tables=d[8].view(S, wide), slot_mapping=d[2], state_slots=d[9], block_size=block_size,
                         q_lens=q_lens, ctx_lens=ctx, rows=None if rows is None else d[3], seq_lens_tensor=d[10], query_start_loc=d[11],
                         seq_start_loc=d[12])

    def last_rows(self) -> List[int]:
        """Row of the last token of every segment."""
        out, a = [], 0
        for n in self.q_lens:
            a += n
            out.append(a - 1)
        return out

    def portions(self) -> int:
        """Number of leading segments that are prompt portions (anything but a single token with a context)."""
        for s, (n, c) in enumerate(zip(self.q_lens, self.ctx_lens)):
            if n == 1 and c > 0:
                return s
        return len(self.q_lens)

    def decode_split(self) -> int:
        """Number of leading segments that are prompt portions when the batch is ordered portions first, single tokens
        with a context last (the order the reference's metadata assumes); raises if it is not."""
        kinds = [n == 1 and c > 0 for n, c in zip(self.q_lens, self.ctx_lens)]
        k = kinds.index(True) if True in kinds else len(kinds)
        if not all(kinds[k:]):
            raise ValueError("segments are not ordered prompt portions first, decoded tokens last")
        return k

    def attention_metadata(self):
        """The same batch as MI355XAttentionMetadata (prefill rows first, decode rows after)."""
        from .attention.backend import MI355XAttentionMetadata
        k = self.decode_split()
        seq_lens = [c + n for c, n in zip(self.ctx_lens, self.q_lens)]
        npt = sum(self.q_lens[:k])
        dev = self.input_ids.device
        # (build() sent these along; a batch put together by hand has none)
        sums = lambda x: torch.from_numpy(np.concatenate([[0], np.cumsum(x[:k], dtype=np.int64)]).astype(np.int32)).to(dev)
        seq_lens_tensor = torch.tensor(seq_lens, dtype=torch.int32, device=dev) if self.seq_lens_tensor is None else self.seq_lens_tensor
        return MI355XAttentionMetadata(
            num_prefills=k, num_prefill_tokens=npt, num_decode_tokens=self.num_tokens - npt, slot_mapping=self.slot_mapping,
            seq_lens=seq_lens, seq_lens_tensor=seq_lens_tensor,
            max_query_len=max(self.q_lens), max_prefill_seq_len=max(seq_lens[:k], default=0),
            max_decode_seq_len=max(seq_lens[k:], default=0),
            query_start_loc=sums(self.q_lens) if self.query_start_loc is None else self.query_start_loc,
            seq_start_loc=sums(seq_lens) if self.seq_start_loc is None else self.seq_start_loc,
            context_lens_tensor=self.ctx_len[:k] if k else self.ctx_len[:0], block_tables=self.block_tables,
            use_cuda_graph=False, max_context_len=max(self.ctx_lens[:k], default=0))
