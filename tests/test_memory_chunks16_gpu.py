"""Prompt portions of the mLSTM and state-space memories on bf16 inputs, whose products run on the 16-bit matrix cores
(csrc/mixers/outer_memory_chunked.hip, om_chunk_update16_kernel, om_chunk_out16_kernel): the recurrence in 64 bits at lengths around chunks
and at dimensions around tiles, and keys and values that are not finite."""
import pytest
import torch

from test_memory_rows_gpu import DEV, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode,heads,groups", [(1, 2, 0), (2, 6, 2)])
@pytest.mark.parametrize("d,e", [(128, 64), (64, 64), (128, 256), (40, 20), (100, 72), (127, 61), (33, 130)])
@pytest.mark.parametrize("lens", [[257], [192, 1, 255, 320, 2], [193, 256, 33]])
def test_recurrence(mode, heads, groups, d, e, lens):
    run(mode, lens, heads, d, e, groups, seed=d + e + len(lens))


@pytest.mark.parametrize("mode", [1, 2])
@pytest.mark.parametrize("where", ["key", "value"])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_numbers_that_are_not_finite(mode, where, bad):
    """They show from their token on, as in the scan: heads beside it and chunks ahead of it keep their bits, the tokens ahead of it in its chunk
    their values (such a chunk sums on the vector ALUs), and what follows is as finite or not."""
    from aphrodite_engine_amd import mixer_ops as mops
    T, H, d, e, at = 300, 2, 64, 64, 150
    g = torch.Generator(device=DEV).manual_seed(5)
    rnd = lambda *s: torch.randn(*s, generator=g, device=DEV)
    q, k, v = (rnd(T, H * 64).bfloat16() for _ in range(3))
    kw = dict(gate_i=rnd(T, H).bfloat16(), gate_f=(rnd(T, H) + 2).bfloat16(), gate_cap=15.0) if mode == 1 else \
        dict(gate_i=rnd(T, H).bfloat16(), qk_heads=H, a_log=rnd(H) * 0.3, dt_bias=rnd(H) * 0.3, skip=rnd(H))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)

    def go(q, k, v, max_q_len=T):
        state = tuple(torch.zeros(s, device=DEV) for s in mops.memory_state_shapes(1, H, d, e, mode))
        o = mops.outer_memory_scan(q, k, v, state, i32([0]), i32([0]), i32([T]), i32([0]), H, mode, max_q_len=max_q_len, **kw)
        return o.view(T, H, e), state[0]

    clean, _ = go(q, k, v)
    (k if where == "key" else v)[at, 3] = bad
    got, state = go(q, k, v)
    scan, scan_state = go(q, k, v, max_q_len=40)              # the token-by-token form
    assert torch.equal(got[:, 1], clean[:, 1]) and torch.equal(got[:at // 64 * 64, 0], clean[:at // 64 * 64, 0])
    # fp32 sums of up to 64 products in another order
    assert float((got[:at, 0] - clean[:at, 0]).norm()) <= 1e-5 * float(clean[:at, 0].norm())
    assert torch.equal(got.isfinite(), scan.isfinite()) and torch.equal(state.isfinite(), scan_state.isfinite())
