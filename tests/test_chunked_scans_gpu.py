"""The recurrences in chunks of 64 tokens against plain 64-bit recurrences, at the edges of chunks and tiles: lengths about 16, 32 and 64,
several segments of one batch, states carried in, rows that are not 16-byte aligned, numbers that are not finite."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.fixture(scope="module")
def mops():
    from aphrodite_engine_amd import mixer_ops
    return mixer_ops


@pytest.fixture(autouse=True)
def chunks_whatever_pays(mops, monkeypatch):
    monkeypatch.setattr(mops, "MEMORY_CHUNKED_FROM", {m: (1, 1) for m in mops.MEMORY_CHUNKED_FROM})
    monkeypatch.setattr(mops, "DELTA_CHUNKED_FROM", 1)
    monkeypatch.setattr(mops, "delta_chunks_pay", lambda *a: True)


def i32(xs):
    return torch.tensor(list(xs), dtype=torch.int32, device=DEV)


def part(g, rows, cols, dtype, pad):
    """Random rows behind ``pad`` other columns of a wider tensor."""
    return torch.randn(rows, cols + pad, generator=g, device=DEV).to(dtype)[:, pad:]


def memory_reference(mops, mode, q, k, v, S, n, m, decay, gi, gf, q_scale, cap, a_log, dt_bias, skip):
    """One head, one segment, token by token in 64 bits."""
    out = torch.empty(v.shape, dtype=torch.float64)
    silu = torch.nn.functional.silu
    for t in range(q.shape[0]):
        qt, kt, vt, den = q[t], k[t], v[t], 1.0
        if mode == mops.MEMORY_DECAY:
            qt, kt, vt, a, b = silu(qt), silu(kt), silu(vt), decay, 1.0
        elif mode == mops.MEMORY_MLSTM:
            i, f = cap * torch.tanh(gi[t] / cap), torch.nn.functional.logsigmoid(cap * torch.tanh(gf[t] / cap))
            now = max(float(f) + m, float(i))
            a, b, m = np.exp(float(f) + m - now), np.exp(float(i) - now), now
            qt = qt * q_scale
            n = a * n + b * kt
            den = max(abs(float(n @ qt)), np.exp(-m)) + 1e-6
        else:
            dt = torch.nn.functional.softplus(gi[t] + dt_bias)
            a, b = torch.exp(-torch.exp(a_log) * dt), dt
        S = a * S + b * kt[:, None] * vt[None, :]
        out[t] = S.T @ qt / den + (skip * vt if mode == mops.MEMORY_STATE_SPACE else 0.0)
    return out, S, n, m


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("dtype,pad", [(torch.bfloat16, 0), (torch.bfloat16, 3), (torch.float32, 4)])
@pytest.mark.parametrize("d,e", [(64, 128), (128, 64), (24, 72), (100, 20)])
def test_memory_chunks(mops, mode, dtype, pad, d, e):
    H, lens, ctx = 2, [64, 1, 33, 129, 31], [0, 7, 5, 0, 9]
    g = torch.Generator(device=DEV).manual_seed(d * 3 + e + mode)
    T, S = sum(lens), len(lens)
    q, k, v = part(g, T, H * d, dtype, pad), part(g, T, H * d, dtype, pad), part(g, T, H * e, dtype, pad)
    gates = torch.randn(T, 2 * H + 1, generator=g, device=DEV).to(dtype)
    gi, gf = gates[:, 1:H + 1], gates[:, H + 1:]
    decay = torch.tensor([0.97, -0.8], device=DEV)
    a_log, dt_bias, skip = (torch.randn(H, generator=g, device=DEV) for _ in range(3))
    state = tuple(torch.randn(s, generator=g, device=DEV) for s in mops.memory_state_shapes(S + 1, H, d, e, mode))
    if mode == mops.MEMORY_MLSTM:                       # every 16 columns hold the same n and m
        state[1][:], state[2][:] = state[1][:, :, :1].clone(), state[2][:, :, :1].abs().clone()
    slots, start = [3, 5, 0, 2, 4], np.concatenate([[0], np.cumsum(lens)[:-1]])
    before = [s.double().cpu() for s in state]
    kw = {0: dict(decay=decay), 1: dict(gate_i=gi, gate_f=gf, q_scale=d ** -0.5, gate_cap=6.0),
          2: dict(gate_i=gi, a_log=a_log, dt_bias=dt_bias, skip=skip)}[mode]
    out = mops.outer_memory_scan(q, k, v, state, i32(slots), i32(start), i32(lens), i32(ctx), H, mode, max_q_len=max(lens), **kw)
    Q, K, V, GI, GF = (x.double().cpu() for x in (q, k, v, gi, gf))
    for s in range(S):
        rows = slice(start[s], start[s] + lens[s])
        for h in range(H):
            S0 = before[0][slots[s], h] if ctx[s] else torch.zeros(d, e, dtype=torch.float64)
            n0, m0 = torch.zeros(d, dtype=torch.float64), 0.0
            if mode == mops.MEMORY_MLSTM and ctx[s]:
                n0, m0 = before[1][slots[s], h, 0], float(before[2][slots[s], h, 0])
            want, Sw, nw, mw = memory_reference(
                mops, mode, Q[rows, h * d:(h + 1) * d], K[rows, h * d:(h + 1) * d], V[rows, h * e:(h + 1) * e], S0, n0, m0, float(decay[h]),
                GI[rows, h], GF[rows, h], d ** -0.5, 6.0, float(a_log[h]) * torch.ones((), dtype=torch.float64), float(dt_bias[h]), float(skip[h]))
            got = out[rows, h * e:(h + 1) * e].double().cpu()
            # fp32 sums of up to 129 + d products behind a few exponentials of 1 ulp; silu and the mLSTM's division as the scan has them
            assert torch.allclose(got, want, rtol=1e-4, atol=3e-5 * float(want.abs().max())), (s, h, (got - want).abs().max())
            assert torch.allclose(state[0][slots[s], h].double().cpu(), Sw, rtol=1e-4, atol=3e-5 * float(Sw.abs().max()))
            if mode == mops.MEMORY_MLSTM:
                for c in range(state[1].shape[2]):
                    assert torch.allclose(state[1][slots[s], h, c].double().cpu(), nw, rtol=1e-4, atol=3e-5 * float(nw.abs().max()))
                    assert abs(float(state[2][slots[s], h, c]) - mw) < 1e-4 * max(1.0, abs(mw))
    assert torch.equal(state[0][1].double().cpu(), before[0][1])          # a slot that no segment names


def test_memory_chunks_long_gates(mops):
    """More tokens than the gate launch folds at a time; strong and weak decays in turn."""
    T, H, d, e = 4096 + 77, 1, 16, 16
    g = torch.Generator(device=DEV).manual_seed(5)
    q, k, v = part(g, T, d, torch.float32, 0), part(g, T, d, torch.float32, 0), part(g, T, e, torch.float32, 0)
    gi, gf = part(g, T, 1, torch.float32, 0) * 4, part(g, T, 1, torch.float32, 0) * 9
    state = tuple(torch.zeros(s, device=DEV) for s in mops.memory_state_shapes(1, H, d, e, 1))
    out = mops.outer_memory_scan(q, k, v, state, i32([0]), i32([0]), i32([T]), i32([0]), H, 1, gate_i=gi, gate_f=gf, q_scale=0.25,
                                 gate_cap=15.0, max_q_len=T).double().cpu()
    z = torch.zeros(d, dtype=torch.float64)
    want, S, n, m = memory_reference(mops, 1, q.double().cpu(), k.double().cpu(), v.double().cpu(), torch.zeros(d, e, dtype=torch.float64), z, 0.0,
                                     0.0, gi[:, 0].double().cpu(), gf[:, 0].double().cpu(), 0.25, 15.0, None, None, None)
    rel = (out - want).norm(dim=1) / want.norm(dim=1)
    assert float(rel.median()) < 1e-6 and float(rel.max()) < 2e-3, (float(rel.median()), float(rel.max()))   # (a normaliser near zero)
    assert torch.allclose(state[0][0, 0].double().cpu(), S, rtol=1e-4, atol=1e-5 * float(S.abs().max()))


@pytest.mark.parametrize("mode", [0, 1, 2])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_memory_chunks_keep_the_tokens_ahead_of_a_bad_value(mops, mode, bad):
    T, H, d, e, at = 100, 1, 32, 24, 70
    g = torch.Generator(device=DEV).manual_seed(9)
    q, k, v = (part(g, T, n, torch.float32, 0) for n in (d, d, e))
    gi, gf, one = part(g, T, 1, torch.float32, 0), part(g, T, 1, torch.float32, 0), torch.ones(1, device=DEV)
    kw = {0: dict(decay=0.9 * one), 1: dict(gate_i=gi, gate_f=gf), 2: dict(gate_i=gi, a_log=one, dt_bias=one, skip=one)}[mode]

    def go(vv):
        state = tuple(torch.zeros(s, device=DEV) for s in mops.memory_state_shapes(1, H, d, e, mode))
        return mops.outer_memory_scan(q, k, vv, state, i32([0]), i32([0]), i32([T]), i32([0]), H, mode, max_q_len=T, **kw)
    want, w = go(v), v.clone()
    w[at, 3] = bad
    got = go(w)
    cols = [c for c in range(e) if c != 3]
    assert torch.allclose(got[:at], want[:at], rtol=1e-4, atol=1e-5) and torch.allclose(got[:, cols], want[:, cols], rtol=1e-4, atol=1e-5)
    assert not torch.isfinite(got[at:, 3]).any()


def delta_reference(q, k, v, beta, g, S):
    """One head, one segment, token by token in 64 bits; g [T, d]."""
    out = torch.empty(v.shape, dtype=torch.float64)
    for t in range(q.shape[0]):
        S = g[t][:, None] * S
        S = S + k[t][:, None] * (beta[t] * (v[t] - S.T @ k[t]))[None, :]
        out[t] = S.T @ q[t]
    return out, S


@pytest.mark.parametrize("channel", [True, False])
@pytest.mark.parametrize("dtype,pad", [(torch.bfloat16, 0), (torch.bfloat16, 3), (torch.float32, 4)])
@pytest.mark.parametrize("d,e", [(128, 128), (64, 72), (24, 20), (100, 200)])
@pytest.mark.parametrize("strong", [False, True])
def test_delta_chunks(mops, channel, dtype, pad, d, e, strong):
    H, G, lens, ctx = 2, 1, [64, 1, 33, 193, 31], [0, 7, 5, 0, 9]
    g = torch.Generator(device=DEV).manual_seed(d * 3 + e + channel)
    T, S = sum(lens), len(lens)
    q, k, v = part(g, T, G * d, dtype, pad), part(g, T, G * d, dtype, pad), part(g, T, H * e, dtype, pad)
    b = part(g, T, H, dtype, 1)
    na = H * d if channel else H
    a = part(g, T, na, dtype, pad) * (4.0 if strong else 1.0)
    a_log, dt_bias = torch.randn(H, generator=g, device=DEV), torch.randn(na, generator=g, device=DEV) - (0.0 if strong else 3.0)
    state = torch.randn(S + 1, H, d, e, generator=g, device=DEV)
    slots, start = [3, 5, 0, 2, 4], np.concatenate([[0], np.cumsum(lens)[:-1]])
    before = state.double().cpu()
    out = mops.gated_delta_scan(q, k, v, b, a, a_log, dt_bias, state, i32(slots), i32(start), i32(lens), i32(ctx), H, G, d ** -0.5,
                                max_q_len=max(lens))
    Q, K, V, B, A, AL, DT = (x.double().cpu() for x in (q, k, v, b, a, a_log, dt_bias))
    for s in range(S):
        rows = slice(start[s], start[s] + lens[s])
        for h in range(H):
            qh, kh = (x[rows, :d] / torch.sqrt((x[rows, :d] ** 2).sum(1, keepdim=True) + 1e-6) for x in (Q, K))
            ah = A[rows, h * d:(h + 1) * d] + DT[h * d:(h + 1) * d] if channel else (A[rows, h] + DT[h])[:, None].expand(-1, d)
            gh = torch.exp(-torch.exp(AL[h]) * torch.nn.functional.softplus(ah))
            S0 = before[slots[s], h] if ctx[s] else torch.zeros(d, e, dtype=torch.float64)
            want, Sw = delta_reference(qh * d ** -0.5, kh, V[rows, h * e:(h + 1) * e], torch.sigmoid(B[rows, h]), gh, S0)
            got = out[rows, h * e:(h + 1) * e].double().cpu()
            # fp32 sums of d + 64 products through a triangle of 64 corrections of size below one
            assert torch.allclose(got, want, rtol=1e-4, atol=2e-5 * float(want.abs().max())), (s, h, (got - want).abs().max())
            assert torch.allclose(state[slots[s], h].double().cpu(), Sw, rtol=1e-4, atol=2e-5 * float(Sw.abs().max()))
    assert torch.equal(state[1].double().cpu(), before[1])                # a slot that no segment names


@pytest.mark.parametrize("where", ["v", "k", "q", "b", "u"])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_delta_chunks_keep_the_tokens_ahead_of_a_bad_value(mops, where, bad):
    T, H, d, e, at = 170, 1, 32, 24, 70
    g = torch.Generator(device=DEV).manual_seed(9)
    x = {n: part(g, T, w, torch.float32, 0).contiguous() for n, w in (("q", d), ("k", d), ("v", e), ("b", 1), ("a", d))}

    def go(y):
        state = torch.zeros(1, H, d, e, device=DEV)
        o = mops.gated_delta_scan(y["q"], y["k"], y["v"], y["b"], y["a"], torch.zeros(1, device=DEV), torch.zeros(d, device=DEV) - 2, state,
                                  i32([0]), i32([0]), i32([T]), i32([0]), H, H, 1.0, max_q_len=T)
        return o, state
    want, w = go(x)[0], {n: t.clone() for n, t in x.items()}
    if where == "u":                                     # finite values whose correction is beyond fp32: v against what the same key holds
        w["k"][at], w["b"][at - 1:at + 1], w["v"][at - 1, 3], w["v"][at, 3] = w["k"][at - 1], 20.0, 3e38, -3e38
        want = go({**w, "v": torch.cat([w["v"][:at], x["v"][at:]])})[0]
    else:
        w[where][at, 0 if where == "b" else 3] = bad
    got, state = go(w)
    assert torch.allclose(got[:at], want[:at], rtol=1e-4, atol=1e-5)
    old = mops.DELTA_CHUNKED_FROM
    try:
        mops.DELTA_CHUNKED_FROM = 1 << 30
        scanned, state2 = go(w)
    finally:
        mops.DELTA_CHUNKED_FROM = old
    assert torch.equal(torch.isfinite(got), torch.isfinite(scanned)) and torch.equal(torch.isfinite(state), torch.isfinite(state2))
    fine = torch.isfinite(scanned)
    assert torch.allclose(got[fine], scanned[fine], rtol=1e-4, atol=1e-5)


@pytest.mark.parametrize("mode", [0, 1, 2, "delta"])
@pytest.mark.parametrize("chunks", [1, 3])
def test_chunks_in_spans(mops, monkeypatch, mode, chunks):
    """A workspace of one or three chunks instead of all: segments cut at any of theirs, the same bits."""
    H, d, e, lens, ctx = 2, 100, 72, [200, 1, 33, 500, 64, 7], [0, 4, 6, 3, 0, 0]
    g = torch.Generator(device=DEV).manual_seed(7)
    T, S = sum(lens), len(lens)
    start = i32(np.concatenate([[0], np.cumsum(lens)[:-1]]))
    q, k, v = (part(g, T, H * n, torch.bfloat16, 0) for n in (d, d, e))
    gi, gf, one = part(g, T, H, torch.bfloat16, 0), part(g, T, H, torch.bfloat16, 0), torch.ones(H, device=DEV)
    shapes = [(S, H, d, e)] if mode == "delta" else mops.memory_state_shapes(S, H, d, e, mode)
    first = [torch.randn(s, generator=g, device=DEV) for s in shapes]
    if mode == 1:
        first[1][:], first[2][:] = first[1][:, :, :1].clone(), first[2][:, :, :1].clone()
    lib = mops._lib.mixers_lib()
    query = "aphro_gated_delta_chunked_workspace" if mode == "delta" else "aphro_outer_memory_chunked_workspace"

    def go():
        state = tuple(s.clone() for s in first)
        if mode == "delta":
            out = mops.gated_delta_scan(q, k, v, gi, gf, one, one, state[0], i32(range(S)), start, i32(lens), i32(ctx), H, H, 1.0, max_q_len=500)
        else:
            kw = {0: dict(decay=0.9 * one), 1: dict(gate_i=gi, gate_f=gf), 2: dict(gate_i=gi, a_log=one, dt_bias=one, skip=one)}[mode]
            out = mops.outer_memory_scan(q, k, v, state, i32(range(S)), start, i32(lens), i32(ctx), H, mode, max_q_len=500, **kw)
        return (out, ) + state
    want, full = go(), getattr(lib, query)
    one_chunk = (lambda *a: full(1, 64, *a[2:-1], 64)) if mode != 1 else (lambda *a: full(1, 64, *a[2:-1], 64) + 12 * H * (T - 64))
    monkeypatch.setattr(lib, query, lambda *a: one_chunk(*a) if chunks == 1 else 3 * one_chunk(*a) - (24 * H * T if mode == 1 else 0))
    for x, y in zip(go(), want):
        assert torch.equal(x, y)


def test_chunks_do_not_take_memory_with_the_prompt(mops):
    """The workspace of prompts of a hundred thousand tokens: 256 MiB, and mode 1's three numbers a head and token."""
    lib, T = mops._lib.mixers_lib(), 100_000
    assert 200 << 20 < lib.aphro_gated_delta_chunked_workspace(1, T, 32, 128, 128, 32) <= 256 << 20
    for mode in (0, 1, 2):
        extra = 12 * 32 * T if mode == 1 else 0
        assert 200 << 20 < lib.aphro_outer_memory_chunked_workspace(1, T, 32, 128, 256, mode, 32) - extra <= 256 << 20
