"""What is measured of this framework: model steps as a serving program runs them, from one sequence to a full batch.

Three groups, by how the package is used:

* Llama geometry with quantised weights -- the package's main path.  Decoding is one forward and the LM head under a captured graph (the
  form bench.py serves); prompts, fresh or continued over cached context, go through the engine's ModelRunner.  Weights are GPTQ / AWQ
  int4 with groups of 128 or FP8 W8A8 with one scale per channel and token, keys and values 16-bit or FP8.  Fewer layers than the
  checkpoint has keep a state small; every layer does the same work.
* the routed experts of a Mixtral layer (int4), decoding and prompt-sized: FusedMoE with the router's logits at hand.
* the mixer families the engine serves (Fatudra, Nukezen, Vivisun: attention with distance tables, windows, chunks, latents; decaying,
  gated and delta-rule memories; state spaces) at the sizes of bench.py --mixers: fresh prompts, decoding, and prompt portions beside
  decoded tokens.

Weights, tokens and cached keys are made from the seed; lengths are made from the case alone."""
import dataclasses
import functools
import math
import random

import torch
from torch.nn import functional as F

PAGE = 16                                       # tokens of a page
HIDDEN, INTER, HEADS, KV_HEADS, HEAD, VOCAB, THETA, EPS = 4096, 14336, 32, 8, 128, 128256, 500000.0, 1e-5      # Llama-3-8B
GROUP = 128                                     # int4 quantisation group
EXPERTS, TOP = 8, 2                             # Mixtral-8x7B
MIX_VOCAB, MIX_LAYERS = 32000, 4
DEVICE = "cuda"


def listed():
    return [
        # one user: a chat reply, the smallest step there is
        {"name": "llama-int4-decode-1", "kind": "decode", "weights": "gptq", "kv": "auto", "dtype": "float16", "layers": 16, "seqs": 1,
         "ctx": 611, "ragged": False},
        # the package's headline: GPTQ int4, 32 sequences around a context of 1024
        {"name": "llama-int4-decode-32", "kind": "decode", "weights": "gptq", "kv": "auto", "dtype": "float16", "layers": 16, "seqs": 32,
         "ctx": 1040, "ragged": False},
        # a loaded server: AWQ int4, sequences of every age in one batch
        {"name": "llama-awq-decode-150", "kind": "decode", "weights": "awq", "kv": "auto", "dtype": "float16", "layers": 16, "seqs": 150,
         "ctx": 1500, "ragged": True},
        # long contexts: FP8 weights and FP8 keys and values
        {"name": "llama-fp8-decode-long", "kind": "decode", "weights": "fp8", "kv": "fp8", "dtype": "float16", "layers": 8, "seqs": 32,
         "ctx": 8192, "ragged": False},
        # a few prompts of ordinary length arriving together
        {"name": "llama-int4-prompts", "kind": "prompt", "weights": "gptq", "kv": "auto", "dtype": "float16", "layers": 4, "seqs": 5,
         "tokens": 430, "ctx": 0},
        # one long document
        {"name": "llama-fp8-prompt-8192", "kind": "prompt", "weights": "fp8", "kv": "fp8", "dtype": "bfloat16", "layers": 4, "seqs": 1,
         "tokens": 8192, "ctx": 0},
        # a Mixtral layer's experts while 32 sequences decode, and under a prompt
        {"name": "experts-decode-32", "kind": "experts", "weights": "gptq", "dtype": "float16", "tokens": 32},
        {"name": "experts-prompt-3000", "kind": "experts", "weights": "gptq", "dtype": "float16", "tokens": 3000},
        # a long prompt of each family (Vivisun: several, at the larger size)
        {"name": "fatudra-prompt-4096", "kind": "mixers", "family": "fatudra", "width": 2048, "prompts": 1, "tokens": 4096, "before": 0,
         "decodes": 0, "ctx": 0},
        {"name": "vivisun-prompts", "kind": "mixers", "family": "vivisun", "width": 4096, "prompts": 3, "tokens": 1400, "before": 0,
         "decodes": 0, "ctx": 0},
        # continuous batching: the next portion of a prompt beside decoded tokens
        {"name": "nukezen-mixed", "kind": "mixers", "family": "nukezen", "width": 2048, "prompts": 1, "tokens": 2000, "before": 1024,
         "decodes": 24, "ctx": 700},
        # a batch of recurrent states and keys that decodes
        {"name": "fatudra-decode-32", "kind": "mixers", "family": "fatudra", "width": 4096, "prompts": 0, "tokens": 0, "before": 0,
         "decodes": 32, "ctx": 1024},
    ]


def _between(rng, low, high):
    """A whole number from low to high, spread over its logarithm."""
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "experts", "mixers", "mixers"])
    if kind == "decode":
        weights = rng.choice(["gptq", "awq", "fp8"])
        seqs = _between(rng, 1, 192)
        ctx = _between(rng, 17, max(64, min(8192, 262144 // seqs)))
        return {"kind": kind, "weights": weights, "kv": rng.choice(["auto", "fp8"]),
                "dtype": rng.choice(["float16", "bfloat16"]) if weights == "fp8" else "float16",
                "layers": rng.choice([4, 8] if weights == "fp8" else [4, 8, 12]), "seqs": seqs, "ctx": ctx, "ragged": rng.random() < 0.5}
    if kind == "prompt":
        weights = rng.choice(["gptq", "awq", "fp8"])
        seqs = _between(rng, 1, 8)
        tokens = _between(rng, 24, 6144 // seqs)
        return {"kind": kind, "weights": weights, "kv": rng.choice(["auto", "fp8"]),
                "dtype": rng.choice(["float16", "bfloat16"]) if weights == "fp8" else "float16", "layers": rng.choice([2, 3, 4]), "seqs": seqs,
                "tokens": tokens, "ctx": rng.choice([0, 0, _between(rng, 16, 2048)])}
    if kind == "experts":
        return {"kind": kind, "weights": rng.choice(["gptq", "awq"]), "dtype": "float16", "tokens": _between(rng, 1, 4096)}
    family, width = rng.choice(["fatudra", "nukezen", "vivisun"]), rng.choice([2048, 2048, 4096])
    what = rng.choice(["prompts", "prompts", "mixed", "decode"])
    prompts = 0 if what == "decode" else _between(rng, 1, 6)
    return {"kind": kind, "family": family, "width": width, "prompts": prompts,
            "tokens": _between(rng, 48, (4096 if width == 2048 else 2560) // prompts) if prompts else 0,
            "before": _between(rng, 16, 1024) if what == "mixed" else 0,
            "decodes": 0 if what == "prompts" else _between(rng, 1, 32), "ctx": 0 if what == "prompts" else _between(rng, 16, 1024)}


# ---- shapes of a case -----------------------------------------------------------------------------------------------------------
def _lengths(count, most, ragged, salt):
    """``count`` lengths up to ``most``: all of them ``most``, or anything from a quarter of it."""
    r = random.Random(count * 100003 + most * 31 + salt)
    return [r.randint(max(1, most // 4), most) if ragged else most for _ in range(count)]


def _segments(case):
    """[(tokens in the caches, tokens of this step)]: prompt portions first, decoded tokens last."""
    if case["kind"] == "decode":
        return [(n, 1) for n in _lengths(case["seqs"], case["ctx"], case["ragged"], 1)]
    if case["kind"] == "prompt":
        n = _lengths(case["seqs"], case["tokens"], case["seqs"] > 1, 2)
        c = _lengths(case["seqs"], case["ctx"], case["seqs"] > 1, 3) if case["ctx"] else [0] * case["seqs"]
        return list(zip(c, n))
    n = _lengths(case["prompts"], case["tokens"], case["prompts"] > 1, 4)
    c = _lengths(case["prompts"], case["before"], case["prompts"] > 1, 5) if case["before"] else [0] * case["prompts"]
    return list(zip(c, n)) + [(x, 1) for x in _lengths(case["decodes"], case["ctx"], True, 6)]


def _pages(segments):
    """Page numbers of every segment, scattered over the pool as a server's are; the size of the pool."""
    need = [(c + n + PAGE - 1) // PAGE for c, n in segments]
    order = list(range(sum(need)))
    random.Random(7).shuffle(order)
    out, a = [], 0
    for k in need:
        out.append(order[a:a + k])
        a += k
    return out, len(order)


def _gen(seed, stream):
    return torch.Generator(device=DEVICE).manual_seed(seed * 1009 + stream)


def _normal(g, shape, std=1.0, mean=0.0, dtype=torch.float32):
    return torch.randn(shape, generator=g, device=DEVICE).mul_(std).add_(mean).to(dtype)


def _token_lists(case, seed, vocab):
    """Every segment's tokens, cached ones included."""
    g = torch.Generator().manual_seed(seed * 1009 + 3)
    return [torch.randint(0, vocab, (c + n, ), generator=g).tolist() for c, n in _segments(case)]


# ---- quantised linears ----------------------------------------------------------------------------------------------------------
def _words(g, shape, low=0, high=16):
    """Words of eight int4 values from low to high - 1."""
    word = torch.zeros(shape, dtype=torch.int32, device=DEVICE)
    for i in range(8):
        word |= torch.randint(low, high, shape, generator=g, device=DEVICE, dtype=torch.int32) << (4 * i)
    return word


def _quantised(g, weights, k, n, dtype, gain=1.0):
    """Checkpoint tensors of a [k -> n] linear: outputs of about ``gain`` times the inputs' size."""
    if weights == "fp8":
        w = _normal(g, (n, k), gain * k ** -0.5)
        scale = w.abs().amax(dim=1, keepdim=True) / 448.0
        return {"weight": (w / scale).to(torch.float8_e4m3fn), "weight_scale": scale}
    shape = (k // 8, n) if weights == "gptq" else (k, n // 8)
    scale = (torch.rand((k // GROUP, n), generator=g, device=DEVICE) * 0.5 + 0.75) * (gain / (4.4 * math.sqrt(k)))
    zero = 6 if weights == "gptq" else 7          # 7 to 9 about the weights' middle; GPTQ stores them less one
    return {"qweight": _words(g, shape, 1), "qzeros": _words(g, (k // GROUP, n // 8), zero, zero + 3), "scales": scale.to(dtype)}


def _nibbles(words, dim, order=range(8)):
    """int4 values of int32 words along ``dim``; ``order``: which nibble holds the j-th value."""
    parts = [(words >> (4 * i)) & 15 for i in order]
    return torch.stack(parts, dim + 1).flatten(dim, dim + 1)


AWQ_ORDER = (0, 4, 1, 5, 2, 6, 3, 7)


def _dequantised(t, weights):
    """[k, n] in 64 bits, as the checkpoint formats define it."""
    if weights == "fp8":
        return (t["weight"].double() * t["weight_scale"].double()).t()
    if weights == "gptq":
        q, z = _nibbles(t["qweight"], 0), _nibbles(t["qzeros"], 1) + 1
    else:
        q, z = _nibbles(t["qweight"], 1, AWQ_ORDER), _nibbles(t["qzeros"], 1, AWQ_ORDER)
    rows = torch.arange(q.shape[0], device=q.device) // GROUP
    return (q - z[rows]).double() * t["scales"].double()[rows]


def _linear_bytes(weights, k, n):
    return k * n + 4 * n if weights == "fp8" else k * n // 2 + (k // GROUP) * n * 2 + (k // GROUP) * n // 2


# ---- Llama ------------------------------------------------------------------------------------------------------------------------
LINEARS = {"qkv_proj": (HIDDEN, (HEADS + 2 * KV_HEADS) * HEAD), "o_proj": (HEADS * HEAD, HIDDEN), "gate_up_proj": (HIDDEN, 2 * INTER),
           "down_proj": (INTER, HIDDEN)}
# what joins the residual stream is small beside it, as in a checkpoint of 32 layers: 1 / sqrt(2 * 32)
GAINS = {"o_proj": 0.125, "down_proj": 0.125}


def _llama_weights(case, seed):
    """embedding, LM head and final norm, then one dict per layer -- made one after the other, so that a reader holds one layer."""
    g, dtype = _gen(seed, 1), getattr(torch, case["dtype"])
    yield {"embed": _normal(g, (VOCAB, HIDDEN), dtype=dtype), "head": _normal(g, (VOCAB, HIDDEN), HIDDEN ** -0.5, dtype=dtype),
           "norm": _normal(g, (HIDDEN, ), 0.1, 1.0, dtype)}
    for _ in range(case["layers"]):
        layer = {name: _quantised(g, case["weights"], k, n, dtype, GAINS.get(name, 1.0)) for name, (k, n) in LINEARS.items()}
        for name in ("input_layernorm", "post_attention_layernorm"):
            layer[name] = _normal(g, (HIDDEN, ), 0.1, 1.0, dtype)
        yield layer


def _llama_model(case, seed):
    """The model as a serving program holds it: loaded, and with the layouts of its decode kernels."""
    from aphrodite_engine_amd import model as M
    from aphrodite_engine_amd.quantization.awq import AWQConfig
    from aphrodite_engine_amd.quantization.fp8 import CompressedTensorsW8A8Fp8Config
    from aphrodite_engine_amd.quantization.gptq import GPTQConfig
    quant = {"gptq": lambda: GPTQConfig(4, GROUP, False), "awq": lambda: AWQConfig(4, GROUP, True, prepack=True),
             "fp8": lambda: CompressedTensorsW8A8Fp8Config(strategy="channel", is_static_input_scheme=False)}[case["weights"]]()
    cfg = dataclasses.replace(M.LLAMA3_8B, num_hidden_layers=case["layers"], max_position_embeddings=16384)
    dtype = getattr(torch, case["dtype"])
    with torch.device(DEVICE):
        model = M.LlamaForCausalLM(cfg, quant, dtype, case["kv"])
    parts = _llama_weights(case, seed)
    top = next(parts)
    model.embed_tokens.copy_(top["embed"])
    model.lm_head.copy_(top["head"])
    model.norm.copy_(top["norm"])
    del top
    for layer, t in zip(model.layers, parts):
        for name in LINEARS:
            for key, value in t[name].items():
                getattr(getattr(layer, name), key).data.copy_(value)
        layer.input_layernorm.copy_(t["input_layernorm"])
        layer.post_attention_layernorm.copy_(t["post_attention_layernorm"])
    model.cos_sin = M._rope_cache(HEAD, cfg.max_position_embeddings, THETA, dtype, torch.device(DEVICE))
    model.process_weights_after_loading()
    if case["weights"] == "fp8":
        for layer in model.layers:
            layer.enable_fp8_strips(32)
    else:
        for layer in model.layers:
            layer.enable_fused_silu(32, keep_original=False)
        for layer in model.layers:
            layer.enable_one_copy()
    return model


def _llama_caches(case, seed, pages, fill):
    """Paged keys and values of every layer: unit-variance numbers where ``fill``, else zero."""
    g, dtype = _gen(seed, 2), getattr(torch, case["dtype"])
    out = []
    for _ in range(case["layers"]):
        shape = (2, pages, PAGE * KV_HEADS * HEAD)
        if case["kv"] == "fp8":
            c = _normal(g, shape).to(torch.float8_e4m3fn).view(torch.uint8) if fill else torch.zeros(shape, dtype=torch.uint8, device=DEVICE)
        else:
            c = _normal(g, shape, dtype=dtype) if fill else torch.zeros(shape, dtype=dtype, device=DEVICE)
        out.append(c)
    return out


def _prepare_decode(case, seed):
    from aphrodite_engine_amd.attention.backend import MI355XAttentionMetadata
    model, segments = _llama_model(case, seed), _segments(case)
    tables, pool = _pages(segments)
    caches = _llama_caches(case, seed, pool, True)
    lens = [c + 1 for c, _ in segments]

    def dev(values, dtype):
        return torch.tensor(values, dtype=dtype, device=DEVICE)

    wide = max(len(t) for t in tables)
    meta = MI355XAttentionMetadata(
        num_prefills=0, num_prefill_tokens=0, num_decode_tokens=len(lens),
        slot_mapping=dev([t[c // PAGE] * PAGE + c % PAGE for t, (c, _) in zip(tables, segments)], torch.int64), seq_lens=None,
        seq_lens_tensor=dev(lens, torch.int32), max_query_len=None, max_prefill_seq_len=0, max_decode_seq_len=max(lens),
        query_start_loc=None, seq_start_loc=None, context_lens_tensor=None,
        block_tables=dev([t + [0] * (wide - len(t)) for t in tables], torch.int32), use_cuda_graph=False)
    ids = dev([t[-1] for t in _token_lists(case, seed, VOCAB)], torch.int64)
    positions = dev([c for c, _ in segments], torch.int64)
    state = {"model": model, "caches": caches, "meta": meta, "ids": ids, "positions": positions}

    def step():
        state["logits"] = model.compute_logits(model(ids, positions, caches, meta))

    with torch.no_grad():
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            step()
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, capture_error_mode="thread_local"):
            step()
    state["graph"] = graph
    return state


def _runner(model, caches, pool, slots):
    from aphrodite_engine_amd.engine import ModelRunner
    runner = ModelRunner(model, 1 if caches is not None else pool, PAGE, slots, DEVICE)
    if caches is not None:
        runner.caches = caches
    return runner


def _requests(segments, tables, tokens):
    from aphrodite_engine_amd.engine import Request
    return [(Request(str(i), t, len(t), num_computed=c, pages=p, slot=i), t[c:]) for i, ((c, _), p, t) in
            enumerate(zip(segments, tables, tokens))]


def _prepare_prompt(case, seed):
    segments = _segments(case)
    tables, pool = _pages(segments)
    runner = _runner(_llama_model(case, seed), _llama_caches(case, seed, pool, case["ctx"] > 0), pool, len(segments))
    return {"runner": runner, "segments": _requests(segments, tables, _token_lists(case, seed, VOCAB)), "want": [[n - 1] for _, n in segments]}


# ---- experts ----------------------------------------------------------------------------------------------------------------------
def _expert_weights(case, seed):
    g, dtype = _gen(seed, 1), getattr(torch, case["dtype"])
    for _ in range(EXPERTS):
        yield {"w1": _quantised(g, case["weights"], HIDDEN, INTER, dtype), "w3": _quantised(g, case["weights"], HIDDEN, INTER, dtype),
               "w2": _quantised(g, case["weights"], INTER, HIDDEN, dtype)}


def _expert_inputs(case, seed):
    g, dtype = _gen(seed, 2), getattr(torch, case["dtype"])
    return _normal(g, (case["tokens"], HIDDEN), dtype=dtype), _normal(g, (case["tokens"], EXPERTS), 1.5, dtype=dtype)


def _prepare_experts(case, seed):
    from aphrodite_engine_amd.moe import FusedMoE
    from aphrodite_engine_amd.quantization.awq import AWQConfig
    from aphrodite_engine_amd.quantization.gptq import GPTQConfig
    quant = GPTQConfig(4, GROUP, False) if case["weights"] == "gptq" else AWQConfig(4, GROUP, True, prepack=True)
    with torch.device(DEVICE):
        moe = FusedMoE(EXPERTS, TOP, HIDDEN, INTER, params_dtype=getattr(torch, case["dtype"]), renormalize=True, quant_config=quant)
    for e, t in enumerate(_expert_weights(case, seed)):
        for shard, tensors in t.items():
            for key, value in tensors.items():
                name = ("w2_" if shard == "w2" else "w13_") + key
                moe.weight_loader(getattr(moe, name), value, name, shard, e)
    for name, k in (("w13_g_idx", HIDDEN), ("w2_g_idx", INTER)):
        if hasattr(moe, name):
            p = getattr(moe, name)
            p.data.copy_((torch.arange(k, device=DEVICE) // GROUP).to(p.dtype).expand_as(p))
    moe.quant_method.process_weights_after_loading(moe)
    hidden, logits = _expert_inputs(case, seed)
    return {"moe": moe, "hidden": hidden, "logits": logits}


# ---- mixer families -----------------------------------------------------------------------------------------------------------------
def _sizes(width):
    if width == 2048:
        return {"ff": 5632, "heads": 16, "kv_heads": 4, "dim": 128, "mem_heads": 8, "ml_heads": 4}
    return {"ff": 11008, "heads": 32, "kv_heads": 8, "dim": 128, "mem_heads": 16, "ml_heads": 8}


def _mixer_config(family, width):
    """config.json of a stack (bench.py --mixers)."""
    s = _sizes(width)
    H, G, d = s["heads"], s["kv_heads"], s["dim"]
    mlp = {"kind": "dense", "ff": s["ff"]}
    c = {"architecture": family.capitalize(), "vocab": MIX_VOCAB, "width": width, "norm": {"eps": 1e-5}}
    if family == "fatudra":
        M = s["mem_heads"]
        par = {"type": "parallel", "mlp": mlp,
               "mixer": {"left": {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "bias_max": 4096, "scale": d ** -0.5,
                                  "q_temp": {"coef": 0.1, "every": 512}},
                         "right": {"heads": M, "dim": 64, "vdim": 128, "decay": [1.0 - 2.0 ** -(2 + 6 * i / (M - 1)) for i in range(M)]},
                         "left_scale": 1.0, "right_scale": 1.0}}
        ml = {"type": "mlstm", "mlp": mlp, "mixer": {"heads": s["ml_heads"], "dim": 128, "vdim": 256, "gate_cap": 15.0}}
        return {**c, "embedding": {"scale": 1.0}, "layers": [par, ml, par, par]}
    if family == "nukezen":
        delta = {"type": "channel_delta", "mlp": mlp, "mixer": {"heads": H, "kv_heads": H, "dim": d, "vdim": d, "conv": 4}}
        par = {"type": "parallel", "mlp": mlp,
               "mixer": {"left": {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "mask": {"size": 1024}, "rot": {"base": 500000.0, "dims": d},
                                  "scale": d ** -0.5},
                         "right": {"heads": 2 * width // 64, "vdim": 64, "state": 128, "groups": 8, "norm_groups": 8, "conv": 4},
                         "left_scale": 1.0, "right_scale": 1.0}}
        attn = {"type": "attention", "mlp": mlp, "mixer": {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "mask": {"size": 2048},
                                                           "softcap": 30.0, "bias_max": 4096, "scale": d ** -0.5}}
        return {**c, "embedding": {"scale": 1.0}, "layers": [delta, par, attn, dict(par, weights_of=1)]}
    attn = {"type": "attention", "mlp": mlp,
            "mixer": {"heads": H, "kv_heads": G, "dim": d, "vdim": d, "conv": 4, "scale": d ** -0.5,
                      "rot": {"base": 10000.0, "dims": d // 2, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}}
    latent = {"type": "latent_attention", "mlp": mlp, "mixer": {"heads": H, "dim": d, "vdim": d, "kv_rank": 512, "scale": d ** -0.5}}
    return {**c, "layers": [attn, latent], "loop": {"start": 0, "stop": 2, "times": 2}}


RANK, TABLE = 128, 32                           # low-rank inner size of decays and gates; rows of a distance table


def _mixer_weights(cfg, seed):
    """A checkpoint's tensors by name, in bfloat16."""
    g, W, width = _gen(seed, 1), {}, cfg["width"]

    def mat(name, rows, cols, gain=1.0):
        W[name] = _normal(g, (rows, cols), gain * cols ** -0.5, dtype=torch.bfloat16)

    def vec(name, n, mean=1.0, std=0.2):
        W[name] = _normal(g, (n, ), std, mean, torch.bfloat16)

    def ff(p, m, gain=1.0):
        mat(p + "gate", m["ff"], width, gain), mat(p + "up", m["ff"], width, gain), mat(p + "down", width, m["ff"])

    def conv(name, channels, taps):
        W[name] = _normal(g, (channels, taps), 0.5, dtype=torch.bfloat16)

    W["embed"] = _normal(g, (MIX_VOCAB, width), dtype=torch.bfloat16)
    family = cfg["architecture"].lower()
    vec("final.norm", width)
    if family != "nukezen":
        mat("head", MIX_VOCAB, width)
        vec("final.norm.b", width, 0.0)
    if family == "vivisun":
        W["final.norm.alpha"] = torch.tensor(0.5, dtype=torch.bfloat16, device=DEVICE)
    for i, lc in enumerate(cfg["layers"]):
        if lc.get("weights_of") is not None:
            continue
        p, m = f"l{i}.mix.", lc["mixer"]
        ff(f"l{i}.mlp.", lc["mlp"])
        for n in ("norm1", "norm2") + (("norm1b", "norm2b") if family == "fatudra" else ()):
            vec(f"l{i}.{n}", width)
            if family != "nukezen":
                vec(f"l{i}.{n}.b", width, 0.0)
            if family == "vivisun":
                W[f"l{i}.{n}.alpha"] = torch.tensor(0.5, dtype=torch.bfloat16, device=DEVICE)
        if lc["type"] == "mlstm":
            H, d, e = m["heads"], m["dim"], m["vdim"]
            mat(p + "q", H * d, width), mat(p + "k", H * d, width), mat(p + "v", H * e, width), mat(p + "g", H * e, width)
            mat(p + "i", H, width), mat(p + "f", H, width), vec(p + "i.b", H, 0.0, 1.0), vec(p + "f.b", H, 3.0, 1.0)
            vec(p + "norm", H * e), mat(p + "o", width, H * e)
        elif lc["type"] == "channel_delta":
            H, d, e = m["heads"], m["dim"], m["vdim"]
            for n, rows in (("q", H * d), ("k", H * d), ("v", H * e)):
                mat(p + n, rows, width), conv(p + n + ".conv", rows, m["conv"])
            mat(p + "b", H, width), mat(p + "a1", RANK, width), mat(p + "a2", H * d, RANK)
            mat(p + "g1", RANK, width), mat(p + "g2", H * e, RANK)
            W[p + "A_log"] = torch.rand(H, generator=g, device=DEVICE).mul_(1.9).add_(0.1).log_().to(torch.bfloat16)
            vec(p + "dt_bias", H * d, -3.0, 1.0), vec(p + "norm", e), mat(p + "o", width, H * e)
        elif lc["type"] == "parallel":
            L, R, l, r = m["left"], m["right"], p + "left.", p + "right."
            H, G, d, e = L["heads"], L["kv_heads"], L["dim"], L["vdim"]
            for n, rows in (("q", H * d), ("k", G * d), ("v", G * e)):
                mat(l + n, rows, width), vec(l + n + ".b", rows, 0.0)
            mat(l + "o", width, H * e)
            if family == "fatudra":
                W[l + "rel"] = _normal(g, (TABLE, H), dtype=torch.bfloat16)
                mat(l + "g", H, width), vec(l + "o.b", width, 0.0)
                N, dr, er = R["heads"], R["dim"], R["vdim"]
                mat(r + "q", N * dr, width), mat(r + "k", N * dr, width), mat(r + "v", N * er, width), mat(r + "g", N * er, width)
                mat(r + "o", width, N * er), vec(r + "norm", N * er)
            else:
                vec(l + "q.norm", d), vec(l + "k.norm", d), mat(l + "g", H * e, width)
                N, er = R["heads"], R["vdim"]
                ch = N * er + 2 * R["groups"] * R["state"]
                mat(r + "in", N * er + ch + N, width), conv(r + "conv", ch, R["conv"]), vec(r + "conv.b", ch, 0.0)
                W[r + "A_log"] = torch.rand(N, generator=g, device=DEVICE).mul_(1.9).add_(0.1).log_().to(torch.bfloat16)
                vec(r + "dt_bias", N, -3.0, 1.0), vec(r + "D", N), vec(r + "norm", N * er), mat(r + "o", width, N * er)
        elif lc["type"] == "attention":
            H, G, d, e = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
            for n, rows in (("q", H * d), ("k", G * d), ("v", G * e)):
                mat(p + n, rows, width)
                if family == "vivisun":
                    conv(p + n + ".conv", rows, m["conv"])
            mat(p + "o", width, H * e)
            per = (d, d) if family == "vivisun" else (H * d, G * d)
            vec(p + "q.norm", per[0]), vec(p + "k.norm", per[1])
            if family == "vivisun":
                mat(p + "g", H * e, width)
            else:
                W[p + "rel"] = _normal(g, (TABLE, H), dtype=torch.bfloat16)
        else:
            H, d, e, R = m["heads"], m["dim"], m["vdim"], m["kv_rank"]
            mat(p + "q", H * d, width), mat(p + "dkv", R, width), vec(p + "dkv.norm", R), mat(p + "uk", H * d, R), mat(p + "uv", H * e, R)
            vec(p + "sink", H, 1.0, 1.0), mat(p + "g", H, width), mat(p + "o", width, H * e)
    return W


def _mixer_model(case, seed):
    from aphrodite_engine_amd.fatudra import FatudraConfig, FatudraForCausalLM
    from aphrodite_engine_amd.nukezen import NukezenConfig, NukezenForCausalLM
    from aphrodite_engine_amd.vivisun import VivisunConfig, VivisunForCausalLM
    cfg = _mixer_config(case["family"], case["width"])
    W = _mixer_weights(cfg, seed)
    with torch.device(DEVICE):
        if case["family"] == "nukezen":
            model = NukezenForCausalLM(NukezenConfig.from_dict(cfg, {n: tuple(t.shape) for n, t in W.items()}))
        elif case["family"] == "fatudra":
            model = FatudraForCausalLM(FatudraConfig.from_dict(cfg))
        else:
            model = VivisunForCausalLM(VivisunConfig.from_dict(cfg))
    model.load_weights(W.items())
    return model.finalize()


def _prepare_mixers(case, seed):
    segments = _segments(case)
    tables, pool = _pages(segments)
    runner = _runner(_mixer_model(case, seed), None, pool, len(segments))
    tokens = _token_lists(case, seed, MIX_VOCAB)
    # what the caches hold is what a server's hold: the earlier tokens have gone through the model
    earlier = [(c, r) for (c, _), r in zip(segments, _requests([(0, c) for c, _ in segments], tables, tokens)) if c]
    while earlier:
        group, rows = [], 0
        while earlier and (not group or rows + earlier[0][0] <= 8192):
            c, (r, _) = earlier.pop(0)
            group.append((r, r.tokens[:c]))
            rows += c
        runner.execute(group, [[] for _ in group])
    return {"runner": runner, "segments": _requests(segments, tables, tokens), "want": [[n - 1] for _, n in segments]}


# ---- the interface ------------------------------------------------------------------------------------------------------------------
def prepare(case, seed):
    with torch.no_grad():
        return {"kind": case["kind"], **{"decode": _prepare_decode, "prompt": _prepare_prompt, "experts": _prepare_experts,
                                         "mixers": _prepare_mixers}[case["kind"]](case, seed)}


def run(state):
    if state["kind"] == "decode":
        state["graph"].replay()
        return {"logits": state["logits"]}
    if state["kind"] == "experts":
        with torch.no_grad():
            return {"hidden": state["moe"](state["hidden"], state["logits"])}
    logits = state["runner"].execute(state["segments"], state["want"])
    caches = state["runner"].caches
    if state["kind"] == "prompt":
        caches = [c.view(torch.float8_e4m3fn) if c.dtype == torch.uint8 else c for c in caches]
    return {"logits": logits, "caches": caches}


def _visible(c, n, window=0, chunk=0):
    """(query, key) pairs of n rows behind c cached ones."""
    if not window and not chunk:
        return n * c + n * (n + 1) // 2
    return sum(min(i + 1, window) if window else i % chunk + 1 for i in range(c, c + n))


def work(case):
    if case["kind"] == "experts":
        # every expert that some token chose; all of them once there are a few tokens
        reached = min(EXPERTS, EXPERTS * (1 - (1 - TOP / EXPERTS) ** case["tokens"]))
        weights = 2 * _linear_bytes(case["weights"], HIDDEN, INTER) + _linear_bytes(case["weights"], INTER, HIDDEN)
        return {"bytes": reached * weights + case["tokens"] * (2 * HIDDEN * 2 + 2 * EXPERTS), "flops": case["tokens"] * TOP * 6 * HIDDEN * INTER}
    segments = _segments(case)
    rows, ends = sum(n for _, n in segments), len(segments)
    if case["kind"] in ("decode", "prompt"):
        macs = sum(k * n for k, n in LINEARS.values())
        kv = 2 * KV_HEADS * HEAD * (1 if case["kv"] == "fp8" else 2)
        layer = sum(_linear_bytes(case["weights"], k, n) for k, n in LINEARS.values()) + sum(c + 2 * n if c else n for c, n in segments) * kv
        pairs = sum(_visible(c, n) for c, n in segments)
        return {"bytes": case["layers"] * layer + VOCAB * HIDDEN * 2 + rows * HIDDEN * 2 + ends * VOCAB * 2,
                "flops": case["layers"] * (2 * rows * macs + 4 * pairs * HEADS * HEAD) + 2 * ends * HIDDEN * VOCAB}
    cfg, width = _mixer_config(case["family"], case["width"]), case["width"]
    order = list(range(len(cfg["layers"]))) * (cfg.get("loop") or {"times": 1})["times"]
    nbytes, flops = MIX_VOCAB * width * 2 + rows * width * 2 + ends * MIX_VOCAB * 4, 2 * ends * width * MIX_VOCAB
    cached = sum(c + n for c, n in segments)
    for i in order:
        lc = cfg["layers"][i]
        m, params = lc["mixer"], 3 * width * lc["mlp"]["ff"]
        if lc["type"] == "mlstm":
            H, d, e = m["heads"], m["dim"], m["vdim"]
            params += width * H * (2 * d + 3 * e + 2)
            nbytes += 2 * ends * H * d * e * 4
            flops += 4 * rows * H * d * e
        elif lc["type"] == "channel_delta":
            H, d, e = m["heads"], m["dim"], m["vdim"]
            params += width * H * (2 * d + 2 * e + 1) + RANK * (2 * width + H * (d + e))
            nbytes += 2 * ends * H * d * e * 4
            flops += 6 * rows * H * d * e
        elif lc["type"] == "latent_attention":
            H, d, e, R = m["heads"], m["dim"], m["vdim"], m["kv_rank"]
            params += width * (H * (d + e + 1) + R) + R * H * (d + e)
            nbytes += cached * R * 2
            flops += 2 * sum(_visible(c, n) for c, n in segments) * H * (d + e)
        else:
            L = m.get("left", m)
            H, G, d, e = L["heads"], L["kv_heads"], L["dim"], L["vdim"]
            size = (L.get("mask") or {}).get("size", 0)
            sees = (lambda c, n: _visible(c, n, window=size)) if "left" in m else (lambda c, n: _visible(c, n, chunk=size))
            params += width * (H * d + G * (d + e) + H * e)
            nbytes += 2 * G * (d + e) * sum(min(c, size or c) + n for c, n in segments)
            flops += 2 * sum(sees(c, n) for c, n in segments) * H * (d + e)
            if case["family"] != "fatudra" and lc["type"] != "attention" or case["family"] == "vivisun":
                params += width * H * e
            if "right" in m and "decay" in m["right"]:
                R = m["right"]
                params += width * R["heads"] * (2 * R["dim"] + 3 * R["vdim"])
                nbytes += 2 * ends * R["heads"] * R["dim"] * R["vdim"] * 4
                flops += 4 * rows * R["heads"] * R["dim"] * R["vdim"]
            elif "right" in m:
                R = m["right"]
                params += width * (3 * R["heads"] * R["vdim"] + 2 * R["groups"] * R["state"] + R["heads"])
                nbytes += 2 * ends * R["heads"] * R["vdim"] * R["state"] * 4
                flops += 4 * rows * R["heads"] * R["vdim"] * R["state"]
        nbytes += 2 * params
        flops += 2 * rows * params
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # about four times the distance from 64 bits: 16-bit activations through a few layers (0.0013 in float16, 0.007 in the bfloat16
    # families); FP8 activations and keys add values that round the other way (0.008)
    if case["kind"] == "experts":
        return {"rel": 2e-3, "max": 0.05}
    if case["kind"] in ("decode", "prompt"):
        if case["weights"] == "fp8" or case["kv"] == "fp8":
            return {"rel": 0.03, "max": 0.5}
        return {"rel": 5e-3, "max": 0.1}
    return {"rel": 0.028, "max": 0.5}


# ---- 64 bits --------------------------------------------------------------------------------------------------------------------------
def _rms(x, w, eps, dims=-1):
    y = x / torch.sqrt((x * x).mean(dims, keepdim=True) + eps)
    return y if w is None else y * w


def _layer_norm(x, w, b, eps):
    return F.layer_norm(x, x.shape[-1:], w, b, eps)


def _attend(q, k, v, scale, first, window=0, chunk=0, cap=0.0, bias=None, sink=None):
    """Causal attention of one sequence: q [n, H, d] at positions first .., k [S, G, d], v [S, G, e] from position 0; ``bias`` [S, H] by
    distance; ``sink`` [H] joins the denominator."""
    n, H, _ = q.shape
    S, G = k.shape[0], k.shape[1]
    out = torch.empty(n, H, v.shape[-1], dtype=q.dtype, device=q.device)
    j = torch.arange(S, device=q.device)
    kt, vt = k.permute(1, 2, 0).contiguous(), v.transpose(0, 1).contiguous()
    step = max(1, min(n, (1 << 28) // (H * S)))
    for a in range(0, n, step):
        rows = q[a:a + step]
        i = torch.arange(first + a, first + a + rows.shape[0], device=q.device)
        gap = i[:, None] - j[None, :]
        see = gap >= 0
        if window:
            see &= gap < window
        if chunk:
            see &= i[:, None] // chunk == j[None, :] // chunk
        grouped = rows.transpose(0, 1).reshape(G, -1, rows.shape[2]).contiguous()
        s = torch.bmm(grouped, kt).view(H, rows.shape[0], S) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        if bias is not None:
            s = s + bias[gap.clamp(min=0)].permute(2, 0, 1)
        s = s.masked_fill(~see, -math.inf)
        if sink is not None:
            s = torch.cat([s, sink.view(H, 1, 1).expand(H, rows.shape[0], 1)], -1)
        p = torch.softmax(s, -1)[..., :S].contiguous()
        out[a:a + step] = torch.bmm(p.view(G, -1, S), vt).view(H, rows.shape[0], -1).transpose(0, 1)
    return out


def _rotate(x, positions, freq, mag=1.0, neighbours=False):
    """x [T, heads, n]: the first 2 len(freq) numbers of a head turn, as two halves or as neighbouring pairs."""
    a = positions.double()[:, None] * freq
    cos, sin = torch.cos(a)[:, None, :] * mag, torch.sin(a)[:, None, :] * mag
    h = freq.shape[0]
    at = (slice(0, 2 * h, 2), slice(1, 2 * h, 2)) if neighbours else (slice(0, h), slice(h, 2 * h))
    u, v = x[..., at[0]], x[..., at[1]]
    out = x.clone()
    out[..., at[0]], out[..., at[1]] = u * cos - v * sin, v * cos + u * sin
    return out


def _to_e4m3(x):
    return x.float().clamp(-448.0, 448.0).to(torch.float8_e4m3fn).double()


def _llama_exact(case, seed):
    segments = _segments(case)
    tables, pool = _pages(segments)
    filled = case["kind"] == "decode" or case["ctx"] > 0
    caches = _llama_caches(case, seed, pool, True) if filled else [None] * case["layers"]
    tokens = _token_lists(case, seed, VOCAB)
    new = [t[c:] for t, (c, _) in zip(tokens, segments)]
    ids = torch.tensor([x for t in new for x in t], device=DEVICE)
    pos = torch.cat([torch.arange(c, c + n, device=DEVICE) for c, n in segments])
    parts = _llama_weights(case, seed)
    top = next(parts)
    x = top["embed"][ids].double()
    freq = THETA ** (-torch.arange(0, HEAD, 2, device=DEVICE).double() / HEAD)
    kv8, w8 = case["kv"] == "fp8", case["weights"] == "fp8"

    def linear(t, name, h):
        w = _dequantised(t[name], case["weights"])
        if not w8:
            return h @ w
        scale = (h.abs().amax(-1, keepdim=True) / 448.0).clamp(min=1.0 / (448.0 * 512.0))
        return (_to_e4m3(h / scale) * scale) @ w

    def cached(cache, s, count):
        """Keys and values of the first ``count`` tokens of segment s."""
        c = cache[:, torch.tensor(tables[s][:(count + PAGE - 1) // PAGE], device=DEVICE)]
        c = c.view(torch.float8_e4m3fn) if kv8 else c
        width = 16 // c.element_size()
        k = c[0].view(-1, KV_HEADS, HEAD // width, PAGE, width).double().permute(0, 3, 1, 2, 4).reshape(-1, KV_HEADS, HEAD)
        v = c[1].view(-1, KV_HEADS, HEAD, PAGE).double().permute(0, 3, 1, 2).reshape(-1, KV_HEADS, HEAD)
        return k[:count], v[:count]

    for t, cache in zip(parts, caches):
        qkv = linear(t, "qkv_proj", _rms(x, t["input_layernorm"].double(), EPS)).view(-1, HEADS + 2 * KV_HEADS, HEAD)
        q, k, v = _rotate(qkv[:, :HEADS], pos, freq), _rotate(qkv[:, HEADS:HEADS + KV_HEADS], pos, freq), qkv[:, HEADS + KV_HEADS:]
        out, a = torch.empty_like(q), 0
        for s, (c, n) in enumerate(segments):
            kn, vn = k[a:a + n], v[a:a + n]
            if c:
                if kv8 and n == 1:                 # a decoded token attends to its own key as the cache holds it
                    kn, vn = _to_e4m3(kn), _to_e4m3(vn)
                ko, vo = cached(cache, s, c)
                kn, vn = torch.cat([ko, kn]), torch.cat([vo, vn])
            out[a:a + n] = _attend(q[a:a + n], kn, vn, HEAD ** -0.5, c)
            a += n
        x = x + linear(t, "o_proj", out.reshape(-1, HIDDEN))
        gate, up = linear(t, "gate_up_proj", _rms(x, t["post_attention_layernorm"].double(), EPS)).chunk(2, -1)
        x = x + linear(t, "down_proj", F.silu(gate) * up)
    last = torch.tensor([sum(n for _, n in segments[:i + 1]) - 1 for i in range(len(segments))], device=DEVICE)
    return _rms(x[last], top["norm"].double(), EPS) @ top["head"].double().t()


def _experts_exact(case, seed):
    hidden, logits = _expert_inputs(case, seed)
    x, p = hidden.double(), torch.softmax(logits.double(), -1)
    top, ids = p.topk(TOP, -1)
    top = top / top.sum(-1, keepdim=True)
    out = torch.zeros_like(x)
    for e, t in enumerate(_expert_weights(case, seed)):
        row, place = torch.where(ids == e)
        if not row.numel():
            continue
        w = {n: _dequantised(q, case["weights"]) for n, q in t.items()}
        out[row] += (F.silu(x[row] @ w["w1"]) * (x[row] @ w["w3"])) @ w["w2"] * top[row, place][:, None]
    return out


class _MixerExact:
    """The mixer families over whole sequences, without caches.  Rows of all sequences lie one after the other."""

    def __init__(self, cfg, W, lengths):
        self.cfg, self.raw, self.lengths, self.eps = cfg, W, lengths, cfg["norm"]["eps"]
        self.starts = [sum(lengths[:i]) for i in range(len(lengths))]
        self.pos = torch.cat([torch.arange(n, device=DEVICE) for n in lengths])

    def w(self, name):
        return self.raw[name].double()

    def lin(self, h, name):
        return h @ self.w(name).t()

    def per_sequence(self, fn, *tensors):
        return torch.cat([fn(*(t[a:a + n] for t in tensors)) for a, n in zip(self.starts, self.lengths)])

    def padded(self, t):
        """[sequences, longest, ...]; zeros behind the shorter ones."""
        return torch.nn.utils.rnn.pad_sequence([t[a:a + n] for a, n in zip(self.starts, self.lengths)], batch_first=True)

    def flat(self, t):
        return torch.cat([t[i, :n] for i, n in enumerate(self.lengths)])

    def conv(self, u, w, b=None):
        def one(x):
            taps = w.shape[1]
            pad = torch.cat([x.new_zeros(taps - 1, x.shape[1]), x])
            return sum(pad[j:j + x.shape[0]] * w[:, j] for j in range(taps))
        y = self.per_sequence(one, u)
        return y if b is None else y + b

    def bias(self, name, far):
        rel = self.w(name)
        rows, half = rel.shape[0], rel.shape[0] // 2
        at = [n if n < half else min(rows - 1, half + math.floor(math.log(n / half) / math.log(far / half) * (rows - half)))
              for n in range(max(self.lengths))]
        return rel[torch.tensor(at, device=DEVICE)]

    def fatudra_parallel(self, h, p, m):
        L, R, l, r = m["left"], m["right"], p + "left.", p + "right."
        H, G, d, e = L["heads"], L["kv_heads"], L["dim"], L["vdim"]
        q, k, v = (self.lin(h, l + n) + self.w(l + n + ".b") for n in "qkv")
        every, coef = L["q_temp"]["every"], L["q_temp"]["coef"]
        temp = 1.0 + coef * torch.log(((self.pos + 1) // every + 1).double())
        bias = self.bias(l + "rel", L["bias_max"])
        o = self.per_sequence(lambda a, b, c: _attend(a, b, c, L["scale"], 0, bias=bias[:a.shape[0]]),
                              q.view(-1, H, d) * temp[:, None, None], k.view(-1, G, d), v.view(-1, G, e))
        o = (o * torch.sigmoid(self.lin(h, l + "g"))[:, :, None]).reshape(-1, H * e)
        left = self.lin(o, l + "o") + self.w(l + "o.b")
        N, d, e = R["heads"], R["dim"], R["vdim"]
        q, k, v = (self.padded(F.silu(self.lin(h, r + n)).view(-1, N, z)) for n, z in (("q", d), ("k", d), ("v", e)))
        decay = torch.tensor(R["decay"], dtype=torch.float64, device=DEVICE)[None, :, None, None]
        S, o = q.new_zeros(q.shape[0], N, d, e), torch.empty_like(v)
        for t in range(q.shape[1]):
            S = decay * S + k[:, t, :, :, None] * v[:, t, :, None, :]
            o[:, t] = (S * q[:, t, :, :, None]).sum(2)
        o = _rms(self.flat(o).reshape(-1, N * e), self.w(r + "norm"), self.eps) * torch.sigmoid(self.lin(h, r + "g"))
        return m["left_scale"] * left + m["right_scale"] * self.lin(o, r + "o")

    def mlstm(self, h, p, m):
        H, d, e, cap = m["heads"], m["dim"], m["vdim"], m["gate_cap"]
        q, k, v = (self.padded(self.lin(h, p + n).view(-1, H, z)) for n, z in (("q", d), ("k", d), ("v", e)))
        q = q * d ** -0.5
        gi, gf = (cap * torch.tanh((self.lin(h, p + n) + self.w(p + n + ".b")) / cap) for n in "if")
        gi, gf = self.padded(gi), self.padded(F.logsigmoid(gf))
        S, n, top, o = q.new_zeros(q.shape[0], H, d, e), q.new_zeros(q.shape[0], H, d), q.new_zeros(q.shape[0], H), torch.empty_like(v)
        for t in range(q.shape[1]):
            now = torch.maximum(gf[:, t] + top, gi[:, t])
            a, b = torch.exp(gf[:, t] + top - now), torch.exp(gi[:, t] - now)
            S = a[..., None, None] * S + b[..., None, None] * k[:, t, :, :, None] * v[:, t, :, None, :]
            n, top = a[..., None] * n + b[..., None] * k[:, t], now
            den = torch.maximum((n * q[:, t]).sum(-1).abs(), torch.exp(-now)) + 1e-6
            o[:, t] = (S * q[:, t, :, :, None]).sum(2) / den[..., None]
        o = _rms(self.flat(o), None, self.eps).reshape(-1, H * e) * self.w(p + "norm") * torch.sigmoid(self.lin(h, p + "g"))
        return self.lin(o, p + "o")

    def channel_delta(self, h, p, m):
        H, d, e = m["heads"], m["dim"], m["vdim"]
        q, k, v = (F.silu(self.conv(self.lin(h, p + n), self.w(p + n + ".conv"))).view(-1, H, z) for n, z in (("q", d), ("k", d), ("v", e)))
        q, k = (z / torch.sqrt((z * z).sum(-1, keepdim=True) + 1e-6) for z in (q, k))
        beta = torch.sigmoid(self.lin(h, p + "b"))
        a = (self.lin(self.lin(h, p + "a1"), p + "a2") + self.w(p + "dt_bias")).view(-1, H, d)
        g = torch.exp(-torch.exp(self.w(p + "A_log"))[:, None] * F.softplus(a))
        q, k, v, beta, g = (self.padded(z) for z in (q * d ** -0.5, k, v, beta, g))
        S, o = q.new_zeros(q.shape[0], H, d, e), torch.empty_like(v)
        for t in range(q.shape[1]):
            S = g[:, t, :, :, None] * S
            u = beta[:, t, :, None] * (v[:, t] - (S * k[:, t, :, :, None]).sum(2))
            S = S + k[:, t, :, :, None] * u[:, :, None, :]
            o[:, t] = (S * q[:, t, :, :, None]).sum(2)
        gate = torch.sigmoid(self.lin(self.lin(h, p + "g1"), p + "g2"))
        return self.lin(_rms(self.flat(o), self.w(p + "norm"), self.eps).reshape(-1, H * e) * gate, p + "o")

    def nukezen_parallel(self, h, p, m):
        L, R, l, r = m["left"], m["right"], p + "left.", p + "right."
        H, G, d, e = L["heads"], L["kv_heads"], L["dim"], L["vdim"]
        q, k, v = (self.lin(h, l + n) + self.w(l + n + ".b") for n in "qkv")
        freq = L["rot"]["base"] ** (-torch.arange(0, L["rot"]["dims"], 2, device=DEVICE).double() / L["rot"]["dims"])
        q, k = (_rotate(_rms(z.view(-1, n, d), self.w(l + x + ".norm"), self.eps), self.pos, freq, neighbours=True)
                for z, n, x in ((q, H, "q"), (k, G, "k")))
        o = self.per_sequence(lambda a, b, c: _attend(a, b, c, L["scale"], 0, window=L["mask"]["size"]), q, k, v.view(-1, G, e))
        left = self.lin(o.reshape(-1, H * e) * torch.sigmoid(self.lin(h, l + "g")), l + "o")
        N, e, n, groups = R["heads"], R["vdim"], R["state"], R["groups"]
        inner = N * e
        z, xbc, dt = self.lin(h, r + "in").split([inner, inner + 2 * groups * n, N], -1)
        xbc = F.silu(self.conv(xbc, self.w(r + "conv"), self.w(r + "conv.b")))
        u, B, C = xbc.split([inner, groups * n, groups * n], -1)
        u, dt = u.reshape(-1, N, e), F.softplus(dt + self.w(r + "dt_bias"))
        B, C = (x.reshape(-1, groups, n).repeat_interleave(N // groups, 1) for x in (B, C))
        g = torch.exp(-torch.exp(self.w(r + "A_log")) * dt)
        pu, pB, pC, pdt, pg = (self.padded(x) for x in (u, B, C, dt, g))
        S, o = pu.new_zeros(pu.shape[0], N, n, e), torch.empty_like(pu)
        for t in range(pu.shape[1]):
            S = pg[:, t, :, None, None] * S + (pdt[:, t, :, None] * pB[:, t])[..., None] * pu[:, t, :, None, :]
            o[:, t] = (S * pC[:, t, :, :, None]).sum(2)
        y = (self.flat(o) + self.w(r + "D")[:, None] * u).reshape(-1, inner) * F.silu(z)
        y = _rms(y.view(-1, R["norm_groups"], inner // R["norm_groups"]), None, self.eps).reshape(-1, inner) * self.w(r + "norm")
        return m["left_scale"] * left + m["right_scale"] * self.lin(y, r + "o")

    def nukezen_attention(self, h, p, m):
        H, G, d, e = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k = (_rms(self.lin(h, p + n), self.w(p + n + ".norm"), self.eps) for n in "qk")
        bias, sink = self.bias(p + "rel", m["bias_max"]), torch.zeros(H, dtype=torch.float64, device=DEVICE)
        o = self.per_sequence(lambda a, b, c: _attend(a, b, c, m["scale"], 0, chunk=m["mask"]["size"], cap=m["softcap"],
                                                      bias=bias[:a.shape[0]], sink=sink),
                              q.view(-1, H, d), k.view(-1, G, d), self.lin(h, p + "v").view(-1, G, e))
        return self.lin(o.reshape(-1, H * e), p + "o")

    def vivisun_attention(self, h, p, m):
        H, G, d, e = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
        q, k, v = (self.conv(self.lin(h, p + n), self.w(p + n + ".conv")) for n in "qkv")
        rot, sc = m["rot"], m["rot"]["scaling"]
        dims, base = rot["dims"], rot["base"]
        freq = base ** (-torch.arange(0, dims, 2, device=DEVICE).double() / dims)
        low, high = (dims * math.log(sc["original"] / (2.0 * math.pi * n)) / (2.0 * math.log(base)) for n in (sc["fast"], sc["slow"]))
        low, high = max(math.floor(low), 0), min(math.ceil(high), dims - 1)
        ramp = ((torch.arange(dims // 2, device=DEVICE).double() - low) / max(high - low, 0.001)).clamp(0.0, 1.0)
        freq, mag = freq / sc["factor"] * ramp + freq * (1.0 - ramp), 0.1 * math.log(sc["factor"]) + 1.0
        q, k = (_rotate(_rms(z.view(-1, n, d), self.w(p + x + ".norm"), self.eps), self.pos, freq, mag) for z, n, x in ((q, H, "q"), (k, G, "k")))
        o = self.per_sequence(lambda a, b, c: _attend(a, b, c, m["scale"], 0), q, k, v.view(-1, G, e))
        return self.lin(o.reshape(-1, H * e) * torch.sigmoid(self.lin(h, p + "g")), p + "o")

    def latent_attention(self, h, p, m):
        H, d, e = m["heads"], m["dim"], m["vdim"]
        c = _rms(self.lin(h, p + "dkv"), self.w(p + "dkv.norm"), self.eps)
        k, v, sink = self.lin(c, p + "uk").view(-1, H, d), self.lin(c, p + "uv").view(-1, H, e), self.w(p + "sink")
        o = self.per_sequence(lambda a, b, z: _attend(a, b, z, m["scale"], 0, sink=sink), self.lin(h, p + "q").view(-1, H, d), k, v)
        return self.lin((o * torch.sigmoid(self.lin(h, p + "g"))[:, :, None]).reshape(-1, H * e), p + "o")

    def ff(self, h, p, act):
        return self.lin(act(self.lin(h, p + "gate")) * self.lin(h, p + "up"), p + "down")

    def forward(self, ids):
        cfg, eps, family = self.cfg, self.eps, self.cfg["architecture"].lower()
        gelu = functools.partial(F.gelu, approximate="tanh")
        x = start = self.raw["embed"][ids].double()
        times, count = (cfg.get("loop") or {"times": 1})["times"], len(cfg["layers"])
        for j in range(count * times):
            i = j % count
            lc = cfg["layers"][i]
            p = f"l{lc.get('weights_of', i)}."
            mix = getattr(self, {"mlstm": "mlstm", "channel_delta": "channel_delta", "latent_attention": "latent_attention"}.get(
                lc["type"], family + "_" + lc["type"]))
            if family == "vivisun":
                if j and i == 0:
                    x = x + start
                n1, n2 = (torch.tanh(self.w(p + n + ".alpha") * x) * self.w(p + n) + self.w(p + n + ".b") for n in ("norm1", "norm2"))
                x = x + mix(n1, p + "mix.", lc["mixer"]) + self.ff(n2, p + "mlp.", F.silu)
            elif family == "nukezen":
                x = x + _rms(mix(x, p + "mix.", lc["mixer"]), self.w(p + "norm1"), eps)
                x = x + _rms(self.ff(x, p + "mlp.", gelu), self.w(p + "norm2"), eps)
            else:
                def norm(z, n):
                    return _layer_norm(z, self.w(p + n), self.w(p + n + ".b"), eps)
                x = x + norm(mix(norm(x, "norm1"), p + "mix.", lc["mixer"]), "norm1b")
                x = x + norm(self.ff(norm(x, "norm2"), p + "mlp.", gelu), "norm2b")
        x = x[torch.tensor([a + n - 1 for a, n in zip(self.starts, self.lengths)], device=DEVICE)]
        if family == "vivisun":
            x = torch.tanh(0.5 * x) * self.w("final.norm") + self.w("final.norm.b")
        elif family == "nukezen":
            return self.lin(_rms(x, self.w("final.norm"), eps), "embed")
        else:
            x = _layer_norm(x, self.w("final.norm"), self.w("final.norm.b"), eps)
        return self.lin(x, "head")


def exact(case, seed):
    with torch.no_grad():
        if case["kind"] == "experts":
            return {"hidden": _experts_exact(case, seed)}
        if case["kind"] != "mixers":
            logits = _llama_exact(case, seed)
            return {"logits": logits} if case["kind"] == "decode" else {"logits": logits, "caches": None}
        cfg = _mixer_config(case["family"], case["width"])
        tokens = _token_lists(case, seed, MIX_VOCAB)
        ids = torch.tensor([x for t in tokens for x in t], device=DEVICE)
        return {"logits": _MixerExact(cfg, _mixer_weights(cfg, seed), [len(t) for t in tokens]).forward(ids), "caches": None}
