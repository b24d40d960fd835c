"""The work that a user of this framework has it do, as cases that a program can time and compare: generation with
greedy and nucleus sampling at the batch sizes and prompt lengths of single requests, of the serving loop and of a
full batch, scoring and every-position forwards from a few short requests to 16 x 2048 tokens, one decoder layer and the
sampler called on their own, in bfloat16 and float32.  Sizes are those of the repository's configurations and tests or
lie between them; `draw` gives further ones over the same ranges.

Weights are random, made once per configuration and kept while cases of that configuration are prepared, as a program
that serves a model keeps them; prompts, uniforms, activations and logits come from the seed.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "mesh-transformer-jax_amd"))

from mesh_transformer import layers, sampling  # noqa: E402
from mesh_transformer.engine import ROOT  # noqa: E402
from mesh_transformer.transformer_shard import CausalTransformer  # noqa: E402

DEV = "cuda:0"
REAL_VOCAB = 50257
SHIFT = 7919                     # the token that these weights make likely after token t is (t + SHIFT) % n_vocab

MODELS = {
    # GPT-J-6B as it is served: bfloat16 weights
    "6b_bf16": dict(layers=28, d_model=4096, n_heads=16, n_vocab=50400, norm="layernorm", pe="rotary", pe_rotary_dims=64,
                    seq=2048, cores_per_replica=1, early_cast=True),
    # the same model with the float32 weights that a configuration without early_cast gives
    "6b_f32": dict(layers=28, d_model=4096, n_heads=16, n_vocab=50400, norm="layernorm", pe="rotary", pe_rotary_dims=64,
                   seq=2048, cores_per_replica=1),
    # the two-layer float32 stack of the tests
    "tiny_f32": dict(layers=2, d_model=512, n_heads=8, n_vocab=50400, norm="layernorm", pe="rotary", pe_rotary_dims=32,
                     seq=168, cores_per_replica=1),
}


def listed():
    return [
        # the sampler called on its own with the logits of a serving batch
        dict(name="sample_b8", kind="sample", rows=8, top_k=0),
        # the small float32 stack: a 128-token prompt and 32 greedy steps, where launches and host work count
        dict(name="generate_tiny_f32", kind="generate", model="tiny_f32", batch=1, prompt=128, ragged=False, seq=168, steps=32,
             sampler="greedy", top_k=0),
        # a caller that drives a single decoder layer: one token on top of 1023 others
        dict(name="layer_decode_once", kind="layer_decode", model="6b_bf16", window=2047, keys=1023),
        # one request, greedy: 512-token prompt padded to 2048
        dict(name="generate_b1_greedy", kind="generate", model="6b_bf16", batch=1, prompt=512, ragged=False, seq=2048, steps=64,
             sampler="greedy", top_k=0),
        # a few short requests together
        dict(name="generate_b3_nucleus", kind="generate", model="6b_bf16", batch=3, prompt=97, ragged=True, seq=1024, steps=48,
             sampler="nucleus", top_k=0),
        # the serving loop's batch of 8 with prompts of unequal length and both filters
        dict(name="generate_b8_ragged", kind="generate", model="6b_bf16", batch=8, prompt=640, ragged=True, seq=2048, steps=32,
             sampler="nucleus", top_k=40),
        # a full batch on long prompts
        dict(name="generate_b32_nucleus", kind="generate", model="6b_bf16", batch=32, prompt=1024, ragged=False, seq=2048, steps=32,
             sampler="nucleus", top_k=0),
        # one request on float32 weights
        dict(name="generate_b1_f32", kind="generate", model="6b_f32", batch=1, prompt=200, ragged=False, seq=1024, steps=16,
             sampler="greedy", top_k=0),
        # scoring four short continuations, as zero-shot evaluation does with shrunk sequences
        dict(name="eval_4x61", kind="eval", model="6b_bf16", batch=4, tokens=61),
        # every-position logits of one prompt of odd length
        dict(name="forward_1x511", kind="forward", model="6b_bf16", batch=1, tokens=511),
        # evaluation loss on a batch of long rows
        dict(name="eval_5x1531", kind="eval", model="6b_bf16", batch=5, tokens=1531),
        # the full-context forward with logits at every position
        dict(name="forward_16x2048", kind="forward", model="6b_bf16", batch=16, tokens=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["sample", "layer_decode", "generate", "generate", "generate", "generate", "eval", "forward"])
    if kind == "sample":
        return dict(kind=kind, rows=_log_int(rng, 1, 64), top_k=rng.choice([0, 0, rng.randint(1, 200)]))
    if kind == "layer_decode":
        window = rng.randint(512, 2047)
        return dict(kind=kind, model=rng.choice(["6b_bf16", "6b_bf16", "6b_f32"]), window=window, keys=_log_int(rng, 16, window - 1))
    if kind == "generate":
        model = rng.choice(["6b_bf16"] * 6 + ["6b_f32", "tiny_f32"])
        steps = rng.randint(9, 48)
        if model == "tiny_f32":
            prompt = _log_int(rng, 8, 1500)
            return dict(kind=kind, model=model, batch=rng.randint(1, 4), prompt=prompt, ragged=rng.random() < 0.5,
                        seq=prompt + steps + rng.randint(0, 200), steps=steps, sampler=rng.choice(["greedy", "nucleus"]),
                        top_k=0)
        batch = 1 if model == "6b_f32" else _log_int(rng, 1, 32)
        prompt = _log_int(rng, 16, 512 if model == "6b_f32" else min(1900, 16384 // batch))
        return dict(kind=kind, model=model, batch=batch, prompt=prompt, ragged=rng.random() < 0.5,
                    seq=rng.choice([2048, min(2048, prompt + steps + rng.randint(0, 100))]), steps=steps,
                    sampler=rng.choice(["greedy", "nucleus"]), top_k=rng.choice([0, rng.randint(1, 100)]))
    tokens = _log_int(rng, 24, 2048)
    return dict(kind=kind, model="6b_bf16", batch=_log_int(rng, 1, max(1, 8192 // tokens)), tokens=tokens)


# ---------------------------------------------------------------------------------------------------------------- weights
def _tree(cfg, layer_ids, embed=True):
    """Random parameters with the scales of a trained stack: unit embeddings to which every layer adds a part, matrices
    that keep the size of their input, and a projection that favours one next token by a clear margin, as trained models
    do for most tokens (so that streams of two implementations that round differently can be compared)."""
    g = torch.Generator(device=DEV)
    g.manual_seed(2)
    d, V, F, n = cfg["d_model"], cfg["n_vocab"], 4 * cfg["d_model"], cfg["layers"]
    dt = torch.bfloat16 if cfg.get("early_cast") else torch.float32
    rn = lambda std, *s: torch.empty(*s, dtype=dt, device=DEV).normal_(0.0, std, generator=g)
    ln = lambda: {"scale": 1 + rn(0.1, 1, d), "offset": rn(0.05, 1, d)}
    t = {}
    for i in layer_ids:
        p = f"{ROOT}layer_{i}/~/"
        t[p + "replicated_layer_norm"] = ln()
        for name, std in (("linear", 1.28), ("linear_1", 1.28), ("linear_2", 1.28), ("linear_3", 0.64)):    # q, v, k, out
            t[p + name] = {"w": rn(std / d ** 0.5, 1, d, d)}
        t[p + "linear_4"] = {"w": rn(1.28 / d ** 0.5, 1, d, F), "b": rn(0.02, 1, F)}
        t[p + "linear_5"] = {"w": rn(0.35 / F ** 0.5, 1, F, d), "b": rn(0.02, 1, d)}
    if embed:
        emb = rn(1.0, 1, V, d)
        t[ROOT + "embedding_shard/~/linear"] = {"w": emb, "b": rn(0.02, 1, d)}
        t[ROOT + "projection_shard/~/replicated_layer_norm"] = ln()
        wp = rn(1.28 / d ** 0.5, 1, d, V)
        wp += (40.0 * (1 + 0.13 * n) ** 0.5 / d) * emb[0].roll(SHIFT, 0).t()
        t[ROOT + "projection_shard/~/linear"] = {"w": wp, "b": rn(0.02, 1, V)}
    return t


_kept = {}                       # the one model in use: (model name, case) -> network


def _network(case):
    """The model of a case, with its weights laid out.  One at a time: a program does not keep a second 6B model, nor
    the windows of every batch geometry it ever ran."""
    key = tuple(sorted((k, str(v)) for k, v in case.items()))
    if key not in _kept:
        _kept.clear()
        torch.cuda.empty_cache()
        cfg = MODELS[case["model"]]
        net = CausalTransformer(cfg, _tree(cfg, range(cfg["layers"])))
        net.engine()
        _kept[key] = net
    return _kept[key]


# ---------------------------------------------------------------------------------------------------------------- inputs
def _lengths(case):
    """Prompt lengths: all alike, or from a B-th of the longest to the longest."""
    B, P = case["batch"], case["prompt"]
    return np.array([max(1, P * (b + 1) // B) if case["ragged"] else P for b in range(B)], np.uint32)


def prepare(case, seed):
    rng = np.random.Generator(np.random.Philox(seed))
    kind = case["kind"]
    if kind == "sample":
        g = torch.Generator(device=DEV)
        g.manual_seed(seed)
        logits = torch.randn(case["rows"], 50400, generator=g, device=DEV) * 2.0
        opts = {"top_p": 0.9, "temp": 0.8}
        if case["top_k"]:
            opts["top_k"] = case["top_k"]
        return dict(kind=kind, logits=logits, u=rng.random(case["rows"]), opts=opts)
    cfg = MODELS[case["model"]]
    if kind == "layer_decode":
        one = dict(cfg, layers=1)
        layer = layers.TransformerLayerShard(one, "layer_0", 2.0, params=_tree(one, [0], embed=False))
        g = torch.Generator(device=DEV)
        g.manual_seed(seed)
        x = torch.randn(case["window"], cfg["d_model"], generator=g, device=DEV)
        _, state = layer.get_init_decode_state(x, case["keys"])
        return dict(kind=kind, layer=layer, state=state, x=torch.randn(1, cfg["d_model"], generator=g, device=DEV))
    net = _network(case)
    if kind == "generate":
        B, L, G = case["batch"], case["seq"], case["steps"]
        length = _lengths(case)
        ctx = np.zeros((B, L), np.uint32)                                  # left-padded with zeros
        for b in range(B):
            ctx[b, L - length[b]:] = rng.integers(0, REAL_VOCAB, int(length[b]))
        opts = {}
        if case["sampler"] == "nucleus":
            opts = {"top_p": np.full(B, 0.9), "temp": np.full(B, 0.8)}
            if case["top_k"]:
                opts["top_k"] = np.full(B, case["top_k"])
        return dict(kind=kind, net=net, ctx=ctx, length=length, steps=G, opts=opts, u=rng.random((B, G)),
                    sampler=sampling.greedy_sample if case["sampler"] == "greedy" else sampling.nucleaus_sample)
    B, T = case["batch"], case["tokens"]
    tokens = rng.integers(0, REAL_VOCAB, (B, T)).astype(np.uint32)
    if kind == "forward":
        return dict(kind=kind, net=net, tokens=tokens)
    likely = (tokens.astype(np.int64) + SHIFT) % cfg["n_vocab"]            # half of the targets are what the model expects
    target = np.where(rng.random((B, T)) < 0.5, likely, rng.integers(0, REAL_VOCAB, (B, T))).astype(np.uint32)
    target[:, -1] = rng.integers(0, REAL_VOCAB, B)                         # (the last token's loss is returned on its own)
    length = np.array([max(1, T - b) for b in range(B)])
    return dict(kind=kind, net=net, sample={"obs": tokens, "target": target, "ctx_length": length})


def run(state):
    kind = state["kind"]
    if kind == "sample":
        return sampling.nucleaus_sample(state["u"], state["logits"], None, **state["opts"])[0]
    if kind == "layer_decode":
        delta, after = state["layer"].decode_once(state["state"], state["x"])
        return {"delta": delta, "k": after["k"], "v": after["v"]}
    if kind == "generate":
        _, out = state["net"].generate(state["ctx"], state["length"], state["steps"], state["opts"], return_logits=True,
                                       uniforms=state["u"], sampler=state["sampler"])
        return {"tokens": out[0], "logits": out[2]}
    if kind == "forward":
        return state["net"].forward(state["tokens"])
    return state["net"].eval(state["sample"])


# ---------------------------------------------------------------------------------------------------------------- cost
def work(case):
    """Weights once per pass over the stack (once per decode step, once per prefill), the keys and values of every step,
    the operations of the matrix products and of causal attention, the results."""
    kind = case["kind"]
    if kind == "sample":
        return {"bytes": case["rows"] * (50400 * 4 + 4), "flops": 0}
    cfg = MODELS[case["model"]]
    d, V, n = cfg["d_model"], cfg["n_vocab"], cfg["layers"]
    e = 2 if cfg.get("early_cast") else 4                                  # bytes of a weight, a key and a value
    layer = 12 * d * d
    if kind == "layer_decode":
        return {"bytes": layer * e + 2 * (case["keys"] + 1) * d * e + 2 * d * 4, "flops": 2 * layer + 4 * d * (case["keys"] + 1)}
    causal = lambda t: 4 * d * t * (t + 1) / 2
    if kind == "generate":
        B, G = case["batch"], case["steps"]
        pre = [int(p) - 1 for p in _lengths(case)]                         # the last prompt token is the first step's input
        nbytes = (n * layer * e if sum(pre) else 0) + sum(pre) * n * 2 * d * e
        flops = sum(pre) * 2 * n * layer + n * sum(causal(p) for p in pre)
        for t in range(G):
            nbytes += (n * layer + d * V) * e + sum(p + t + 1 for p in pre) * n * 2 * d * e + B * V * 4
            flops += B * 2 * (n * layer + d * V) + n * sum(4 * d * (p + t + 1) for p in pre)
        return {"bytes": nbytes, "flops": flops}
    B, T = case["batch"], case["tokens"]
    flops = B * T * 2 * (n * layer + d * V) + n * B * causal(T)
    out = B * T * V * 4 if kind == "forward" else B * T * 5
    return {"bytes": (n * layer + d * V) * e + B * T * d * e + out, "flops": flops}


def tolerance(case):
    """float32: two kernels for the same product (matrix-vector, matrix-matrix) give logits 2e-6 apart.  bfloat16: the same
    weights with float32 operands throughout give logits 5e-4 (one row: 4e-4) and losses 3e-4 away, at most 3e-3 of their
    root mean square.  Tokens are the same in all of them."""
    if case["kind"] == "sample":
        return "exact"
    if case["model"] != "6b_bf16":
        return {"rel": 1e-5, "max": 1e-4}
    return {"rel": 2e-3, "max": 2e-2}
