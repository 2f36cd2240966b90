"""What the speed of this engine is measured on: steps as a serving program runs them, through the step runner.

A case names a model, its type and a step (or a short run of steps); ``prepare`` builds the model, the paged cache and the
requests that are in it, ``run`` is one pass, and ``exact`` is the same pass in 64-bit arithmetic over whole sequences.

Sizes are those of the benchmark (``bench.py``): the Qwen3-0.6B shape with all its layers, the Qwen3-8B and 32B shapes with
6 and 4 of theirs, and the Papivik and Mukenex designs at the width of the 0.6B shape.  Weights are random, prompts are
uniform token ids, requests in one step have contexts of unlike lengths.

A step's chosen tokens are worked out in the step (they are what the next one is fed) and are not compared: among 151,936
random logits the two largest are often closer than bfloat16 resolves.  The logits are.
"""

from __future__ import annotations

import math
import random

import numpy as np
import torch

DEVICE = "cuda:0"
BLOCK_SIZE = 16
VOCAB = 151936
DTYPES = {"bf16": torch.bfloat16, "f32": torch.float32}

QWEN3 = {
    "architectures": ["Qwen3ForCausalLM"], "model_type": "qwen3", "hidden_act": "silu", "attention_bias": False,
    "sliding_window": None, "head_dim": 128, "num_key_value_heads": 8, "rms_norm_eps": 1e-6, "rope_theta": 1000000.0,
    "vocab_size": VOCAB,
}


def _qwen3(hidden, inter, layers, heads, positions, tied):
    return dict(QWEN3, hidden_size=hidden, intermediate_size=inter, num_hidden_layers=layers, num_attention_heads=heads,
                max_position_embeddings=positions, tie_word_embeddings=tied)


def _papivik():
    mlp = {"kind": "dense", "ff": 3072}
    kinds = [
        {"type": "lightning", "mlp": mlp,
         "mixer": {"heads": 8, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** (-5 - 3 * h / 7) for h in range(8)]}},
        {"type": "mlstm", "mlp": mlp, "mixer": {"heads": 4, "dim": 128, "vdim": 256, "gate_cap": 15.0}},
        {"type": "parallel", "mlp": mlp, "mixer": {
            "left": {"heads": 16, "kv_heads": 8, "dim": 128, "vdim": 128, "conv": 4, "scale": 128 ** -0.5,
                     "rot": {"dims": 64, "base": 1000000.0}},
            "right": {"heads": 8, "kv_heads": 4, "dim": 128, "vdim": 128, "conv": 4},
            "left_scale": 0.5, "right_scale": 0.5}},
    ]
    return {"architecture": "Papivik", "embedding": {"scale": 1.0}, "norm": {"eps": 1e-6}, "vocab": VOCAB, "width": 1024,
            "layers": kinds + kinds}


def _mukenex():
    experts = {"kind": "moe", "expert": {"ff": 1536}, "router": {"experts": 8, "top": 2}}
    kinds = [
        {"type": "lightning", "mlp": {"kind": "dense", "ff": 3072},
         "mixer": {"heads": 8, "dim": 128, "vdim": 128, "decay": [1.0 - 2.0 ** (-5 - 3 * h / 7) for h in range(8)]}},
        {"type": "latent_attention", "mlp": experts,
         "mixer": {"heads": 16, "dim": 64, "rot_dim": 64, "vdim": 128, "kv_rank": 192, "scale": 128 ** -0.5,
                   "rot": {"dims": 64, "base": 1000000.0}, "mask": {"size": 512}}},
        {"type": "attention", "mlp": experts,
         "mixer": {"heads": 16, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": {"size": 512}}},
    ]
    return {"architecture": "Mukenex", "norm": {"eps": 1e-6}, "vocab": VOCAB, "width": 1024, "streams": 4,
            "logit_softcap": 30.0, "layers": kinds + kinds}


CONFIGS = {
    "qwen3-0.6b": _qwen3(1024, 3072, 28, 16, 4096, True),
    "qwen3-8b": _qwen3(4096, 12288, 6, 32, 16384, False),
    "qwen3-32b": _qwen3(5120, 25600, 4, 64, 16384, False),
    "papivik": _papivik(),
    "mukenex": _mukenex(),
}


def _case(name, model, dtype, decodes=0, context=0, prompts=0, tokens=0, behind=0, steps=0):
    """``decodes`` requests of up to ``context`` tokens decode one token each; beside them ``prompts`` requests bring up to
    ``tokens`` tokens of their prompts, each ``behind`` tokens that are in the cache already; behind the first step come ``steps`` further
    ones in which the requests with prompts decode one token each."""
    case = {"model": model, "dtype": dtype, "decodes": decodes, "context": context, "prompts": prompts, "tokens": tokens,
            "behind": behind, "steps": steps}
    return {"name": name, **case} if name else case


def listed():
    return [
        # one user, one token at a time: the smallest step there is, all chains and launches
        _case("decode_1", "qwen3-0.6b", "bf16", decodes=1, context=512),
        # the headline: a few users
        _case("decode_8", "qwen3-0.6b", "bf16", decodes=8, context=512),
        # a full server with long conversations: the keys and values are most of the bytes
        _case("decode_64_long", "qwen3-0.6b", "bf16", decodes=64, context=3968),
        # a large model's layers: the weights are most of the bytes
        _case("decode_24_32b", "qwen3-32b", "bf16", decodes=24, context=1500),
        # a short question; its length is no multiple of anything
        _case("prompt_37", "qwen3-0.6b", "bf16", prompts=1, tokens=37),
        # the headline's prompt
        _case("prompt_2048", "qwen3-0.6b", "bf16", prompts=1, tokens=2048),
        # a document before a large model's layers: the largest step
        _case("prompt_8192_8b", "qwen3-8b", "bf16", prompts=1, tokens=8192),
        # a server under load: a portion of one prompt beside everybody's next token
        _case("mixed_63_512_8b", "qwen3-8b", "bf16", decodes=63, context=1024, prompts=1, tokens=512, behind=1024),
        # the 32-bit type, which checks of a checkpoint and trace replays run in
        _case("decode_8_f32", "qwen3-0.6b", "f32", decodes=8, context=512),
        _case("prompt_700_f32", "qwen3-0.6b", "f32", prompts=1, tokens=700),
        # the designs with state: two questions of unlike length and the first tokens of their answers
        _case("papivik_2x1500_4", "papivik", "bf16", prompts=2, tokens=1500, steps=4),
        # copies of the stream, experts, latent attention
        _case("mukenex_3x600", "mukenex", "bf16", prompts=3, tokens=600),
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prompt", "prompt", "mixed", "decode_f32", "prompt_f32", "papivik", "mukenex", "large"])
    if kind == "decode":
        decodes = _log(rng, 1, 64)
        return _case("", "qwen3-0.6b", "bf16", decodes=decodes, context=_log(rng, 24, 3968))
    if kind == "prompt":
        prompts = _log(rng, 1, 6)
        return _case("", "qwen3-0.6b", "bf16", prompts=prompts, tokens=_log(rng, 2, 3000 // prompts), behind=rng.choice([0, 0, _log(rng, 1, 1000)]))
    if kind == "mixed":
        return _case("", rng.choice(["qwen3-0.6b", "qwen3-8b"]), "bf16", decodes=_log(rng, 1, 63), context=_log(rng, 24, 1024),
                     prompts=1, tokens=_log(rng, 16, 1024), behind=rng.choice([0, _log(rng, 1, 2000)]))
    if kind == "decode_f32":
        return _case("", "qwen3-0.6b", "f32", decodes=_log(rng, 1, 16), context=_log(rng, 24, 1000))
    if kind == "prompt_f32":
        prompts = _log(rng, 1, 3)
        return _case("", "qwen3-0.6b", "f32", prompts=prompts, tokens=_log(rng, 2, 700 // prompts))
    if kind == "papivik":
        return _case("", "papivik", "bf16", prompts=_log(rng, 1, 8), tokens=_log(rng, 5, 380), steps=rng.randrange(0, 6))
    if kind == "mukenex":
        return _case("", "mukenex", "bf16", prompts=_log(rng, 1, 8), tokens=_log(rng, 5, 380), steps=0)
    model = rng.choice(["qwen3-8b", "qwen3-32b"])
    if rng.random() < 0.5:
        return _case("", model, "bf16", decodes=_log(rng, 1, 24), context=_log(rng, 24, 1500))
    return _case("", model, "bf16", prompts=1, tokens=_log(rng, 2, 4096))


# -- weights -------------------------------------------------------------------------------------------------------------------

def _declared(config):
    """(name, shape, how it is drawn) of every tensor of a checkpoint of this configuration, in a fixed order."""
    def matrix(name, *shape):
        return [(name, shape, "matrix")]

    def gain(name, *shape):
        return [(name, shape, "gain")]

    out = []
    if "num_hidden_layers" in config:
        h, i, d = config["hidden_size"], config["intermediate_size"], config["head_dim"]
        q, kv = config["num_attention_heads"] * d, config["num_key_value_heads"] * d
        out += matrix("model.embed_tokens.weight", VOCAB, h)
        for n in range(config["num_hidden_layers"]):
            p = f"model.layers.{n}."
            out += gain(p + "input_layernorm.weight", h) + gain(p + "post_attention_layernorm.weight", h)
            out += matrix(p + "self_attn.q_proj.weight", q, h) + matrix(p + "self_attn.k_proj.weight", kv, h)
            out += matrix(p + "self_attn.v_proj.weight", kv, h) + matrix(p + "self_attn.o_proj.weight", h, q)
            out += gain(p + "self_attn.q_norm.weight", d) + gain(p + "self_attn.k_norm.weight", d)
            out += matrix(p + "mlp.gate_proj.weight", i, h) + matrix(p + "mlp.up_proj.weight", i, h)
            out += matrix(p + "mlp.down_proj.weight", h, i)
        out += gain("model.norm.weight", h)
        if not config["tie_word_embeddings"]:
            out += matrix("lm_head.weight", VOCAB, h)
        return out
    w = config["width"]
    copies = config.get("streams")
    stream_gain = "gain_around_zero" if copies else "gain"
    out += matrix("embed", VOCAB, w)
    for n, layer in enumerate(config["layers"]):
        p, x, m = f"l{n}.", f"l{n}.mix.", layer["mixer"]
        out += [(p + "norm1", (w,), stream_gain), (p + "norm2", (w,), stream_gain)]
        if copies:
            for hc in ("hc1.", "hc2."):
                out += [(p + hc + "in", (copies,), "copy_in"), (p + hc + "out", (copies,), "gain"),
                        (p + hc + "mix", (copies, copies), "copy_mix")]
        if layer["type"] in ("lightning", "mlstm"):
            k, v = m["heads"] * m["dim"], m["heads"] * m["vdim"]
            out += matrix(x + "q", k, w) + matrix(x + "k", k, w) + matrix(x + "v", v, w) + matrix(x + "g", v, w)
            out += matrix(x + "o", w, v) + gain(x + "norm", v)
            if layer["type"] == "mlstm":
                for g in ("i", "f"):
                    out += matrix(x + g, m["heads"], w) + matrix(x + g + ".b", m["heads"])
        elif layer["type"] == "parallel":
            a, b = m["left"], m["right"]
            q, k, v = a["heads"] * a["dim"], a["kv_heads"] * a["dim"], a["kv_heads"] * a["vdim"]
            l, r = x + "left.", x + "right."
            for name, width in (("q", q), ("k", k), ("v", v)):
                out += matrix(l + name, width, w) + [(l + name + ".conv", (width, a["conv"]), "filter")]
            out += matrix(l + "o", w, a["heads"] * a["vdim"]) + gain(l + "q.norm", a["dim"]) + gain(l + "k.norm", a["dim"])
            k, v = b["kv_heads"] * b["dim"], b["heads"] * b["vdim"]
            for name, width in (("q", k), ("k", k), ("v", v)):
                out += matrix(r + name, width, w) + [(r + name + ".conv", (width, b["conv"]), "filter")]
            out += matrix(r + "b", b["heads"], w) + matrix(r + "a", b["heads"], w)
            out += matrix(r + "A_log", b["heads"]) + matrix(r + "dt_bias", b["heads"])
            out += gain(r + "norm", b["vdim"]) + matrix(r + "g", v, w) + matrix(r + "o", w, v)
        elif layer["type"] == "latent_attention":
            H, rank = m["heads"], m["kv_rank"]
            out += matrix(x + "q", H * (m["dim"] + m["rot_dim"]), w) + matrix(x + "dkv", rank + m["rot_dim"], w)
            out += gain(x + "dkv.norm", rank) + matrix(x + "uk", H * m["dim"], rank) + matrix(x + "uv", H * m["vdim"], rank)
            out += matrix(x + "sink", H) + matrix(x + "g", H * m["vdim"], w) + matrix(x + "o", w, H * m["vdim"])
        else:
            q, k, v = m["heads"] * m["dim"], m["kv_heads"] * m["dim"], m["kv_heads"] * m["vdim"]
            for name, width in (("q", q), ("k", k), ("v", v)):
                out += matrix(x + name, width, w) + matrix(x + name + ".b", width)
            out += matrix(x + "o", w, m["heads"] * m["vdim"]) + gain(x + "q.norm", m["dim"]) + gain(x + "k.norm", m["dim"])
        mlp, f = layer["mlp"], p + "mlp."
        if mlp["kind"] == "dense":
            out += matrix(f + "up", mlp["ff"], w) + matrix(f + "down", w, mlp["ff"])
        else:
            ff, count = mlp["expert"]["ff"], mlp["router"]["experts"]
            for e in range(count):
                out += matrix(f"{f}e{e}.gate", ff, w) + matrix(f"{f}e{e}.up", ff, w) + matrix(f"{f}e{e}.down", w, ff)
            out += [(f + "table", (VOCAB, mlp["router"]["top"]), f"table:{count}")]
    out += [("final.norm", (w,), stream_gain)]
    out += matrix("head", VOCAB, w)
    return out


def _weights(model, dtype):
    """The tensors of a checkpoint, drawn on the GPU: matrices N(0, 0.02), gains around one."""
    g = torch.Generator(device=DEVICE)
    g.manual_seed(20240611)
    out = {}
    for name, shape, how in _declared(CONFIGS[model]):
        if how.startswith("table:"):
            x = torch.rand((shape[0], int(how[6:])), generator=g, device=DEVICE)
            out[name] = x.argsort(dim=1)[:, :shape[1]].to(torch.int32).contiguous()
            continue
        x = torch.randn(shape, generator=g, device=DEVICE, dtype=torch.float32)
        if how == "gain":
            x = 1.0 + 0.1 * x
        elif how == "gain_around_zero":
            x = 0.1 * x
        elif how == "filter":       # the taps of a short convolution: the current token's leads
            x = x * 0.3 / shape[-1] ** 0.5
            x[:, -1] += 0.7
        elif how == "copy_in":      # around an even share of every copy of the stream
            x = (1.0 + 0.1 * x) / shape[0]
        elif how == "copy_mix":     # around keeping every copy as it is
            x = torch.eye(shape[0], device=DEVICE) + 0.05 * x
        else:
            x = 0.02 * x
        out[name] = x.to(dtype)
    return out


_built: dict = {}       # the model of the last case: a program loads its weights once and keeps them for all its requests


def _model(name, dtype):
    from paged_llm_rs_amd import load_config
    from paged_llm_rs_amd.parts.model import build_model

    key = (name, dtype)
    if key not in _built:
        _built.clear()
        _built[key] = build_model(load_config(CONFIGS[name]), _weights(name, DTYPES[dtype]), dtype, DEVICE)
    return _built[key]


# -- requests -------------------------------------------------------------------------------------------------------------------

def _lengths(rng, count, most):
    """``count`` lengths from about half of ``most`` up to it; the first is ``most`` itself."""
    return [most if i == 0 else rng.randint((most + 1) // 2, most) for i in range(count)]


def _requests(case, seed):
    """[(token ids, how many of them are in the cache before the pass, how many the first step brings)]; what is left of a
    request's ids is decoded one a step behind the first."""
    rng = random.Random(seed * 1000003 + 17)
    draws = np.random.RandomState(seed % (1 << 31))
    sizes = [(n, 1) for n in _lengths(rng, case["decodes"], case["context"])] if case["decodes"] else []
    if case["prompts"]:
        sizes += [(case["behind"], n) for n in _lengths(rng, case["prompts"], case["tokens"])]
    out = []
    for i, (inside, brings) in enumerate(sizes):
        more = case["steps"] if i >= case["decodes"] else 0
        out.append((draws.randint(0, VOCAB, inside + brings + more).tolist(), inside, brings))
    return out


class State:
    """A serving program between two steps.  The step's keys and values in the pages of the last layer, which follow from
    those of all layers before it, stand for what a step writes."""

    def __init__(self, case, model, cache, runner, requests):
        self.case, self.model, self.cache, self.runner = case, model, cache, runner
        self.requests = requests
        self.last_layer = len(model.blocks) - 1


FILL = 2048     # tokens of a step that brings contexts into the cache


def prepare(case, seed):
    from paged_llm_rs_amd.cache import PagedCache
    from paged_llm_rs_amd.engine.batch import StepEntry
    from paged_llm_rs_amd.engine.step import StepRunner, commit_step, run_step

    model = _model(case["model"], case["dtype"])
    requests = _requests(case, seed)
    # (room for requests of the case's largest sizes, whatever sizes these are of)
    longest = case["behind"] + case["tokens"] + case["steps"]
    pages = case["decodes"] * (case["context"] // BLOCK_SIZE + 1) + case["prompts"] * (-(-longest // BLOCK_SIZE))
    cache = PagedCache(model.cache_layout, BLOCK_SIZE, pages, DTYPES[case["dtype"]], torch.device(DEVICE), max_seqs=len(requests) + 1)
    runner = StepRunner(model, cache)
    for i, (ids, inside, brings) in enumerate(requests):
        if inside == 0:
            continue
        slot = cache.manager.add_sequence(i + 1)
        for at in range(0, inside, FILL):
            part = ids[at:min(at + FILL, inside)]
            if not cache.manager.reserve(i + 1, len(part)):
                raise MemoryError("no pages")
            step = [StepEntry(i + 1, part, at, [], state_slot=slot, fresh_state=at == 0 and slot >= 0)]
            run_step(model, cache, step)
            commit_step(cache, step)
        if not cache.manager.reserve(i + 1, brings):
            raise MemoryError("no pages")
    return State(case, model, cache, runner, requests)


def run(state):
    """One step of all requests (and the further steps of those that come in), as the engine runs it: entries, the runner,
    and the bookkeeping of what entered.  A request that was there before the pass is left where it stood, so that the same
    pass can be run again."""
    from paged_llm_rs_amd.engine.batch import StepEntry
    from paged_llm_rs_amd.engine.step import commit_step

    manager = state.cache.manager
    entries, entered = [], []
    for i, (ids, inside, brings) in enumerate(state.requests):
        if inside == 0:
            slot = manager.add_sequence(i + 1)
            if not manager.reserve(i + 1, len(ids)):
                raise MemoryError("no pages")
            entered.append(i)
        else:
            slot = manager.state_slot(i + 1)
        entries.append(StepEntry(i + 1, ids[inside:inside + brings], inside, [brings - 1], state_slot=slot,
                                 fresh_state=inside == 0 and slot >= 0))
    logits = [state.runner.run(entries).logits]
    steps = state.case["steps"]
    if steps:
        commit_step(state.cache, entries)
        for k in range(steps):
            entries = [StepEntry(i + 1, [ids[inside + brings + k]], inside + brings + k, [0], state_slot=manager.state_slot(i + 1))
                       for i, (ids, inside, brings) in enumerate(state.requests)]
            # (a decoding step's logits are the runner's own buffer: what is to outlast the next step is copied)
            logits.append(state.runner.run(entries).logits.clone())
            commit_step(state.cache, entries)
    for i in entered:
        manager.free_sequence(i + 1)
    if entered:
        return {"logits": logits}       # (the pages go back with their requests)
    return {"logits": logits, "pages": list(state.cache.layer_pools(state.last_layer))}


# -- what a pass cannot do without ----------------------------------------------------------------------------------------------

def _sizes(case):
    """(rows multiplied, requests with logits, keys read by a step's requests, query-key pairs) of a pass, from the mean
    lengths of its requests."""
    def mean(count):        # of what ``_lengths`` gives, as a share of the longest
        return (1 + 0.75 * (count - 1)) / max(count, 1)

    d, ctx = case["decodes"], case["context"] * mean(case["decodes"])
    rows, wanted = d + case["prompts"] * case["tokens"] * mean(case["prompts"]), d + case["prompts"]
    each = (rows - d) / max(case["prompts"], 1)
    keys = d * ctx + case["prompts"] * (case["behind"] + each)
    pairs = d * ctx + case["prompts"] * each * (case["behind"] + each / 2)
    return rows, wanted, keys, pairs


def work(case):
    config = CONFIGS[case["model"]]
    size = 2 if case["dtype"] == "bf16" else 4
    rows, wanted, keys, pairs = _sizes(case)
    steps = case["steps"]
    shapes = _declared(config)
    head = VOCAB * (config.get("hidden_size") or config["width"])
    matrices = expert = 0
    for name, shape, how in shapes:
        if how == "matrix" and len(shape) == 2 and name not in ("model.embed_tokens.weight", "embed", "head", "lm_head.weight"):
            if ".mlp.e" in name:
                expert += shape[0] * shape[1]
            else:
                matrices += shape[0] * shape[1]
    flops = 2.0 * rows * (matrices + expert / 4) + 2.0 * wanted * head
    flops += steps * 2.0 * case["prompts"] * (matrices + expert / 4 + head)
    if "num_hidden_layers" in config:
        layers, heads, d = config["num_hidden_layers"], config["num_attention_heads"], config["head_dim"]
        kv = 2 * layers * config["num_key_value_heads"] * d * size
        flops += 4.0 * layers * heads * d * pairs
        reads = kv * (keys - (rows - case["decodes"] if case["prompts"] else 0)) + kv * rows
    else:
        # a state of 128 x 1,024 values a layer, twice the pass of its chunks, or keys and values of 8 heads of 128
        layers = len(config["layers"])
        flops += rows * layers * 4.0 * 128 * 1024
        reads = layers * (2 * 4 * 128 * 1024 * case["prompts"] * (1 + steps) + 2 * 1024 * size * rows / 3)
    weights = (matrices + expert + head) * size
    return {"bytes": weights * (1 + steps) + reads + 4.0 * VOCAB * wanted * (1 + steps), "flops": flops}


def tolerance(case):
    # about four times how far the results of the present kernels are from 64-bit arithmetic: 32-bit sums through 28 layers
    # (2.4e-6); bfloat16, which rounds every product's result for the next to multiply (0.6B 0.008, 8B and 32B 0.017, where the
    # weights of 0.02 weigh more in a wide product; Mukenex 0.006; Papivik 0.006 to 0.022, whose read-outs are normalised however
    # small they are: a sum near zero shows its rounding in full)
    if case["dtype"] == "f32":
        return {"rel": 1e-5}
    return {"rel": {"qwen3-0.6b": 3e-2, "papivik": 8e-2, "mukenex": 2.5e-2}.get(case["model"], 6e-2)}


# -- the same in 64-bit arithmetic ------------------------------------------------------------------------------------------------

F = torch.float64


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _silu(x):
    return x * torch.sigmoid(x)


def _softmax_attention(q, k, v, scale, first, sink=None):
    """q [T, H, D], k [T, G, D], v [T, G, V] -> [T, H, V]; query i sees keys first[i]..i."""
    T, H, _ = q.shape
    out = torch.empty(T, H, v.shape[-1], dtype=q.dtype, device=q.device)
    each = H // k.shape[1]
    at = torch.arange(T, device=q.device)
    for h in range(H):
        for a in range(0, T, 2048):
            b = min(a + 2048, T)
            s = (q[a:b, h] @ k[:b, h // each].T) * scale
            hidden = (at[None, :b] > at[a:b, None]) | (at[None, :b] < first[a:b, None])
            s.masked_fill_(hidden, -math.inf)
            top = s.amax(-1, keepdim=True)
            if sink is not None:
                top = torch.clamp(top, min=float(sink[h]))
            e = torch.exp(s - top)
            total = e.sum(-1, keepdim=True)
            if sink is not None:
                total = total + torch.exp(sink[h] - top)
            out[a:b, h] = (e @ v[:b, h // each]) / total
    return out


def _turn(x, dims, base, neighbours=False):
    """x [T, ..., n]: the first ``dims`` values turn by position * base^(-2i/dims), value i with i + dims/2 or 2i with 2i + 1."""
    half = dims // 2
    freq = base ** (-2.0 * torch.arange(half, dtype=F, device=x.device) / dims)
    angle = torch.arange(x.shape[0], dtype=F, device=x.device)[:, None] * freq
    while angle.dim() < x.dim():
        angle = angle.unsqueeze(1)
    cos, sin = angle.cos(), angle.sin()
    if neighbours:
        a, b = x[..., 0:dims:2], x[..., 1:dims:2]
        return torch.cat([torch.stack([a * cos - b * sin, b * cos + a * sin], -1).flatten(-2), x[..., dims:]], -1)
    a, b = x[..., :half], x[..., half:dims]
    return torch.cat([a * cos - b * sin, b * cos + a * sin, x[..., dims:]], -1)


def _qwen3_rows(config, w, ids):
    h, d, eps, theta = config["hidden_size"], config["head_dim"], config["rms_norm_eps"], config["rope_theta"]
    nq, nkv, T = config["num_attention_heads"], config["num_key_value_heads"], len(ids)
    x = w("model.embed_tokens.weight", rows=ids)
    first = torch.zeros(T, dtype=torch.long, device=DEVICE)
    for n in range(config["num_hidden_layers"]):
        p = f"model.layers.{n}."
        y = _rms(x, eps) * w(p + "input_layernorm.weight")
        q = (y @ w(p + "self_attn.q_proj.weight").T).view(T, nq, d)
        k = (y @ w(p + "self_attn.k_proj.weight").T).view(T, nkv, d)
        v = (y @ w(p + "self_attn.v_proj.weight").T).view(T, nkv, d)
        q = _turn(_rms(q, eps) * w(p + "self_attn.q_norm.weight"), d, theta)
        k = _turn(_rms(k, eps) * w(p + "self_attn.k_norm.weight"), d, theta)
        x = x + _softmax_attention(q, k, v, d ** -0.5, first).reshape(T, nq * d) @ w(p + "self_attn.o_proj.weight").T
        y = _rms(x, eps) * w(p + "post_attention_layernorm.weight")
        y = _silu(y @ w(p + "mlp.gate_proj.weight").T) * (y @ w(p + "mlp.up_proj.weight").T)
        x = x + y @ w(p + "mlp.down_proj.weight").T
    head = "model.embed_tokens.weight" if config["tie_word_embeddings"] else "lm_head.weight"
    return _rms(x, eps) * w("model.norm.weight"), lambda rows: rows @ w(head).T


def _lightning(u, w, x, m, eps):
    T, H, D, V = u.shape[0], m["heads"], m["dim"], m["vdim"]
    q, k, v = ((_silu(u @ w(x + n).T)).view(T, H, -1) for n in "qkv")
    decay = torch.tensor(m["decay"], dtype=F, device=DEVICE)[:, None, None]
    S = torch.zeros(H, D, V, dtype=F, device=DEVICE)
    o = torch.empty(T, H, 1, V, dtype=F, device=DEVICE)
    for t in range(T):
        S.mul_(decay).baddbmm_(k[t, :, :, None], v[t, :, None, :])
        torch.bmm(q[t, :, None, :], S, out=o[t])
    o = _rms(o.view(T, H * V), eps) * w(x + "norm") * torch.sigmoid(u @ w(x + "g").T)
    return o @ w(x + "o").T


def _mlstm(u, w, x, m, eps):
    T, H, D, V, cap = u.shape[0], m["heads"], m["dim"], m["vdim"], m["gate_cap"]
    q = (u @ w(x + "q").T).view(T, H, D) * D ** -0.5
    k, v = (u @ w(x + "k").T).view(T, H, D), (u @ w(x + "v").T).view(T, H, V)
    i = cap * torch.tanh((u @ w(x + "i").T + w(x + "i.b")) / cap)
    f = torch.nn.functional.logsigmoid(cap * torch.tanh((u @ w(x + "f").T + w(x + "f.b")) / cap))
    # the running maximum, which starts at 0, and from it every step's factors
    b = torch.cumsum(f, 0)
    top = b + torch.clamp(torch.cummax(i - b, 0).values, min=0.0)
    before = torch.cat([torch.zeros(1, H, dtype=F, device=DEVICE), top[:-1]])
    keep, add = torch.exp(f + before - top), torch.exp(i - top)
    S = torch.zeros(H, D, V + 1, dtype=F, device=DEVICE)       # (the normaliser is a column of its own)
    k = k * add[:, :, None]
    v = torch.cat([v, torch.ones(T, H, 1, dtype=F, device=DEVICE)], -1)
    o = torch.empty(T, H, 1, V + 1, dtype=F, device=DEVICE)
    for t in range(T):
        S.mul_(keep[t, :, None, None]).baddbmm_(k[t, :, :, None], v[t, :, None, :])
        torch.bmm(q[t, :, None, :], S, out=o[t])
    o = o[:, :, 0]
    below = torch.maximum(o[..., V].abs(), torch.exp(-top)) + 1e-6
    o = _rms(o[..., :V] / below[..., None], eps).reshape(T, H * V) * w(x + "norm") * torch.sigmoid(u @ w(x + "g").T)
    return o @ w(x + "o").T


def _short_conv(u, taps):
    T, n = u.shape[0], taps.shape[1]
    padded = torch.cat([torch.zeros(n - 1, u.shape[1], dtype=F, device=DEVICE), u])
    return sum(padded[j:j + T] * taps[:, j] for j in range(n))


def _delta(u, w, x, m, eps):
    T, H, G, D, V = u.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k, v = (_silu(_short_conv(u @ w(x + n).T, w(x + n + ".conv"))) for n in "qkv")
    q, k, v = q.view(T, G, D), k.view(T, G, D), v.view(T, H, V)
    q = (q / torch.sqrt((q * q).sum(-1, keepdim=True) + 1e-6) * D ** -0.5).repeat_interleave(H // G, 1)
    k = (k / torch.sqrt((k * k).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
    beta = torch.sigmoid(u @ w(x + "b").T)
    decay = torch.exp(-torch.exp(w(x + "A_log")) * torch.nn.functional.softplus(u @ w(x + "a").T + w(x + "dt_bias")))
    S = torch.zeros(H, D, V, dtype=F, device=DEVICE)
    o = torch.empty(T, H, 1, V, dtype=F, device=DEVICE)
    for t in range(T):
        S.mul_(decay[t, :, None, None])
        S.baddbmm_(k[t, :, :, None], beta[t, :, None, None] * (v[t, :, None, :] - torch.bmm(k[t, :, None, :], S)))
        torch.bmm(q[t, :, None, :], S, out=o[t])
    o = (_rms(o[:, :, 0], eps) * w(x + "norm")).reshape(T, H * V) * _silu(u @ w(x + "g").T)
    return o @ w(x + "o").T


def _conv_attention(u, w, x, m, eps):
    T, H, G, D, V = u.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k, v = (_short_conv(u @ w(x + n).T, w(x + n + ".conv")) for n in "qkv")
    q = _turn(_rms(q.view(T, H, D), eps) * w(x + "q.norm"), m["rot"]["dims"], m["rot"]["base"])
    k = _turn(_rms(k.view(T, G, D), eps) * w(x + "k.norm"), m["rot"]["dims"], m["rot"]["base"])
    first = torch.zeros(T, dtype=torch.long, device=DEVICE)
    return _softmax_attention(q, k, v.view(T, G, V), m["scale"], first).reshape(T, H * V) @ w(x + "o").T


def _latent(u, w, x, m, eps):
    T, H, D, rot, R = u.shape[0], m["heads"], m["dim"], m["rot_dim"], m["kv_rank"]
    both = u @ w(x + "dkv").T
    c = _rms(both[:, :R], eps) * w(x + "dkv.norm")
    k_rot = _turn(both[:, R:], m["rot"]["dims"], m["rot"]["base"], neighbours=True)
    q = (u @ w(x + "q").T).view(T, H, D + rot)
    q = torch.cat([q[..., :D], _turn(q[..., D:], m["rot"]["dims"], m["rot"]["base"], neighbours=True)], -1)
    k = torch.cat([(c @ w(x + "uk").T).view(T, H, D), k_rot[:, None].expand(T, H, rot)], -1)
    first = torch.clamp(torch.arange(T, device=DEVICE) - m["mask"]["size"] + 1, min=0)
    o = _softmax_attention(q, k, (c @ w(x + "uv").T).view(T, H, -1), m["scale"], first, w(x + "sink")).reshape(T, -1)
    return (o * torch.sigmoid(u @ w(x + "g").T)) @ w(x + "o").T


def _block_attention(u, w, x, m, eps):
    T, H, G, D, V = u.shape[0], m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k, v = (u @ w(x + n).T + w(x + n + ".b") for n in "qkv")
    q = _rms(q.view(T, H, D), eps) * w(x + "q.norm")
    k = _rms(k.view(T, G, D), eps) * w(x + "k.norm")
    first = torch.arange(T, device=DEVICE) // m["mask"]["size"] * m["mask"]["size"]
    return _softmax_attention(q, k, v.view(T, G, V), m["scale"], first).reshape(T, H * V) @ w(x + "o").T


def _experts(u, w, f, ids):
    chosen = w(f + "table", rows=ids)
    out = torch.zeros_like(u)
    for e in range(8):
        at, _ = torch.where(chosen == e)
        y = u[at]
        y = _silu(y @ w(f"{f}e{e}.gate").T) * (y @ w(f"{f}e{e}.up").T)
        out.index_add_(0, at, y @ w(f"{f}e{e}.down").T / chosen.shape[1])
    return out


def _design_rows(config, w, ids):
    eps, copies = config["norm"]["eps"], config.get("streams")
    gelu = torch.nn.functional.gelu

    def mixer(n, layer, u):
        x, m = f"l{n}.mix.", layer["mixer"]
        if layer["type"] == "parallel":
            return (m["left_scale"] * _conv_attention(u, w, x + "left.", m["left"], eps)
                    + m["right_scale"] * _delta(u, w, x + "right.", m["right"], eps))
        kinds = {"lightning": _lightning, "mlstm": _mlstm, "latent_attention": _latent, "attention": _block_attention}
        return kinds[layer["type"]](u, w, x, m, eps)

    def feed_forward(n, layer, u):
        f = f"l{n}.mlp."
        if layer["mlp"]["kind"] == "moe":
            return _experts(u, w, f, ids)
        return gelu(u @ w(f + "up").T, approximate="none" if copies else "tanh") @ w(f + "down").T

    x = w("embed", rows=ids)
    if copies:
        x = x.expand(copies, *x.shape).clone()
    for n, layer in enumerate(config["layers"]):
        for norm, hc, part in (("norm1", "hc1.", mixer), ("norm2", "hc2.", feed_forward)):
            gain, p = w(f"l{n}.{norm}"), f"l{n}.{hc}"
            if copies:
                u = torch.einsum("s,stw->tw", w(p + "in"), x)
                y = part(n, layer, _rms(u, eps) * (1.0 + gain))
                x = torch.einsum("sr,stw->rtw", w(p + "mix"), x) + w(p + "out")[:, None, None] * y
            else:
                x = x + _rms(part(n, layer, x), eps) * gain
    if copies:
        cap = config["logit_softcap"]
        return _rms(x.sum(0), eps) * (1.0 + w("final.norm")), lambda rows: cap * torch.tanh(rows @ w("head").T / cap)
    return _rms(x, eps) * w("final.norm"), lambda rows: rows @ w("head").T


EXACT_MOST = 2.5e14     # operations in 64 bits that take some seconds


def exact(case, seed):
    config = CONFIGS[case["model"]]
    requests = _requests(case, seed)
    shapes = {name: shape for name, shape, _ in _declared(config)}
    inner = sum(s[0] * s[1] for n, s in shapes.items() if len(s) == 2 and s[0] != VOCAB)
    cost = sum(2.0 * len(ids) * inner for ids, _, _ in requests)
    if "num_hidden_layers" in config:
        cost += sum(2.0 * len(ids) ** 2 * config["num_attention_heads"] * 128 * config["num_hidden_layers"] * 2 for ids, _, _ in requests)
    if cost > EXACT_MOST:
        return None
    stored = _weights(case["model"], DTYPES[case["dtype"]])

    def w(name, rows=None):
        t = stored[name] if rows is None else stored[name][torch.as_tensor(rows, device=DEVICE)]
        return t.to(F) if t.is_floating_point() else t

    rows_of = _qwen3_rows if "num_hidden_layers" in config else _design_rows
    steps = [[] for _ in range(1 + case["steps"])]
    with torch.no_grad():
        for ids, inside, brings in requests:
            rows, head = rows_of(config, w, ids)
            for k in range(len(steps)):
                steps[k].append(rows[inside + brings - 1 + k])
        logits = [head(torch.stack(rows)) for rows in steps]
    return {"logits": logits, "pages": None} if all(inside for _, inside, _ in requests) else {"logits": logits}
