"""Models whose layers run as chains of products beside layers that do not: a layer with an output bias and a block of another class between them, a layer
that borrows pages, one that runs again behind the embedding.  Against the plain arithmetic in 64 bits, and bit for bit against the same model with every
product a launch of its own."""

from __future__ import annotations

import collections
import math

import pytest
import torch

import plain_qwen3 as plain
import replay_util as ru

pytestmark = pytest.mark.gpu

# (layer, the layer whose keys and values it reads or None, again behind the embedding): 2 has an output bias, 5 a block of its own class.
RUNS = ((0, None, False), (1, None, False), (2, None, False), (3, None, False), (4, 3, False), (0, None, True), (1, None, False), (5, None, False))


class ChainedConfig:
    def __init__(self, d):
        self.d = d

    @classmethod
    def from_dict(cls, d):
        return cls(dict(d))

    def to_dict(self):
        return dict(self.d)

    def model_spec(self):
        from paged_llm_rs_amd.config import (AttentionSpec, GatedMlpSpec, LayerSpec, ModelSpec, NormSpec, PositionSpec, ScheduleEntry)
        d = self.d
        norm = NormSpec("rms_norm", d["rms_norm_eps"])
        ffn = GatedMlpSpec("gated_mlp", d["intermediate_size"], "silu")
        position = PositionSpec("rotary_half", d["head_dim"], d["rope_theta"], d["max_position_embeddings"])
        layers = tuple(LayerSpec("pre_norm_of_its_own" if i == 5 else "pre_norm",
                                 AttentionSpec("paged_attention", d["num_attention_heads"], d["num_key_value_heads"], d["head_dim"], norm, position, None,
                                               None, out_bias=i == 2), ffn, norm, f"model.layers.{i}") for i in range(6))
        schedule = tuple(ScheduleEntry(layer, cache_from=source, cache_key=10 + at if at in (5, 6) else None, add_embedding=again)
                         for at, (layer, source, again) in enumerate(RUNS))
        return ModelSpec(d["hidden_size"], d["vocab_size"], layers, schedule, norm, d["tie_word_embeddings"], d["max_position_embeddings"])


def _config(dtype):
    # (heads of 96, two a key head: single tokens' attention is a stage of the chain; 32-bit chains take streams from 512 on)
    return {"architectures": ["ChainedToyForCausalLM"], "model_type": "chained_toy", "hidden_size": 64 if dtype == "bfloat16" else 1024,
            "intermediate_size": 96 if dtype == "bfloat16" else 192, "num_attention_heads": 4, "num_key_value_heads": 2,
            "head_dim": 96 if dtype == "bfloat16" else 32, "rms_norm_eps": 1e-5, "rope_theta": 1e4, "vocab_size": 89, "max_position_embeddings": 256,
            "tie_word_embeddings": True}


def chained_plain(cfg, weights, tokens):
    w = {k: v.double() for k, v in weights.items()}
    n, eps = len(tokens), cfg["rms_norm_eps"]
    nq, nkv, d = cfg["num_attention_heads"], cfg["num_key_value_heads"], cfg["head_dim"]
    positions = torch.arange(n)
    first = w["model.embed_tokens.weight"][torch.tensor(tokens)]
    x, held = first.clone(), {}

    def heads(h, p, which, count):
        y = (h @ w[f"{p}.self_attn.{which}_proj.weight"].T).reshape(n, count, d)
        return y if which == "v" else plain.apply_rope(plain.rms_norm(y, w[f"{p}.self_attn.{which}_norm.weight"], eps), positions, cfg["rope_theta"])

    for layer, source, again in RUNS:
        p = f"model.layers.{layer}"
        if again:
            x = x + first
        h = plain.rms_norm(x, w[f"{p}.input_layernorm.weight"], eps)
        if source is None:
            held[layer] = heads(h, p, "k", nkv), heads(h, p, "v", nkv)
        k, v = held[layer if source is None else source]
        out = plain.attention_core(heads(h, p, "q", nq), plain.repeat_kv(k, nq // nkv), plain.repeat_kv(v, nq // nkv), 1.0 / math.sqrt(d))
        x = x + out.reshape(n, nq * d) @ w[f"{p}.self_attn.o_proj.weight"].T + w.get(f"{p}.self_attn.o_proj.bias", 0.0)
        x = x + plain.swiglu_mlp(plain.rms_norm(x, w[f"{p}.post_attention_layernorm.weight"], eps), w, f"{p}.mlp")
    return plain.rms_norm(x, w["model.norm.weight"], eps) @ w["model.embed_tokens.weight"].T


@pytest.fixture(scope="module")
def toys(tmp_path_factory):
    """(configuration, folder) by type, made on first use."""
    from paged_llm_rs_amd import register_architecture, write_random_model
    from paged_llm_rs_amd.parts.block import PreNormBlock
    from paged_llm_rs_amd.parts.registry import BLOCKS, register_block

    class OfItsOwn(PreNormBlock):
        def forward(self, resid, delta, ctx):
            assert ctx.chain is None
            return super().forward(resid, delta, ctx)

    if "pre_norm_of_its_own" not in BLOCKS:
        register_block("pre_norm_of_its_own", OfItsOwn)
    register_architecture("ChainedToyForCausalLM", ChainedConfig, model_type="chained_toy")
    made: dict = {}

    def get(dtype):
        if dtype not in made:
            cfg = _config(dtype)
            made[dtype] = cfg, write_random_model(tmp_path_factory.mktemp("chained") / dtype, cfg, seed=31,
                                                  std=0.15 if dtype == "bfloat16" else 0.05, gain_std=0.2, dtype=dtype)
        return made[dtype]

    return get


def _watch(monkeypatch):
    """Counts of the chains that are launched (or captured): with a stream of the chain before, with a following layer, with its attention; and of the
    products that hand a norm forward and that take one."""
    from paged_llm_rs_amd import kernels

    seen = collections.Counter()
    launch = kernels.gemm_chain

    def watched(stream, laid, rows, room, w_out, w_gated, w_down, gain, eps, activation, following=None, looks=None, attention=None):
        seen.update(chains=1, laid=int(laid), following=int(following is not None), attends=int(attention is not None),
                    borrows=int(attention is not None and not attention.prepare.write_kv))
        return launch(stream, laid, rows, room, w_out, w_gated, w_down, gain, eps, activation, following, looks, attention)

    product = kernels.gemm_skinny

    def watched_product(*args, hand=None, handed=None, **how):
        out = product(*args, hand=hand, handed=handed, **how)
        seen.update(hands=int(hand is not None and hand.filled), takes=int(handed is not None))
        return out

    monkeypatch.setattr(kernels, "gemm_chain", watched)
    monkeypatch.setattr(kernels, "gemm_skinny", watched_product)
    return seen


def _replay(folder, dtype, steps, prompts, live, **how):
    from paged_llm_rs_amd.engine.replay import Replayer

    return ru.collect(Replayer(folder, dtype, max_tokens=ru.pool_tokens(prompts, live), block_size=8, max_live=4, **how), steps)


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_chains_beside_layers_that_are_none(toys, dtype, monkeypatch):
    """Layer 0's chain goes on to 1, whose chain ends before 2, which has none and hands its last norm forward to 3; 3 goes on to 4, whose keys are 3's; 4
    ends before the layer that starts again, and the one behind that before 5.  Whole, decoded, in portions and mixed."""
    from safetensors.torch import load_file

    from paged_llm_rs_amd import kernels

    cfg, folder = toys(dtype)
    weights = load_file(str(folder / "model.safetensors"))
    prompts = ru.make_prompts(cfg["vocab_size"], [28, 13, 100, 32], seed=9)
    want = {name: chained_plain(cfg, weights, toks) for name, toks in prompts.items()}
    tolerance = 1e-5 if dtype == "float32" else 3e-2
    # (the mixed schedule alone has steps of 33 to 64 rows, whose products apart may be other kernels that round a sum another way)
    for steps, live, same in ((ru.whole(prompts), 1, True), (ru.tail_decoded(prompts, 20), 1, True),
                              (ru.portions(prompts, (2, 7, 3, 16, 5, 2, 30, 4, 9)), 1, True), (ru.mixed(prompts, seed=5, max_live=3), 3, False)):
        with monkeypatch.context() as m:
            seen = _watch(m)
            got = _replay(folder, dtype, steps, prompts, live)
            assert seen["chains"] and seen["chains"] % 6 == 0, "layers 0, 1, 3, 4 and the two that run again"
            assert seen["laid"] == seen["following"] == seen["chains"] // 2
            assert seen["hands"] == seen["takes"], "a norm that is handed to a chained layer is taken there"
            assert seen["attends"] == 3 * seen["borrows"], "of three attentions behind chains one borrows its pages"
            assert (seen["attends"] > 0) == (dtype == "bfloat16" and any(len(e["tokens"]) == 1 for step in steps for e in step["entries"]))
        worst, where = ru.worst_error(got, want)
        assert worst <= tolerance, f"{worst:.3e} at {where}"
        with monkeypatch.context() as m:
            m.setattr(kernels, "chain_applies", lambda *args, **kwargs: False)
            seen = _watch(m)
            apart = _replay(folder, dtype, steps, prompts, live)
            assert not seen["chains"] and (dtype == "float32" or seen["takes"])
        assert got.keys() == apart.keys()
        other = [key for key, row in got.items() if not (row == apart[key]).all()]
        assert not same or not other, f"other bits at {other}"


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_a_model_without_chains_gives_the_same_bits(toys, dtype, monkeypatch):
    """Told not to, a model runs no chain, eagerly or captured; nor does one in bfloat16 that keeps no strips."""
    from paged_llm_rs_amd.engine.replay import Replayer

    cfg, folder = toys(dtype)
    prompts = ru.make_prompts(cfg["vocab_size"], [30], seed=2)
    steps = ru.tail_decoded(prompts, 12)
    want = _replay(folder, dtype, steps, prompts, 1)
    with monkeypatch.context() as m:
        seen = _watch(m)
        r = Replayer(folder, dtype, max_tokens=64, block_size=8, max_live=2)
        r.model.chains = False
        got = ru.collect(r, steps)
        assert not seen["chains"] and r.model.step_room_bytes(16) == 0
        assert got.keys() == want.keys() and all((row == want[key]).all() for key, row in got.items())
        if dtype == "bfloat16":
            _replay(folder, dtype, steps, prompts, 1, strips=False)
            assert not seen["chains"]
    assert Replayer(folder, dtype, max_tokens=64, block_size=8, max_live=2).model.step_room_bytes(16) > 0


@pytest.mark.parametrize("hidden,inter,chained", [(1024, 192, True), (1024, 3072, True), (1024, 2560, False), (960, 2048, True), (512, 192, False)])
def test_which_32_bit_steps_of_one_token_are_chains(tmp_path, monkeypatch, hidden, inter, chained):
    """Of a single row a chain is not the faster way at every size that it takes (``kernels.chain_wins``); of eight it is.  Same bits."""
    from paged_llm_rs_amd import kernels, write_random_model
    from conftest import TINY_A

    cfg = dict(TINY_A, hidden_size=hidden, intermediate_size=inter, num_attention_heads=4, num_key_value_heads=2, head_dim=16, num_hidden_layers=2)
    folder = write_random_model(tmp_path / "model", cfg, seed=5, std=0.02, gain_std=0.1, dtype="float32")
    prompts = ru.make_prompts(cfg["vocab_size"], [8], seed=3)
    for steps, expected in ((ru.tail_decoded(prompts, 7), chained), (ru.whole(prompts), True)):
        with monkeypatch.context() as m:
            seen = _watch(m)
            got = _replay(folder, "float32", steps, prompts, 1)
            assert bool(seen["chains"]) == expected
        with monkeypatch.context() as m:
            m.setattr(kernels, "chain_applies", lambda *args, **kwargs: False)
            apart = _replay(folder, "float32", steps, prompts, 1)
        assert all((row == apart[key]).all() for key, row in got.items())
