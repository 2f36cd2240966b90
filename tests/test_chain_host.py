"""What a step asks on the host before its layers run as chains of products."""

from __future__ import annotations

import pytest

from conftest import TINY_A


@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
def test_layers_that_no_chain_takes_are_asked_their_sizes_only(tmp_path, monkeypatch, dtype):
    """A launch a product is what wide layers have anyway, and an eager step pays for every question about every layer (64 layers: 0.5 to 0.8 ms a step
    when the tensors of each were looked at, 0.12 now).  Sizes are asked of the kernel once for all layers that share them."""
    from paged_llm_rs_amd import kernels, write_random_model
    from paged_llm_rs_amd.parts.model import load_model

    cfg = dict(TINY_A, hidden_size=1088, intermediate_size=64, num_attention_heads=2, num_key_value_heads=2, head_dim=16, num_hidden_layers=5)
    folder = write_random_model(tmp_path / "wide", cfg, seed=1, std=0.02, gain_std=0.1, dtype=dtype)
    model = load_model(folder, dtype, "cpu", strips=False)[1]
    asked = []
    applies = kernels.chain_applies
    monkeypatch.setattr(kernels, "in_pieces", lambda *tensors: pytest.fail("a wide layer's tensors were looked at"))
    monkeypatch.setattr(kernels, "chain_applies", lambda *args, **how: asked.append(args) or applies(*args, **how))
    assert model._chains(4, None, None) == {} and len(asked) == 1
    assert model._chains(65, None, None) == {} and len(asked) == 1


def test_layers_with_a_product_or_norm_of_a_class_of_its_own_are_no_chain(tmp_path):
    """A chain reads weights and gains and never asks the objects that hold them: a mixer that puts another product behind its attention (one that adds a
    low-rank part, say, or that keeps its weight in another form) has to go on getting that product's result."""
    from paged_llm_rs_amd import write_random_model
    from paged_llm_rs_amd.parts.linear import Linear
    from paged_llm_rs_amd.parts.model import load_model
    from paged_llm_rs_amd.parts.norm import RmsNorm

    class Doubled(Linear):
        def forward(self, x, *args, **kwargs):
            return super().forward(x, *args, **kwargs) * 2

    class OfAnotherForm:
        bias = None

        def forward(self, x, **how):
            return x

    class Halved(RmsNorm):
        def apply(self, *args, **kwargs):
            return super().apply(*args, **kwargs) / 2

    cfg = dict(TINY_A, hidden_size=512, intermediate_size=128, num_attention_heads=2, num_key_value_heads=2, head_dim=64, num_hidden_layers=7)
    folder = write_random_model(tmp_path / "model", cfg, seed=1, std=0.02, gain_std=0.1, dtype="float32")
    model = load_model(folder, "float32", "cpu")[1]
    assert list(model._chain_places(8)) == [0, 1, 2, 3, 4, 5, 6]
    blocks = model.blocks
    blocks[1].mixer.o_proj.__class__ = Doubled
    blocks[2].mixer.qkv_proj = OfAnotherForm()
    blocks[3].feed_forward.down_proj = OfAnotherForm()
    blocks[4].feed_forward.gate_up_proj.__class__ = Doubled
    blocks[5].norm2.__class__ = Halved
    assert list(model._chain_places(8)) == [0, 6]
