"""Which kernel a call goes to, as far as sizes alone decide it: the rules, asked as the engine asks them (no GPU; a chip of 256 compute units)."""

from types import SimpleNamespace

import pytest
import torch

from paged_llm_rs_amd import kernels
from paged_llm_rs_amd.engine.batch import near_context, token_bucket
from paged_llm_rs_amd.parts.block import PreNormBlock
from paged_llm_rs_amd.parts.linear import Linear
from paged_llm_rs_amd.parts.mlp import GatedMlp


@pytest.fixture(autouse=True)
def a_whole_chip(monkeypatch):
    monkeypatch.setattr(kernels, "_compute_units", 256)


# (tokens, tokens before them) of the requests; query heads; head size; the shares that measured within a twelfth of the best
SEVERAL_PROMPTS = [
    ([(600, 0)] * 3, 16, 256, (1,)), ([(600, 0), (500, 0), (400, 0)], 16, 256, (1,)), ([(600, 0)] * 3, 4, 128, (1, 2)), ([(600, 0)] * 3, 8, 64, (1,)),
    ([(150, 0)] * 8, 16, 256, (1,)), ([(150, 0)] * 8, 4, 128, (1,)), ([(100, 0)] * 16, 16, 256, (1,)), ([(100, 0)] * 16, 8, 64, (1,)),
    ([(250, 0)] * 4, 8, 256, (1,)), ([(250, 0)] * 6, 4, 128, (1,)), ([(40, 0)] * 12, 8, 256, (1,)), ([(64, 400)] * 16, 8, 64, (1,)),
    ([(300, 600)] * 2, 4, 128, (2, 3, 4)), ([(300, 600)] * 2, 16, 256, (2,)), ([(300, 600)] * 2, 8, 256, (3, 4)), ([(300, 600)] * 2, 32, 128, (1,)),
    ([(64, 1900)] * 4, 8, 256, (8,)), ([(200, 3000)] * 3, 16, 256, (2,)), ([(1500, 0)] * 2, 16, 256, (1,)), ([(1500, 0)] * 2, 8, 256, (2,)),
    ([(512, 1024)] + [(1, 900)] * 63, 8, 256, (1, 2, 3)),
]


@pytest.mark.parametrize("requests,nq,d,good", SEVERAL_PROMPTS)
def test_the_shares_of_several_prompts_keys(requests, nq, d, good):
    """A padded step reports all of its rows as the longest portion, which no request's context need be as long as: no shares of keys that no request has, and
    several where requests stand behind many others."""
    rows = token_bucket(sum(t for t, _ in requests))
    near = near_context(max(t + b for t, b in requests))
    assert kernels.prefill_splits(len(requests), rows, nq, d, near, rows, 0) in good
    # (never a share of less than four tiles of keys, as many requests as there may be)
    assert kernels.prefill_splits(len(requests), rows, nq, d, near, rows, 0) * 4 * 64 <= max(near, 256)


@pytest.mark.parametrize("columns", [32768, 50304, 151936, 262144])
def test_a_vocabulary_of_few_rows_goes_by_no_width(columns):
    """The product of many rows takes a vocabulary by the rows and by how the weights lie, whatever the width."""
    for width in (768, 896, 960, 1024, 1088, 1536, 2048, 4096, 5120):
        if columns * width < 2 ** 31:
            assert [kernels.many_vocabulary_wins(n, columns, width, True) for n in (1, 8, 16, 17, 64, 128, 129, 200)] == [False] * 3 + [True] * 3 + [False] * 2
            assert [kernels.many_vocabulary_wins(n, columns, width, False) for n in (1, 16, 17, 64, 65, 128)] == [False, False, True, True, False, False]
    assert not kernels.many_vocabulary_wins(32, columns, 1000, True) and not kernels.many_vocabulary_wins(32, 32752, 1024, True)


# (columns, width): {rows: whether the product of many rows measured at most as long as the library's, out of strips and in rows}, a twenty-fifth either way let pass
PLAIN = {
    (4096, 1024): {65: "yy", 576: "yy", 1024: "yy", 2048: "nn"}, (1024, 1024): {65: "yy", 4096: "yy", 5120: "yn", 8192: "nn"}, (3072, 768): {1024: "yy", 1408: "yn"},
    (1024, 1536): {832: "nn", 1024: "nn", 1216: "yy", 1984: "yy"}, (2048, 1536): {512: "nn", 576: "yy", 1024: "yy"}, (1024, 1152): {321: "nn", 1089: "yy"},
    (2048, 2048): {576: "nn", 704: "nn", 832: "yy", 1024: "yy"}, (3072, 2048): {384: "nn", 576: "yy"}, (4096, 2048): {384: "nn", 448: "yy"},
    (1024, 3072): {1216: "nn", 1408: "nn", 1792: "yn"}, (3072, 3072): {448: "nn", 512: "nn", 576: "yn"}, (4096, 2560): {384: "nn", 448: "yy"}, (4096, 3072): {384: "nn", 512: "yn"},
    (5120, 2048): {65: "nn", 256: "yy", 384: "yy"}, (8192, 3072): {65: "nn", 192: "yn"}, (6144, 3072): {256: "yn"}, (1024, 4096): {1024: "nn", 2048: "nn"},
}


@pytest.mark.parametrize("columns,width", list(PLAIN))
def test_the_plain_product_of_many_rows_is_taken_where_it_measured_faster(columns, width):
    for rows, wanted in PLAIN[columns, width].items():
        assert [kernels.many_store_wins(rows, columns, width, strips) for strips in (True, False)] == [w == "y" for w in wanted], rows


GATED = {
    (3072, 1024): {65: "yy", 2048: "yy", 4096: "yy", 8192: "yn"}, (8192, 1024): {1024: "yy", 1536: "yy", 2048: "yn", 3072: "yn", 4096: "nn"},
    (4096, 2048): {65: "yy", 1024: "yy", 1536: "yn", 2048: "nn"}, (6144, 2048): {200: "yy", 1024: "yy"}, (9728, 2560): {128: "yy", 160: "yy", 192: "yy", 384: "yy"},
    (12288, 4096): {65: "yy", 128: "yy", 160: "nn", 192: "nn", 256: "yy", 320: "nn", 576: "yn", 704: "yn"}, (14336, 4096): {128: "yy", 160: "nn", 256: "yy", 512: "nn"},
    (25600, 5120): {128: "yy", 160: "nn", 256: "nn", 512: "nn"}, (11008, 4096): {160: "nn", 256: "yy", 640: "yn"},
}


@pytest.mark.parametrize("columns,width", list(GATED))
def test_the_gated_product_of_many_rows_is_taken_where_it_measured_faster(columns, width):
    for rows, wanted in GATED[columns, width].items():
        assert [kernels.many_swiglu_wins(rows, columns, width, strips) for strips in (True, False)] == [w == "y" for w in wanted], rows


# (columns of the stream, width before them, columns behind, how): {rows: whether handing the norm forward measured at most as long, out of strips and in rows}
HANDED = {
    (1024, 2048, 3072, "gated"): {448: "nn", 704: "nn", 1024: "nn", 1088: "yy", 2048: "yy", 4096: "yy", 8192: "yn"}, (1024, 1024, 2048, "gated"): {65: "yy", 1024: "yy", 8192: "yn"},
    (1024, 3072, 4096, "plain"): {448: "nn", 1024: "nn", 1536: "yn", 3072: "yn", 4096: "nn", 8192: "nn"}, (1024, 3072, 4096, "heads"): {1024: "nn", 1536: "yn", 4096: "yn", 8192: "yn"},
    (2048, 2048, 6144, "gated"): {448: "nn", 576: "yy", 1024: "yy", 4096: "yn", 8192: "nn"}, (2048, 2048, 4096, "plain"): {300: "nn", 576: "yy", 2048: "yy", 3072: "yn", 4096: "nn"},
    (2048, 4096, 4096, "heads"): {576: "yn", 3072: "yn", 4096: "nn"}, (1024, 1024, 4096, "plain"): {300: "yy", 2048: "yy", 3072: "yn", 4096: "nn"}, (2048, 6144, 4096, "plain"): {2048: "nn"},
}


@pytest.mark.parametrize("columns,width,behind,how", list(HANDED))
def test_a_norm_of_many_rows_is_handed_forward_where_that_measured_faster(columns, width, behind, how):
    for rows, wanted in HANDED[columns, width, behind, how].items():
        got = [kernels.many_add_wins(rows, columns, width, strips) and kernels.many_takes_wins(rows, behind, columns, how == "gated", strips, how == "heads") for strips in (True, False)]
        assert got == [w == "y" for w in wanted], rows


@pytest.fixture
def products(monkeypatch):
    """Which products a layer's parts call, without running them."""
    called = []
    monkeypatch.setattr(kernels, "gemm_many", lambda x, w, *a, **k: called.append("many") or k.get("add_into", torch.empty(0)))
    monkeypatch.setattr(kernels, "linear_bf16", lambda x, *a: called.append("library") or x)
    monkeypatch.setattr(kernels, "gemm_split_library", lambda *a, **k: called.append("library"))
    return called


def test_a_sum_whose_norm_nobody_takes_is_left_to_the_library(products):
    """With no room for the norm behind it the product of many rows that adds is the slower one."""
    down = Linear(torch.zeros(1024, 1024, dtype=torch.bfloat16))
    down.strips = down.weight
    x, stream = torch.zeros(700, 1024, dtype=torch.bfloat16), torch.zeros(700, 1024)
    room = kernels.HandedNorm(torch.ones(1024), 1e-6, 700, 1024, "cpu")
    assert down.forward(x, add_into=stream) is not None and products == ["library"]
    assert down.forward(x, add_into=stream, hand=room) is None and products == ["library", "many"]


def test_room_for_a_norm_of_many_rows_is_made_for_a_part_that_takes_it():
    """A projection with a bias, a gate that is no SiLU and a part that knows nothing of it get the norm's rows from the norm itself."""
    asked, batch = [], SimpleNamespace(max_q_len=700, num_seqs=1)
    norm = SimpleNamespace(handoff=lambda rows, device: asked.append(rows) or "room")
    mlp = lambda act: GatedMlp(SimpleNamespace(activation=act, names=None, intermediate_size=128),
                               1024, {"gate_proj.weight": torch.zeros(128, 1024, dtype=torch.bfloat16), "up_proj.weight": torch.zeros(128, 1024, dtype=torch.bfloat16),
                                      "down_proj.weight": torch.zeros(1024, 128, dtype=torch.bfloat16)}, torch.bfloat16, "cpu", {})
    with_bias = SimpleNamespace(takes_norm=lambda rows, batch: Linear(torch.zeros(128, 1024, dtype=torch.bfloat16), torch.zeros(128)).takes_norm(rows))
    stream = torch.zeros(700, 1024)
    assert PreNormBlock._room(norm, stream, mlp("silu"), batch) == "room"
    for taker in (mlp("gelu"), with_bias, SimpleNamespace(), None):
        assert PreNormBlock._room(norm, stream, taker, batch) is None
    assert asked == [700]
    assert PreNormBlock._room(norm, stream[:64], None, batch) == "room"        # (few rows: as their products decide)
    assert PreNormBlock._room(SimpleNamespace(), stream, mlp("silu"), batch) is None


def test_near_contexts_go_to_one_kernel_while_the_workgroups_are_few():
    """Two workgroups a compute unit, one in steps of single tokens; no window, heads of 128 turned whole, a step that says which rows its requests bring."""
    prepare = kernels.QkFusion(None, None, 1e-6, None, None, 128, True)

    def takes(requests, nq, longest=10, near=128, d=128, window=0, prepare=prepare, **more):
        return kernels.near_applies(SimpleNamespace(q_start=0, q_len=0, ctx_len=0, max_ctx_len=1024, near_ctx_len=near, max_q_len=longest, num_seqs=requests, **more), nq, d, window, prepare)

    assert takes(16, 32) and not takes(17, 32) and takes(8, 64) and not takes(9, 64)
    assert takes(4, 64, longest=1) and not takes(5, 64, longest=1) and not takes(8, 64, longest=1)
    assert takes(17, 32, live_seqs=16) and not takes(1, 16, near=256) and not takes(1, 16, near=None) and not takes(1, 16, window=64) and not takes(1, 16, d=64)
    assert not takes(1, 16, prepare=kernels.QkFusion(None, None, 1e-6, None, None, 64, True)) and not takes(1, 16, prepare=kernels.QkFusion(None, None, 1e-6, None, None, 128, False))


def test_tables_that_are_not_the_rotations_go_to_the_kernel_that_says_so():
    """Tables beside a rotation over nothing were refused, or ignored where they are empty, and one table without the other was ignored or refused: by the stand-alone kernel, as now."""
    table, empty = torch.zeros(128, 64), torch.zeros(128, 0)

    def whole(cos, sin, rot):
        return kernels.prepares_whole_heads(128, kernels.QkFusion(None, None, 1e-6, cos, sin, rot, True))

    assert whole(table, table, 128) and whole(None, None, 128) and whole(None, None, 0)
    assert not whole(table, table, 0) and not whole(empty, empty, 0) and not whole(table, None, 128) and not whole(None, table, 128) and not whole(table, table, 64)
