"""Which kernel a call goes to, as far as sizes alone decide it: the rules, asked as the engine asks them (no GPU; a chip of 256 compute units)."""

import pytest

from paged_llm_rs_amd import kernels
from paged_llm_rs_amd.engine.batch import near_context, token_bucket


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
