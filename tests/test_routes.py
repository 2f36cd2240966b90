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
