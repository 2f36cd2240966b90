"""Two things of the chains' waits that are read from the sources, since no run shows them reliably.  What the waves of a workgroup of a chain share between two tiles of rows lies apart for the two: there is one barrier a tile, so a wave may be in the
next tile while another has not yet read what this one's left.  And the
looks for a tile of rows are counted through: at one piece of them, and at all of them."""

from __future__ import annotations

import re
from pathlib import Path

import pytest

HIP = Path(__file__).resolve().parent.parent / "paged-llm-rs_amd" / "csrc" / "hip"


def _loop_over_rows(name, function):
    source = re.sub(r"//.*", "", (HIP / name).read_text())
    begin = source.index(f"bool {function}(")
    return source[source.index("for (int row0", begin):source.index("\n}\n", begin)]


@pytest.mark.parametrize("name,function,flag", [("gemm_chain.hip", "cn_tile", "late"), ("gemm_chain_f32.hip", "cf_tile", "lds.late")])
def test_a_tile_says_that_its_rows_are_late_where_the_next_does_not(name, function, flag):
    loop = _loop_over_rows(name, function)
    uses = re.findall(rf"(?<![\w.]){re.escape(flag)}\b(\[\w+\])?", loop)
    assert len(uses) >= 2 and set(uses) == {"[turn]"}, uses
    assert loop.count("turn ^= 1") == 1


@pytest.mark.parametrize("name,function", [("gemm_chain.hip", "cn_tile"), ("gemm_chain_f32.hip", "cf_tile")])
def test_looks_for_a_tile_are_counted_through(name, function):
    """One counter for the loop that looks at one piece and the loop (or, where K comes in two halves, the loops) that look at all: with one each a
    tile waits two or three times as long as it is told to."""
    loop = _loop_over_rows(name, function)
    assert loop.count("int left = a.looks;") == 1 and loop.count("a.looks") == 1
    assert loop.count("for (; left > 0 && !there; --left)") == 1
    assert loop.count("for (int again = 0; again <= left; ++again)") == 1
    if "half < S" in loop:
        assert re.search(r"if \(!there\) {\s+left = 0;", loop)
