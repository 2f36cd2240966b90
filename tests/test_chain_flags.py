"""What the waves of a workgroup of a chain share between two tiles of rows lies apart for the two: there is one barrier a tile, so a wave may be in the
next tile while another has not yet read what this one's left.  Read from the sources, since no run shows it reliably."""

from __future__ import annotations

import re
from pathlib import Path

import pytest

HIP = Path(__file__).resolve().parent.parent / "paged-llm-rs_amd" / "csrc" / "hip"


@pytest.mark.parametrize("name,function,flag", [("gemm_chain.hip", "cn_tile", "late"), ("gemm_chain_f32.hip", "cf_tile", "lds.late")])
def test_a_tile_says_that_its_rows_are_late_where_the_next_does_not(name, function, flag):
    source = re.sub(r"//.*", "", (HIP / name).read_text())
    begin = source.index(f"bool {function}(")
    loop = source[source.index("for (int row0", begin):source.index("\n}\n", begin)]
    uses = re.findall(rf"(?<![\w.]){re.escape(flag)}\b(\[\w+\])?", loop)
    assert len(uses) >= 2 and set(uses) == {"[turn]"}, uses
    assert loop.count("turn ^= 1") == 1
