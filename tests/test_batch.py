"""The descriptor of a step on the host: layout, bounds, padding and refusals (no GPU)."""

import numpy as np
import pytest

from paged_llm_rs_amd.cache import CacheManager, GroupGeometry
from paged_llm_rs_amd.engine.batch import (ContextTooLong, ShortTokensOutgrown, StepEntry, TableTooWide, build_batch, context_bound,
                                            token_bucket)
from paged_llm_rs_amd.errors import ConfigError


def manager(blocks=64, block_size=4):
    return CacheManager([GroupGeometry(block_size, blocks, 0)])


def requests(m, lengths, written=None):
    entries = []
    for i, n in enumerate(lengths):
        m.add_sequence(i + 1)
        have = (written or [0] * len(lengths))[i]
        if have:
            assert m.reserve(i + 1, have)
            m.advance(i + 1, have)
        assert m.reserve(i + 1, n)
        entries.append(StepEntry(i + 1, list(range(10, 10 + n)), have, [n - 1]))
    return entries


def piece(batch, name):
    begin, count = batch.layout[name]
    return batch.packed[begin:begin + count].numpy()


def test_buckets():
    assert [token_bucket(n) for n in (1, 16, 17, 33, 64, 65, 128, 1000, 1024, 1025, 2048, 2049)] == \
        [16, 16, 32, 64, 64, 128, 128, 1024, 1024, 1280, 2048, 2304]
    assert [context_bound(n) for n in (1, 1024, 1025, 1537, 5000, 6145)] == [1024, 1024, 1536, 2048, 6144, 8192]


def test_a_step_without_padding_reports_what_it_holds():
    m = manager()
    batch = build_batch(requests(m, [5, 1, 20], written=[0, 9, 3]), m, 1, 100, 0, "cpu")
    assert (batch.num_tokens, batch.num_seqs, batch.live_seqs, batch.num_logit_rows) == (26, 3, 3, 3)
    assert batch.max_q_len == 20 and batch.max_ctx_len == 1024 and batch.tokens_of_short_requests(16) == 6
    assert piece(batch, "positions").tolist() == list(range(5)) + [9] + list(range(3, 23))
    assert piece(batch, "q_start").tolist() == [0, 5, 6] and piece(batch, "ctx_len").tolist() == [5, 10, 23]
    assert piece(batch, "logit_rows").tolist() == [4, 5, 25]


def test_padding_adds_a_request_that_holds_nothing_and_bounds_instead_of_counts():
    m = manager()
    entries = requests(m, [5, 20], written=[0, 3])
    batch = build_batch(entries, m, 1, 100, 0, "cpu", pad_to=32)
    assert (batch.num_tokens, batch.num_seqs, batch.live_seqs) == (32, 3, 2)
    assert batch.max_q_len == 32 and batch.tokens_of_short_requests(16) == 32          # a short request is there: every row might be short
    assert piece(batch, "positions")[25:].tolist() == [-1] * 7 and piece(batch, "seq_of")[25:].tolist() == [2] * 7
    assert piece(batch, "q_start").tolist() == [0, 5, 25] and piece(batch, "q_len").tolist() == [5, 20, 7]
    assert piece(batch, "ctx_len").tolist() == [5, 23, 0] and piece(batch, "state_slots")[2] == -1
    table = piece(batch, "block_table_0").reshape(3, -1)
    assert (table[2] == -1).all() and table[1, 0] >= 0
    # told how many tokens the short requests bring at most, the batch reports that bound; more of them are refused
    bounded = build_batch(entries, m, 1, 100, 0, "cpu", pad_to=32, short_bounds={16: 16})
    assert bounded.tokens_of_short_requests(16) == 16 and bounded.max_q_len == 32
    with pytest.raises(ShortTokensOutgrown):
        build_batch(entries, m, 1, 100, 0, "cpu", pad_to=32, short_bounds={16: 4})
    # the same step without short requests reports no short rows; a full bucket has a request of no rows
    m2 = manager()
    full = build_batch(requests(m2, [16, 16]), m2, 1, 100, 0, "cpu", pad_to=32)
    assert full.tokens_of_short_requests(16) == 0 and piece(full, "q_len").tolist() == [16, 16, 0]
    with pytest.raises(ConfigError):
        build_batch(requests(manager(), [40]), manager(), 1, 100, 0, "cpu", pad_to=32)


def test_fixed_widths_and_bounds_are_kept_or_refused():
    m = manager(block_size=4)
    entries = requests(m, [30])
    batch = build_batch(entries, m, 1, 100, 0, "cpu", widths=[16], ctx_bound=64)
    assert piece(batch, "block_table_0").size == 16 and batch.max_ctx_len == 64
    with pytest.raises(TableTooWide):
        build_batch(entries, m, 1, 100, 0, "cpu", widths=[4])
    with pytest.raises(ContextTooLong):
        build_batch(entries, m, 1, 100, 0, "cpu", ctx_bound=16)


def test_steps_of_one_shape_have_one_layout():
    a, b = manager(), manager()
    one = build_batch(requests(a, [40, 1], written=[0, 7]), a, 1, 100, 0, "cpu", widths=[32], ctx_bound=1024, pad_to=64)
    two = build_batch(requests(b, [13, 30], written=[50, 0]), b, 1, 100, 0, "cpu", widths=[32], ctx_bound=1024, pad_to=64)
    assert one.layout == two.layout and one.packed.numel() == two.packed.numel()
    assert (one.max_q_len, one.tokens_of_short_requests(16), one.num_seqs) == (two.max_q_len, two.tokens_of_short_requests(16), two.num_seqs)


def test_a_step_says_how_near_its_contexts_are():
    """Bounds from 128 on for what shares a prompt's keys out, those of ``context_bound`` past 1,024, and never more than the step was
    laid out for."""
    from paged_llm_rs_amd.engine.batch import near_context

    assert [near_context(n) for n in (1, 128, 129, 256, 257, 513, 1024, 1025, 1537)] == [128, 128, 256, 256, 512, 1024, 1024, 1536, 2048]
    m = manager()
    assert build_batch(requests(m, [5, 1, 20], written=[0, 9, 3]), m, 1, 100, 0, "cpu").near_ctx_len == 128
    m = manager()
    padded = build_batch(requests(m, [40, 1], written=[0, 7]), m, 1, 100, 0, "cpu", widths=[32], ctx_bound=1024, pad_to=64)
    assert (padded.near_ctx_len, padded.max_ctx_len) == (128, 1024)
    m = manager()
    assert build_batch(requests(m, [40], written=[0]), m, 1, 100, 0, "cpu", ctx_bound=64).near_ctx_len == 64


def test_the_wide_product_leaves_full_turns_and_narrow_rows_to_the_others():
    """Which products over very many columns go to the one out of strips: those whose library product would end in a turn of tiles that is
    partly empty, and widths whose rows are a multiple of 4 KB apart; never without strips, past 32 rows, or where the other is the faster."""
    from paged_llm_rs_amd.kernels import wide_wins

    assert all(wide_wins(n, 151936, 5120, True) for n in (1, 8, 16, 17, 24, 32))
    assert not any(wide_wins(n, 131072, w, True) for n in (1, 16, 17, 32) for w in (2560, 3072, 3584, 5120, 7168, 8192))
    assert not any(wide_wins(n, 262144, w, True) for n in (8, 32) for w in (2560, 3072, 5120, 8192))
    assert not any(wide_wins(n, 147456, w, True) for n in (8, 32) for w in (2560, 7168, 8192))
    assert wide_wins(8, 163840, 5120, True) and not wide_wins(24, 163840, 5120, True)          # a turn of few rows' tiles is twice as wide
    assert wide_wins(24, 131072, 2048, True) and wide_wins(24, 131072, 4096, True) and wide_wins(8, 131072, 6144, True)
    assert not wide_wins(16, 131072, 2048, True) and not wide_wins(16, 151936, 4096, True)
    assert not wide_wins(33, 151936, 5120, True) and not wide_wins(24, 151936, 5120, False) and not wide_wins(24, 128256, 5120, True)
    assert not wide_wins(24, 151937, 5120, True) and not wide_wins(24, 151936, 5112, True) and not wide_wins(0, 151936, 5120, True)


def test_only_models_whose_layers_go_by_near_contexts_capture_a_shape_for_each(monkeypatch):
    """One shape with contexts of 40, 100, 300 and 900 tokens: a model without such layers runs it once kernel by kernel and replays one
    capture from then on; one with them has a capture for each bound that its layers see."""
    from types import SimpleNamespace

    import torch

    from paged_llm_rs_amd.engine import step

    made = []

    class Graph:
        def __init__(self, model, cache, entries, widths, ctx_bound, rows, short_bounds):
            made.append(max(e.start + len(e.tokens) for e in entries))

        def run(self, entries):
            return "replayed"

    monkeypatch.setattr(step, "run_step", lambda *args, **kw: "eager")
    monkeypatch.setattr(step, "ShapeGraph", Graph)
    cache = SimpleNamespace(manager=SimpleNamespace(table=lambda seq, group: []), layout=SimpleNamespace(groups=[]), clear_state_slots=None)

    def play(**model):
        made.clear()
        runner = step.StepRunner(SimpleNamespace(device="cpu", portion_limits=(16,), **model), cache)
        for longest in (40, 100, 300, 900) * 3:
            runner.run([StepEntry(1, [0] * 20, longest - 20, [19]), StepEntry(2, [0] * 17, 3, [16])])
        return list(made), runner.eager_steps, runner.graph_steps

    assert play() == ([100], 1, 11)
    assert play(shares_by_near_context=False) == ([100], 1, 11)
    assert play(shares_by_near_context=True) == ([100, 300, 900], 3, 9)        # (bounds of 128, 512 and 1,024)


def test_captured_shapes_are_given_back_by_the_room_that_their_chains_keep(monkeypatch):
    """Steps of few rows may each keep hundreds of kilobytes a row (``step_room_bytes``): the captures that have gone longest without a step go when all of them hold more
    than SHAPE_GRAPH_ROOM_KEPT, those without such room only for their rows."""
    from types import SimpleNamespace

    from paged_llm_rs_amd.engine import step

    class Graph:
        def __init__(self, model, cache, entries, widths, ctx_bound, rows, short_bounds):
            self.rows = rows

        def run(self, entries):
            return "replayed"

    monkeypatch.setattr(step, "run_step", lambda *args, **kw: "eager")
    monkeypatch.setattr(step, "ShapeGraph", Graph)
    cache = SimpleNamespace(manager=SimpleNamespace(table=lambda seq, group: []), layout=SimpleNamespace(groups=[]), clear_state_slots=None)

    def kept(counts, **model):
        runner = step.StepRunner(SimpleNamespace(device="cpu", portion_limits=(), **model), cache)
        for count in counts:
            for _ in range(2):
                runner.run([StepEntry(i + 1, [0] * 2, 0, [1]) for i in range(count)])
        return [(k[0], k[1]) for k, g in runner._shapes.items() if g is not None]

    many = [(16 if 2 * n <= 16 else 32 if 2 * n <= 32 else 64, n) for n in range(1, 33)]
    assert kept(range(1, 33)) == many
    # (room for eight captures of 64 rows)
    monkeypatch.setattr(step, "SHAPE_GRAPH_ROOM_KEPT", 8 * 64 * 1000)
    assert kept(range(1, 33), step_room_bytes=lambda rows: 1000 * rows) == many[-8:]
    assert kept([40, *range(1, 33)], step_room_bytes=lambda rows: 1000 * rows if rows <= 64 else 0) == [(128, 40), *many[-8:]]
    assert kept(range(1, 33), step_room_bytes=lambda rows: 10 ** 9) == many[-1:]


def test_a_captured_step_is_not_replayed_for_contexts_past_its_near_bound(monkeypatch):
    """The near bound chooses a kernel that holds no longer contexts.  A model whose layers do not say that they go by it has none in its captured steps; one whose layers do is refused
    a replay for contexts past the captured ones, whatever the shape says."""
    from types import SimpleNamespace

    import torch

    from paged_llm_rs_amd.engine import step
    from paged_llm_rs_amd.engine.batch import CaptureOutgrown, NotNear

    class Ring:
        def __init__(self, size):
            self.host = torch.zeros(size, dtype=torch.int32)

        advance = sent = lambda self: None

    monkeypatch.setattr(step, "_DescriptorRing", Ring)
    replayed = []

    def graph(**model):
        m = manager(blocks=512)
        entries = requests(m, [20, 17], written=[30, 0])
        model = SimpleNamespace(device="cpu", spec=SimpleNamespace(vocab_size=100, max_positions=0), **model)
        made = step.ShapeGraph(model, SimpleNamespace(manager=m, layout=SimpleNamespace(groups=[0])), entries, [64], 1024, 64, {})
        made.graph = SimpleNamespace(replay=lambda: replayed.append(made))
        return made, m

    def longer(m, written):
        for seq in (1, 2):
            m.free_sequence(seq)
        return requests(m, [20, 17], written=[written, 0])

    for flag in ({}, {"shares_by_near_context": False}):
        made, m = graph(**flag)
        assert made.batch.near_ctx_len == 1024
        made.run(longer(m, 200))
    made, m = graph(shares_by_near_context=True)
    assert made.batch.near_ctx_len == 128
    made.run(longer(m, 100))
    assert len(replayed) == 3
    with pytest.raises(NotNear):
        made.run(longer(m, 109))
    assert issubclass(NotNear, CaptureOutgrown) and len(replayed) == 3
