"""The launch that runs the products behind a layer's attention, against the same products a launch each: the same bits, whether
every workgroup finds its rows in time or has to work them out itself."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = "cuda:0"


def _operands(n, width, inner, ff, after):
    g = torch.Generator(device=DEV).manual_seed(n * 7919 + width + inner + ff + after)

    def draw(*shape):
        return torch.randn(*shape, generator=g, device=DEV)

    weights = [(draw(rows, cols) * cols ** -0.5).bfloat16() for rows, cols in ((width, inner), (2 * ff, width), (width, ff), (after or 16, width))]
    gains = [1 + 0.1 * draw(width) for _ in range(2)]
    return draw(n, width), draw(n, inner).bfloat16(), weights, gains


def _apart(stream, rows, weights, strips, gains, activation, follows=True):
    """The products a launch each; from 16 rows on the norms between them are handed forward."""
    from paged_llm_rs_amd import kernels

    stream = stream.clone()
    n, width = stream.shape
    hands = [kernels.HandedNorm(gain, eps, n, width, DEV) if n >= 16 else None for gain, eps in zip(gains, (1e-6, 1e-5))]

    def behind(hand, w, strip, gain, eps, **how):
        if hand is not None:
            return kernels.gemm_skinny(None, w, handed=hand, strips=strip, **how)
        return kernels.gemm_skinny(stream, w, norm_gain=gain, eps=eps, strips=strip, **how)

    kernels.gemm_skinny(rows, weights[0], add_into=stream, hand=hands[0], strips=strips[0])
    hidden = behind(hands[0], weights[1], strips[1], gains[0], 1e-6, swiglu=True, activation=activation)
    kernels.gemm_skinny(hidden, weights[2], add_into=stream, hand=hands[1] if follows else None, strips=strips[2])
    return stream, behind(hands[1], weights[3], strips[3], gains[1], 1e-5) if follows else None


# Inner widths of 1 to 96 K steps, at the edges where the stretches of K change (32 and 33, 64 and 65 steps); few columns and many.
@pytest.mark.parametrize("looks", [None, 0])
@pytest.mark.parametrize("n,width,inner,ff,after", [
    (1, 1024, 2048, 3072, 4096), (8, 1024, 2048, 3072, 4096), (15, 1024, 2048, 3072, 4096), (3, 32, 32, 32, 16), (15, 64, 1024, 1056, 80),
    (2, 992, 2080, 2048, 48), (7, 512, 3072, 1088, 0), (13, 96, 3040, 64, 112), (16, 1024, 2048, 3072, 4096), (17, 1024, 2048, 3072, 4096),
    (37, 1024, 2048, 2048, 2048), (64, 1024, 2048, 2048, 2048), (33, 96, 3040, 2080, 48), (49, 992, 64, 96, 0), (31, 32, 32, 32, 16)])
def test_a_chain_gives_the_bits_of_its_products(n, width, inner, ff, after, looks):
    from paged_llm_rs_amd import kernels

    activation = "silu" if n % 2 else "gelu_tanh"
    stream, rows, weights, gains = _operands(n, width, inner, ff, after)
    strips = [kernels.weights_in_strips(w) for w in weights]
    assert kernels.chain_applies(n, width, inner, ff, after)
    room = kernels.ChainRoom(n, [(width, ff)] * 3, DEV)
    following = (strips[3], gains[1], 1e-5) if after else None
    want = got = stream
    laid = False
    for layer in room.layers:
        before = got.clone()
        apart = _apart(want, rows, weights, strips, gains, activation, bool(after))
        chain = kernels.gemm_chain(got, laid, rows, layer, strips[0], strips[1], strips[2], gains[0], 1e-6, activation, following, looks=looks)
        assert torch.equal(got, before), "the stream that goes in stays as it is"
        (want, projected), got, laid = apart, chain[0], bool(after)
        if after:
            assert torch.equal(chain[1], projected)
        else:
            assert torch.equal(got, want)
    assert torch.isfinite(want).all()
    # (without a projection behind it, a chain leaves its stream in rows)
    last = kernels.ChainRoom(n, [(width, ff)], DEV).layers[0]
    got, none = kernels.gemm_chain(got, laid, rows, last, strips[0], strips[1], strips[2], gains[0], 1e-6, activation, looks=looks)
    assert none is None and torch.equal(got, _apart(want, rows, weights, strips, gains, activation, False)[0])


@pytest.mark.parametrize("n", [33, 64])
def test_a_chain_of_many_tiles_agrees_with_its_products(n):
    """Where the products of more than 32 rows over many columns are another kernel's, which rounds a sum another way now and then: a
    result in some thousands is the neighbouring bfloat16 (2^-8 of it), so far less than 2^-8 of the whole."""
    from paged_llm_rs_amd import kernels

    stream, rows, weights, gains = _operands(n, 1024, 2048, 3072, 4096)
    strips = [kernels.weights_in_strips(w) for w in weights]
    want = _apart(stream, rows, weights, strips, gains, "silu")[1].double()
    got = kernels.gemm_chain(stream, False, rows, kernels.ChainRoom(n, [(1024, 3072)], DEV).layers[0], strips[0], strips[1], strips[2], gains[0], 1e-6, "silu",
                             (strips[3], gains[1], 1e-5))[1].double()
    assert (got - want).norm() / want.norm() < 2e-4
    assert (got != want).double().mean() < 1e-3


@pytest.mark.parametrize("n", [5, 21])
def test_values_that_are_not_finite_stay_in_their_rows(n):
    """All ones is how a stage sees that a value is not there; a NaN of these bits among the inputs, and infinities in the weights past a
    stretch's end, change neither another row nor whether the chain ends."""
    from paged_llm_rs_amd import kernels

    width, inner, ff = 96, 1056, 96
    stream, rows, weights, gains = _operands(n, width, inner, ff, 48)
    clean = _apart(stream, rows, weights, [kernels.weights_in_strips(w) for w in weights], gains, "silu")
    stream.view(torch.int32)[1, 3] = -1
    rows.view(torch.int16)[3, 10] = -1
    weights[3][5, 7] = float("inf")
    strips = [kernels.weights_in_strips(w) for w in weights]
    want = _apart(stream, rows, weights, strips, gains, "silu")
    for looks in (None, 0):
        got = kernels.gemm_chain(stream, False, rows, kernels.ChainRoom(n, [(width, ff)], DEV).layers[0], strips[0], strips[1], strips[2], gains[0], 1e-6,
                                 "silu", (strips[3], gains[1], 1e-5), looks=looks)[1]
        assert torch.equal(torch.isnan(got), torch.isnan(want[1]))
        assert torch.equal(got.nan_to_num(0.0), want[1].nan_to_num(0.0))
    bad = [r in (1, 3) for r in range(n)]
    assert torch.isnan(want[1]).all(dim=1).tolist() == bad
    assert torch.isinf(want[1][[not b for b in bad], 5]).all() and torch.isfinite(clean[1]).all()


def test_what_a_chain_does_not_take_is_refused():
    from paged_llm_rs_amd import kernels
    from paged_llm_rs_amd.errors import TensorError

    for shape in ((65, 1024, 2048, 3072, 0), (0, 1024, 2048, 3072, 0), (1, 1056, 2048, 3072, 0), (1, 1024, 3104, 3072, 0), (1, 1024, 2048, 3104, 0), (16, 1024, 2048, 3104, 0),
                  (1, 1000, 2048, 3072, 0), (1, 1024, 2040, 3072, 0), (1, 1024, 2048, 3072, 8)):
        assert not kernels.chain_applies(*shape)
    stream, rows, weights, gains = _operands(65, 64, 64, 64, 16)
    strips = [kernels.weights_in_strips(w) for w in weights]
    with pytest.raises(TensorError, match="65 rows"):
        kernels.gemm_chain(stream, False, rows, kernels.ChainRoom(65, [(64, 64)], DEV).layers[0], strips[0], strips[1], strips[2], gains[0], 1e-6, "silu")
    with pytest.raises(TensorError, match="strips"):
        kernels.gemm_chain(stream[:2], False, rows[:2], kernels.ChainRoom(2, [(64, 64)], DEV).layers[0], strips[0][:32], strips[1], strips[2], gains[0], 1e-6, "silu")


def _apart_f32(stream, rows, weights, gains, activation, follows):
    """The 32-bit products, norms and sums a launch each."""
    from paged_llm_rs_amd import kernels

    stream = stream.clone()
    normed = kernels.add_rmsnorm(stream, kernels.gemm_plain(rows, weights[0]), gains[0], 1e-6, torch.empty_like(stream))
    down = kernels.gemm_plain(kernels.gemm_plain_gated(normed, weights[1], activation), weights[2])
    normed = kernels.add_rmsnorm(stream, down, gains[1], 1e-5, torch.empty_like(stream))
    return stream, kernels.gemm_plain(normed, weights[3]) if follows else None


# Parts of K of one, two and three lengths (64, 128 and 192 values), whole and not, fewer of them than sixteen; both tiles of 8 rows.
@pytest.mark.parametrize("looks", [None, 0])
@pytest.mark.parametrize("n,width,inner,ff,after", [
    (1, 1024, 2048, 3072, 4096), (8, 1024, 2048, 3072, 4096), (9, 1024, 2048, 3072, 4096), (16, 1024, 2048, 3072, 4096), (3, 512, 64, 64, 16),
    (7, 576, 960, 1088, 80), (5, 960, 2112, 2048, 0), (13, 1024, 3072, 1024, 48), (12, 640, 1984, 3008, 0)])
def test_a_chain_of_32_bit_products_gives_their_bits(n, width, inner, ff, after, looks):
    from paged_llm_rs_amd import kernels

    g = torch.Generator(device=DEV).manual_seed(n * 7919 + width + inner + ff + after)
    draw = lambda *shape: torch.randn(*shape, generator=g, device=DEV)
    weights = [draw(a, b) * b ** -0.5 for a, b in ((width, inner), (2 * ff, width), (width, ff), (after or 16, width))]
    gains = [1 + 0.1 * draw(width) for _ in range(2)]
    stream, rows = draw(n, width), draw(n, inner)
    if n > 2:       # what is no number, and what is next to none, stays in its row (all ones is how a stage sees that a value is not there)
        stream.view(torch.int32)[1, 3] = -1
        rows[2, 10] = float("inf")
        stream[0, :5], rows[0, :5] = 1e-41, 1e-30
    activation = "silu" if n % 2 else "gelu"
    assert kernels.chain_applies(n, width, inner, ff, after, dtype=torch.float32)
    room = kernels.ChainRoom(n, [(width, ff)] * 3, DEV, torch.float32)
    want = got = stream
    laid = False
    for at, layer in enumerate(room.layers):
        following = (weights[3], gains[1], 1e-5) if after and at < 2 else None
        before = got.clone()
        chain = kernels.gemm_chain(got, laid, rows, layer, weights[0], weights[1], weights[2], gains[0], 1e-6, activation, following, looks=looks)
        assert torch.equal(got.view(torch.int32), before.view(torch.int32)), "the stream that goes in stays as it is"
        (want, projected), got, laid = _apart_f32(want, rows, weights, gains, activation, following is not None), chain[0], following is not None
        for a, b in ((got, want),) if following is None else ((chain[1], projected),):
            assert torch.equal(a.isnan(), b.isnan()) and torch.equal(a.nan_to_num(0.0), b.nan_to_num(0.0))
    finite = want.isfinite().all(dim=1).tolist()
    assert finite == [n <= 2 or r not in (1, 2) for r in range(n)]


def test_what_a_chain_of_32_bit_products_does_not_take_is_refused():
    from paged_llm_rs_amd import kernels
    from paged_llm_rs_amd.errors import TensorError

    for shape in ((17, 1024, 2048, 3072, 0), (0, 1024, 2048, 3072, 0), (1, 1088, 2048, 3072, 0), (1, 448, 2048, 3072, 0), (1, 1024, 3136, 3072, 0),
                  (1, 1024, 2048, 3136, 0), (1, 1000, 2048, 3072, 0), (1, 1024, 2080, 3072, 0), (1, 1024, 2048, 3072, 8)):
        assert not kernels.chain_applies(*shape, dtype=torch.float32)
    draw = lambda *shape: torch.randn(*shape, device=DEV)
    room = kernels.ChainRoom(17, [(512, 64)], DEV, torch.float32).layers[0]
    with pytest.raises(TensorError, match="17 rows"):
        kernels.gemm_chain(draw(17, 512), False, draw(17, 64), room, draw(512, 64), draw(128, 512), draw(512, 64), draw(512), 1e-6, "silu")


# Looks that are over before the attention's rows can be there, and, with a few, not before what the stages in front read: a workgroup then works its
# own heads' rows out, and everything where these have to wait as well.
# One request and many, contexts of no key but the own one and over several rounds of 64, one share and eight; heads of 80 to 128, one and two a key head;
# a window, no rotation, pages of another layer (no write), a row of padding.
@pytest.mark.parametrize("looks", [None, 0, 1, 4, 8, 16])
@pytest.mark.parametrize("nq,nkv,d,rot,contexts,bound,window,writes", [
    (16, 8, 128, 128, [512], 1024, 0, True), (16, 8, 128, 128, [1, 2, 511, 300, 64, 65, 17], 1024, 0, True),
    (16, 8, 128, 128, [1000] * 7, 1024, 0, True), (8, 8, 80, 0, [33, 129], 2048, 100, True), (4, 2, 96, 32, [700, 3, 1], 1024, 0, False),
    (2, 1, 112, 112, [1000], 1024, 0, True)])
def test_a_chain_goes_on_to_the_next_layers_attention(nq, nkv, d, rot, contexts, bound, window, writes, looks):
    """The bits of the chain and then the kernel for single tokens: the stream, the pages, the attended rows."""
    from types import SimpleNamespace

    from paged_llm_rs_amd import kernels

    width, inner, ff, bs, columns = 256, 128, 192, 16, (nq + 2 * nkv) * d
    n = len(contexts) + 1
    stream, rows, weights, gains = _operands(n, width, inner, ff, columns)
    strips = [kernels.weights_in_strips(w) for w in weights]
    blocks = -(-bound // bs)
    g = torch.Generator(device=DEV).manual_seed(n + d)
    table = torch.randperm(len(contexts) * blocks, generator=g, device=DEV).to(torch.int32).view(len(contexts), blocks)
    pools = [torch.randn(table.numel() * bs, nkv * d, generator=g, device=DEV).bfloat16() for _ in range(2)]
    positions = torch.tensor([c - 1 for c in contexts] + [-1], dtype=torch.int32, device=DEV)
    seq_of = torch.tensor([*range(len(contexts)), 0], dtype=torch.int32, device=DEV)
    counters = torch.zeros(n * nq, dtype=torch.int32, device=DEV)
    batch = SimpleNamespace(num_tokens=n, max_q_len=1, max_ctx_len=bound, positions=positions, seq_of=seq_of, has_arrivals=True, arrivals=lambda heads: counters)
    q_gain, k_gain = ((1 + 0.2 * torch.randn(d, generator=g, device=DEV)).bfloat16() for _ in range(2))
    angle = torch.arange(bound, device=DEV)[:, None] * 10000.0 ** (-torch.arange(max(rot // 2, 1), device=DEV) / max(rot // 2, 1))
    prepare = kernels.QkFusion(q_gain, k_gain, 1e-6, angle.cos() if rot else None, angle.sin() if rot else None, rot, writes)
    results = []
    for attends in (False, True):
        kv = SimpleNamespace(k_pool=pools[0].clone(), v_pool=pools[1].clone(), block_table=table, block_size=bs)
        attention = kernels.ChainAttention.of(batch, kv, nq, nkv, d, d ** -0.5, window, prepare) if attends else None
        assert (attention is not None) == attends
        room = kernels.ChainRoom(n, [(width, ff, *((columns,) if attends else ()))], DEV).layers[0]
        out, behind = kernels.gemm_chain(stream, False, rows, room, strips[0], strips[1], strips[2], gains[0], 1e-6, "silu", (strips[3], gains[1], 1e-5),
                                         looks=looks, attention=attention)
        if not attends:
            projected, behind = behind, torch.empty(n, nq * d, dtype=torch.bfloat16, device=DEV)
            kernels.attention_step(projected, behind, batch, kv, nq, nkv, d, d ** -0.5, window, prepare)
        assert not counters.any()
        results.append((out, kv.k_pool, kv.v_pool, behind[:-1]))
    for want, got in zip(*results):
        assert torch.equal(want, got)
    assert torch.equal(results[0][1], pools[0]) != writes


def test_which_attention_a_chain_goes_on_to():
    """Up to a workgroup a compute unit, two query heads a key head, eight shares and 256 keys a share; heads of whole 16 values that sixteen lanes hold."""
    from paged_llm_rs_amd import kernels

    attends, units = kernels.library().pl_gemm_chain_attends, kernels.compute_units()
    assert attends(1, 16, 8, 128, 8, 2048) and attends(1, 8, 8, 80, 1, 256) and attends(1, units, units // 2, 128, 2, 512)
    for n, nq, nkv, d, splits, bound in ((1, 32, 8, 128, 4, 256), (1, 16, 8, 64, 4, 256), (1, 16, 8, 136, 4, 256), (1, 16, 8, 120, 4, 256), (16, 2, 1, 128, 1, 256),
                                         (1, 16, 8, 128, 9, 256), (0, 16, 8, 128, 1, 256), (1, units + 1, units + 1, 128, 1, 256), (1, 16, 8, 128, 4, 1025),
                                         (1, 16, 8, 128, 4, 0), (15, units // 4, units // 8, 128, 4, 256)):
        assert not attends(n, nq, nkv, d, splits, bound)


# Workgroups with two tiles of rows whose looks are over now in the first and now in the second of them, while the stage before is writing: what a
# wave says of one tile must not reach another wave that is still at the other.
@pytest.mark.parametrize("looks", [0, 1, 2, 4, 8])
@pytest.mark.parametrize("n,dtype,ff", [(33, torch.bfloat16, 2048), (64, torch.bfloat16, 2048), (9, torch.float32, 3072), (16, torch.float32, 3072)])
def test_rows_that_come_in_time_for_one_tile_and_not_for_the_next(n, dtype, ff, looks):
    from paged_llm_rs_amd import kernels

    width, inner, after = 1024, 2048, 2048
    stream, rows, weights, gains = _operands(n, width, inner, ff, after)
    weights, rows = [w.to(dtype) for w in weights], rows.to(dtype)
    strips = weights if dtype == torch.float32 else [kernels.weights_in_strips(w) for w in weights]
    results = []
    for tries in (None, looks):
        room = kernels.ChainRoom(n, [(width, ff)] * 12, DEV, dtype)
        got, laid = stream, False
        for layer in room.layers:
            got, projected = kernels.gemm_chain(got, laid, rows, layer, strips[0], strips[1], strips[2], gains[0], 1e-6, "silu", (strips[3], gains[1], 1e-5),
                                                looks=tries)
            laid = True
            results.append((tries, got.clone(), projected))
    for (_, want, want_after), (_, got, got_after) in zip(results[:12], results[12:]):
        assert torch.equal(want, got) and torch.equal(want_after, got_after)
    assert torch.isfinite(results[11][1]).all()


def _time(launch) -> float:
    """Microseconds of ``launch(i)``, the median of nine (the first of which bring the code in)."""
    times = []
    for i in range(9):
        torch.cuda.synchronize()
        begin, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        begin.record()
        launch(i)
        end.record()
        end.synchronize()
        times.append(begin.elapsed_time(end) * 1e3)
    return sorted(times)[4]


@pytest.mark.parametrize("n,dtype", [(1, torch.bfloat16), (8, torch.bfloat16), (8, torch.float32)])
def test_workgroups_without_their_rows_share_what_is_missing(n, dtype):
    """Where no workgroup may wait, each works out what it finds missing and begins with another piece than the next: 45 to 110 us a launch, and 27
    to 44 where they wait.  Each by itself working out all that stands before it took 1,250 (in 32 bits 5,800), so a tenfold tells them apart."""
    from paged_llm_rs_amd import kernels

    stream, rows, weights, gains = _operands(n, 1024, 2048, 3072, 4096)
    weights, rows = [w.to(dtype) for w in weights], rows.to(dtype)
    strips = weights if dtype == torch.float32 else [kernels.weights_in_strips(w) for w in weights]

    def chain(looks):
        rooms = kernels.ChainRoom(n, [(1024, 3072)] * 9, DEV, dtype).layers
        return lambda i: kernels.gemm_chain(stream, False, rows, rooms[i], strips[0], strips[1], strips[2], gains[0], 1e-6, "silu",
                                            (strips[3], gains[1], 1e-5), looks=looks)

    assert _time(chain(0)) < 10 * _time(chain(None))


def test_chains_on_several_streams_give_the_bits_they_give_alone():
    """Four streams whose chains go on to attention, a workgroup a compute unit each: together they fill the chip before any of their projections can begin."""
    from types import SimpleNamespace

    from paged_llm_rs_amd import kernels

    n, nq, nkv, d, bs, layers, splits = 8, 16, 8, 128, 16, 12, 4
    width, inner, ff, columns = 1024, 2048, 3072, (nq + 2 * nkv) * d
    stream, rows, weights, gains = _operands(n, width, inner, ff, columns)
    strips = [kernels.weights_in_strips(w) for w in weights]
    g = torch.Generator(device=DEV).manual_seed(11)
    table = torch.randperm(n * 64, generator=g, device=DEV).to(torch.int32).view(n, 64)
    pools = [torch.randn(n * 64 * bs, nkv * d, generator=g, device=DEV).bfloat16() for _ in range(2)]
    positions, seq_of = torch.arange(505, 505 + n, dtype=torch.int32, device=DEV), torch.arange(n, dtype=torch.int32, device=DEV)
    prepare = kernels.QkFusion(None, None, 1e-6, None, None, 0, False)

    def user():
        counters = torch.zeros(n * nq, dtype=torch.int32, device=DEV)
        batch = SimpleNamespace(num_tokens=n, max_q_len=1, max_ctx_len=1024, positions=positions, seq_of=seq_of, has_arrivals=True, arrivals=lambda heads: counters)
        kv = SimpleNamespace(k_pool=pools[0], v_pool=pools[1], block_table=table, block_size=bs)
        attention = kernels.ChainAttention.of(batch, kv, nq, nkv, d, d ** -0.5, 0, prepare)
        assert attention is not None and attention.splits == splits
        return attention, kernels.ChainRoom(n, [(width, ff, columns)] * layers, DEV), counters

    def run(attention, room):
        got, laid, given = stream, False, []
        for layer in room.layers:
            got, attended = kernels.gemm_chain(got, laid, rows, layer, strips[0], strips[1], strips[2], gains[0], 1e-6, "silu", (strips[3], gains[1], 1e-5),
                                               attention=attention)
            laid = True
            given += [got, attended]
        return given

    alone = run(*user()[:2])
    users = [user() for _ in range(4)]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in users]
    given = []
    for side, (attention, room, _) in zip(streams, users):
        with torch.cuda.stream(side):
            given.append(run(attention, room))
    torch.cuda.synchronize()
    for each, (_, _, counters) in zip(given, users):
        assert all(torch.equal(a, b) for a, b in zip(each, alone)) and not counters.any()
    assert torch.isfinite(alone[-1].float()).all()
