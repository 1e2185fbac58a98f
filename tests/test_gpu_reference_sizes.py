"""The reference operators at the sizes where their kernels change path:
words and scalars of a row, segments and lanes of a norm, tiles of a
projection.  Selections and norms are exact; the projection's tolerance is
derived from its sums."""
import numpy as np
import pytest

import oracle
from tests.gpu_util import B, dev, empty, host, ok, stream

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def _lib(hip):
    return hip


@pytest.mark.parametrize("half", [True, False])
@pytest.mark.parametrize("rows,vocab", [
    (1, 1), (2, 3), (5, 7), (3, 9), (3, 8191), (2, 8192), (4, 8193), (3, 65535), (2, 131075)])
def test_greedy_words_scalars_and_special_values(rows, vocab, half):
    """Rows that start at every offset in a word (odd vocabularies), one word,
    one batch of words and more, with ties, NaN (quiet and signalling),
    infinities and signed zeros at the edges."""
    from market_sim_amd import ops
    rng = np.random.default_rng(vocab + rows)
    for special in range(6):
        x = rng.standard_normal((rows, vocab)).astype(np.float32)
        x = np.round(x * 8) / 8          # many exact ties, also at the maximum
        if special == 1:
            x[:] = -np.inf               # no value above -inf: the lowest id
            x[:, : vocab // 3] = np.nan
        elif special == 2:
            x[:] = np.nan                # nothing comparable: token 0
        elif special == 3:
            x = -np.abs(x)
            x[:, vocab // 2:] = -0.0     # -0 and +0 tie
            x[:, vocab - 1] = 0.0
        elif special == 4:
            x[:, vocab - 1] = np.inf     # the last scalar
        elif special == 5:
            x[:, 0] = 100.0              # the first, among NaN
            x[:, 1::2] = np.nan
        bits = x.astype(np.float16).view(np.uint16) if half else x.view(np.uint32)
        if special == 5:                 # signalling NaN: the quiet bit off
            bits = np.where(np.isnan(x), 0x7C01 if half else 0x7F800001, bits).astype(bits.dtype)
        out = empty(rows, np.uint32)
        ld = dev(bits)
        op = ops.greedy_select_f16 if half else ops.greedy_select_f32
        ok(op(B(ld), B(out), rows, vocab, stream()))
        v = np.where(np.isnan(x), -np.inf, x)
        best = v.max(1, keepdims=True)
        want = np.argmax((v == best) & ~np.isnan(x), axis=1)   # 0 where all are NaN
        assert host(out, np.uint32).tolist() == want.tolist(), special


@pytest.mark.parametrize("rows,hidden", [
    (1, 4), (1, 8), (3, 520), (1023, 576), (1025, 72), (2048, 1000), (2049, 2048), (4099, 960),
    (8195, 520), (2050, 4096), (5, 8192), (3, 8200), (4, 4100)])
def test_rms_norm_segments_bit_exact(rows, hidden):
    """One row a wave to eight, full and partial segments and last waves, the
    widest row of the registers and the first past it, in place."""
    from market_sim_amd import ops
    rng = np.random.default_rng(rows + hidden)
    x = (rng.standard_normal((rows, hidden)) * 3).astype(np.float32)
    w = (1 + 0.02 * rng.standard_normal(hidden)).astype(np.float32)
    x[0, :] *= 1e-6                       # FP16 subnormals
    x16, w16 = x.astype(np.float16).view(np.uint16), w.astype(np.float16).view(np.uint16)
    xd, wd = dev(x), dev(w)
    ok(ops.rms_norm_f32(B(xd), B(wd), B(xd), rows, hidden, 1e-5, stream()))
    got = host(xd, np.float32).reshape(rows, hidden)
    assert np.array_equal(got.view(np.uint32), oracle.rms_norm_f32(x, w, 1e-5).view(np.uint32))
    xd, wd = dev(x16), dev(w16)
    out = empty(rows * hidden, np.uint16)
    ok(ops.rms_norm_f16(B(xd), B(wd), B(out), rows, hidden, 1e-5, stream()))
    # (x * inverse) * weight leaves the FP32 multiplier as a half, rounded once
    # from the exact product (v_fma_mixlo_f16): x * inverse comes from the FP32
    # norm under a weight of one, and its product with a half fits a float64
    scaled = oracle.rms_norm_f32(x16.view(np.float16).astype(np.float32),
                                 np.ones(hidden, np.float32), 1e-5)
    # (its zero addend makes a negative zero positive)
    want = (scaled.astype(np.float64) * w16.view(np.float16).astype(np.float64) + 0.0).astype(np.float16)
    assert np.array_equal(host(out, np.uint16).reshape(rows, hidden), want.view(np.uint16))


@pytest.mark.parametrize("rows,inf,outf", [
    (1, 32, 17), (16, 96, 4129), (17, 64, 5000), (32, 160, 193), (33, 576, 8200), (64, 64, 4097),
    (65, 1024, 300), (128, 96, 12345), (129, 96, 4097), (700, 160, 9001), (1100, 64, 20008),
    (1030, 32, 20008)])
def test_linear_f16_paths_random(rows, inf, outf):
    """The streamed projection at the edges of its row counts (16, 32, 64,
    128) and the tiled one past them, several tiles a workgroup: a half chunk
    of features at the end, partial and single token blocks, odd widths; every output within half an FP16 ulp plus
    the FP32 accumulation bound 2 H 2^-24 sum |x w| of the exact product."""
    from market_sim_amd import ops
    rng = np.random.default_rng(rows * 7 + inf)
    x = rng.uniform(-1.0, 1.0, (rows, inf)).astype(np.float16)
    w = rng.uniform(-1.0, 1.0, (outf, inf)).astype(np.float16)
    out = empty(rows * outf, np.uint16)
    xd, wd = dev(x.view(np.uint16)), dev(w.view(np.uint16))
    ok(ops.linear_f16(B(xd), B(wd), B(out), rows, inf, outf, stream()))
    got = host(out, np.uint16).reshape(rows, outf).view(np.float16).astype(np.float64)
    x64, w64 = x.astype(np.float64), w.astype(np.float64)
    exact = x64 @ w64.T
    mag = np.abs(x64) @ np.abs(w64).T
    half_ulp = np.spacing(np.maximum(np.abs(got), np.abs(exact)).astype(np.float16)).astype(
        np.float64) / 2
    assert np.all(np.abs(got - exact) <= half_ulp + 2.0 * inf * 2.0 ** -24 * mag)


@pytest.mark.parametrize("rows,open_rows,vocab,hidden", [
    (3, 1, 17, 64), (40, 33, 48, 128), (9, 4, 4097, 576), (70, 65, 8200, 640), (5, 2, 70001, 1088)])
def test_stream_head_tiles_match_the_oracle(rows, open_rows, vocab, hidden):
    """Unrestricted rows beside gathered ones: one, two and three panel tiles,
    tiles of two 16-token blocks up to sixteen, two rounds, a partial last
    tile, one token past a block."""
    from market_sim_amd import workloads as wl
    from market_sim_amd.tail import DeviceTail
    w = wl.ragged_pack("stream", 3, vocab, hidden, rows, "uniform", max(1, vocab // 20),
                       open_rows / rows)
    tok, sc, nx = DeviceTail(w, sorted_lists=False).run()
    etok, esc, enx = oracle.decode_tail(w.x, w.norm_weight, w.epsilon, w.embedding, w.row_state,
                                        w.state_offsets, w.state_tokens, threads=8)
    assert w.unrestricted_rows.size == open_rows
    assert np.array_equal(tok, etok) and np.array_equal(nx, enx)
    assert np.array_equal(sc.view(np.uint32), esc.view(np.uint32))


@pytest.mark.parametrize("hidden", [8, 520, 576, 960, 2048, 100])
@pytest.mark.parametrize("width", [1, 3, 128, 129, 515])
def test_head_words_blocks_and_ties(hidden, width):
    """Rows of whole words and not, lists of one block, one candidate more and
    several; equal table rows (the lower id wins), NaN and infinite rows, an
    all-NaN list, a list with an id past the vocabulary and empty ones."""
    from market_sim_amd import ops
    rng = np.random.default_rng(hidden + width)
    rows, vocab = 9, 1200
    h = rng.standard_normal((rows, hidden)).astype(np.float16)
    e = (rng.standard_normal((vocab, hidden)) * 0.05).astype(np.float16)
    e[600:1200] = e[0:600]              # every score twice
    e[5, hidden // 2] = np.nan
    e[7, 0] = np.inf
    e[40:60] = np.nan
    allowed = np.stack([rng.permutation(vocab)[:width] for _ in range(rows)]).astype(np.uint32)
    counts = rng.integers(1, width + 1, rows).astype(np.uint32)
    counts[0] = width
    counts[1] = 0
    counts[2] = width + 1
    allowed[3, :] = 40 + np.arange(width) % 20
    allowed[4, counts[4] - 1] = vocab
    hb, eb = h.view(np.uint16), e.view(np.uint16)
    out = empty(rows, np.uint32)
    keep = [dev(x) for x in (hb, eb, allowed, counts)]
    ok(ops.restricted_output_head_f16(*[B(t) for t in keep], B(out), rows, hidden, vocab, width,
                                      stream()))
    want, _ = oracle.restricted_output_head_f16(hb, eb, allowed, counts, width)
    assert host(out, np.uint32).tolist() == want.tolist()


@pytest.mark.parametrize("order", [0, 1])
@pytest.mark.parametrize("rows,lists,hidden", [
    (600, 1, 576), (530, 9, 64), (513, 8, 4096), (700, 33, 1024), (520, 71, 1024), (520, 127, 576),
    (3, 128, 576), (700, 50, 576), (500, 100, 576), (250, 128, 576), (1030, 16, 2048)])
def test_one_kernel_tail_stages_the_longest_list(rows, lists, hidden, order):
    """Packs of more rows than compute units, one part or two: the stage holds
    exactly the longest list (one row of the table up to all that fit) or a
    share of it, in two rounds and more.  Every second list is the longest; one
    row's state lies beyond the table, one list ends in an id outside the
    vocabulary, one row is all NaN."""
    from market_sim_amd import workloads as wl
    from market_sim_amd.tail import DeviceTail
    w = wl.ragged_pack("short", 11, 3000, hidden, rows, "uniform", lists, 0.0, size_lo=lists)
    keep = np.ones(w.state_tokens.size, bool)
    offs = w.state_offsets.astype(np.int64)
    for s in range(1, w.states, 2):       # shorter by s % lists ids
        keep[offs[s + 1] - s % lists:offs[s + 1]] = False
    cut = np.concatenate([[0], np.cumsum(keep)])[offs]
    w.state_tokens, w.state_offsets = w.state_tokens[keep], cut.astype(np.uint32)
    if w.state_next is not None:
        w.state_next = w.state_next[keep]
    w.row_state = w.row_state.copy()
    w.row_state[rows // 2] = w.states + 7
    w.state_tokens = w.state_tokens.copy()
    w.state_tokens[w.state_offsets[w.row_state[0] + 1] - 1] = w.vocab
    w.x = w.x.copy()
    w.x[2] = np.nan
    tail = DeviceTail(w, order=order)
    assert tail.fused
    tok, sc, nx = tail.run()
    assert tok[0] == tok[rows // 2] == 0xFFFFFFFF and np.isnan(sc[2])
    etok, esc, enx = oracle.decode_tail(w.x, w.norm_weight, w.epsilon, w.embedding, w.row_state,
                                        w.state_offsets, w.state_tokens, state_next=w.state_next,
                                        next_table=w.next_table, order=order, threads=8)
    nan = np.isnan(esc)
    assert np.array_equal(tok, etok) and np.array_equal(nx, enx)
    assert np.array_equal(np.isnan(sc), nan)
    assert np.array_equal(sc.view(np.uint32)[~nan], esc.view(np.uint32)[~nan])


@pytest.mark.parametrize("rows,vocab,hidden", [
    (3, 17, 64), (65, 203, 64), (130, 4099, 576), (257, 1026, 640), (9, 8193, 1088)])
def test_full_comparator_scores_at_row_ends(rows, vocab, hidden):
    """The FP32 projection under the full-vocabulary comparator: rows that end
    inside a lane's four tokens, in a block and in a tile; one M-tile and two;
    half a chunk at the end of K."""
    from market_sim_amd import workloads as wl
    from market_sim_amd.tail import DeviceTail
    w = wl.ragged_pack("full", 7, vocab, hidden, rows, "uniform", max(1, vocab // 3), 0.4)
    tok, sc, nx = DeviceTail(w, full=True).run()
    etok, esc, enx = oracle.decode_tail(w.x, w.norm_weight, w.epsilon, w.embedding, w.row_state,
                                        w.state_offsets, w.state_tokens, threads=8)
    assert np.array_equal(tok, etok) and np.array_equal(nx, enx)
    assert np.array_equal(sc.view(np.uint32), esc.view(np.uint32))
