"""GPU parity of the balanced work split of paged batches (va_balance.hpp): the cut points
move with the lengths, so batches of many shapes are decoded, each against the oracle's
double reference within the fp16 rounding bound widened by 8 fp32 ulps of each output's
terms (tests/numerics.py cond_bound: among 10^5 outputs some cancel far below the terms
summed, where any fp32 sum's rounding is set by those). Which form ran is read from the
workspace (batch_util: the floats written). Covered: merge groups inside one run, over two
and over many (either side of the most that one merge takes, the pieces counted by the
plan's host model), more sequences than one scan of 64 lengths, empty sequences, equal
lengths with and without the plan, sub-groups and masked query slots, every kernel form,
invalid lengths and page ids, S too small for the plan (static splits), no ticket slot (two
passes), replays of a captured step whose lengths change on the device, and two streams."""
import numpy as np
import pytest

import voltattn_amd as va
from tests import batch_util, runs_model
from tests.numerics import cond_bound

pytestmark = pytest.mark.gpu

TILED = [va.Fmt.F16M, va.Fmt.Q8M, va.Fmt.Q4M, va.Fmt.Q3M]


def _check(got, ref, mag, what):
    err, bound = np.abs(got.astype(np.float64) - ref), cond_bound(ref, mag)
    assert np.all(np.isfinite(got)), what
    assert np.all(err <= bound), (what, int((err > bound).sum()), float((err / bound).max()))


def _check_batch(pb, got, skip=()):
    for b, L in enumerate(pb.lens):
        if b in skip:
            continue
        if L == 0:
            assert np.all(got[b] == 0.0), b
        else:
            _check(got[b], pb.ref[b], pb.mag[b], (pb.fmt.label, b, L))


def _run(fmt, lens, Hq, Hkv, D, G, P, seed, S=0, max_seq_len=None):
    print(f"balance {fmt.label} B={len(lens)} Hq={Hq} Hkv={Hkv} D={D} P={P} S={S} longest={max(lens)}", flush=True)
    cap = max_seq_len or max(lens)
    pb = batch_util.PagedBatch(fmt, lens, Hq, Hkv, D, G, P, seed=seed, max_seq_len=cap, max_pages=-(-cap // P))
    try:
        got = pb.run(S=S)
    finally:
        pb.free()
    _check_batch(pb, got)
    return pb.ws_floats


def _ragged(seed, B, top):
    r = np.random.default_rng(seed)
    lens = np.exp(r.uniform(np.log(max(1, top / 64)), np.log(top), B)).astype(int).tolist()
    lens[seed % B] = top
    return lens


@pytest.mark.parametrize("fmt", TILED, ids=lambda f: f.label)
@pytest.mark.parametrize("heads", [(8, 8), (16, 8), (32, 8), (14, 2)], ids=lambda h: f"Hq{h[0]}-Hkv{h[1]}")
def test_more_merge_groups_than_cus(fmt, heads):
    """70 sequences (two scans of lengths), some empty: most runs hold several merge groups."""
    Hq, Hkv = heads
    B = 70 if Hkv == 8 else 140
    lens = _ragged(3, B, 400)
    lens[5] = lens[6] = lens[B - 1] = 0
    cap = 2048 if Hq == Hkv else None            # one query slot: short capacities keep static splits
    assert _run(fmt, lens, Hq, Hkv, 128, 32, 64, seed=Hq, max_seq_len=cap) > 0


@pytest.mark.parametrize("fmt", TILED, ids=lambda f: f.label)
@pytest.mark.parametrize("D,G,Hq", [(128, 64, 4), (64, 32, 2), (64, 64, 8)])
def test_few_long_sequences(fmt, D, G, Hq):
    """A capacity far above the lengths: few merge groups in many pieces."""
    assert _run(fmt, [9000, 130, 1, 700], Hq, 2, D, G, 256, seed=D + G + Hq, max_seq_len=1 << 17) > 0
    assert _run(fmt, [2100] * 4, Hq, 2, D, G, 64, seed=D + G + Hq + 1, max_seq_len=65536) > 0


# (format, query heads over 2 K/V heads, positions of a tile of the plan, work-groups)
FORMS = [(va.Fmt.Q8M, 8, 256, 256), (va.Fmt.Q4M, 4, 256, 256), (va.Fmt.F16M, 2, 128, 512)]


@pytest.mark.parametrize("form", FORMS, ids=lambda f: f"{f[0].label}-Hq{f[1]}")
@pytest.mark.parametrize("over", [0, 1])
def test_most_pieces_of_one_merge(form, over):
    """One long sequence beside short ones, at the longest length whose merge takes all but
    two of the 64 pieces, and a tile more, where the shortest run grows."""
    fmt, Hq, tile, wgs = form
    L = (62 * (256 // tile) + over) * tile - 5              # a run is 256 positions at least
    lens = [L, 1, 3, 200]
    _, pieces, partials = runs_model.plan(lens, tile, 2, wgs)
    assert pieces == 62 if not over else pieces < 50, pieces
    wrote = _run(fmt, lens, Hq, 2, 128, 32, 256, seed=L, max_seq_len=1 << 17)
    assert wrote == partials * (Hq // 2) * (128 + 2)


@pytest.mark.parametrize("fmt", TILED, ids=lambda f: f.label)
@pytest.mark.parametrize("D", [128, 64])
@pytest.mark.parametrize("Hq,P", [(8, 64), (2, 64), (2, 256), (4, 64)], ids=lambda x: str(x))
@pytest.mark.parametrize("B,L,cap", [(4, 9000, 1 << 17), (4, 8193, 1 << 17), (128, 515, 8192), (128, 1, 8192)])
def test_equal_lengths(fmt, D, Hq, P, B, L, cap):
    """8 merge groups in 32 (or 64) pieces, the fewest tiles for them and more, and 256 merge
    groups in one piece each; one tile each, the last one partial or a single row."""
    wrote = _run(fmt, [L] * B, Hq, 2, D, 32, P, seed=D + Hq + P + B, max_seq_len=cap)
    if B == 128:
        assert wrote == 0 or (Hq == 2 and fmt in (va.Fmt.Q4M, va.Fmt.Q3M)), wrote   # one piece; two per CU


BAD = [(va.Fmt.Q8M, 32, 8, 64), (va.Fmt.Q4M, 32, 8, 64), (va.Fmt.Q3M, 14, 2, 64), (va.Fmt.F16M, 16, 8, 64),
       (va.Fmt.F16M, 8, 8, 64), (va.Fmt.Q8M, 8, 8, 128), (va.Fmt.Q3M, 8, 8, 64)]


def _bad_inputs(pb, bad_len, bad_page):
    """Sequences 1 (negative), 3 (above the capacity) and 5, 6, 7 (a page id outside the pool
    on the first, a middle and the last page)."""
    table, seq = pb.table.copy(), pb.seq_lens.copy()
    seq[1], seq[3] = -5, bad_len
    for b, at in ((5, 0), (6, 1), (7, 2)):
        last = -(-pb.lens[b] // pb.P) - 1
        table[b, (0, last // 2, last)[at]] = bad_page
    return table, seq


@pytest.mark.parametrize("case", BAD, ids=lambda c: f"{c[0].label}-Hq{c[1]}-Hkv{c[2]}-P{c[3]}")
@pytest.mark.parametrize("cut", [False, True], ids=["items", "pieces"])
def test_invalid_lengths_and_pages(case, cut):
    """Several items of a run (more merge groups than CUs), or merge groups in many pieces (a
    few sequences far below the capacity): NaN for the invalid sequences only, zeros for the
    empty one, and the neighbours in the same runs exact."""
    fmt, Hq, Hkv, P = case
    if cut:
        lens, cap = [3000, 400, 0, 900, 2500, 5000, 9000, 7000], 1 << 17
    else:
        lens = [90, 300, 0, 280, 300, 200, 310, 250] + _ragged(6, 36 if Hkv == 8 else 140, 320)
        cap = 2048 if Hq == Hkv else 320
    for page in (-1, 1 << 20):
        pb = batch_util.PagedBatch(fmt, lens, Hq, Hkv, 128, 32, P, seed=Hq + P, max_seq_len=cap, max_pages=-(-cap // P))
        try:
            table, seq = _bad_inputs(pb, cap + 1 if page < 0 else 0x7FFFFFFF, page)
            print(f"balance bad inputs {fmt.label} Hq={Hq} Hkv={Hkv} P={P} cut={cut} page={page}", flush=True)
            got = pb.run(table=table, seq_lens=seq)
        finally:
            pb.free()
        assert pb.ws_floats > 0
        for b in (1, 3, 5, 6, 7):
            assert np.all(np.isnan(got[b])), b
        _check_batch(pb, got, skip=(1, 3, 5, 6, 7))


@pytest.mark.parametrize("fmt,D,cap", [(va.Fmt.F16M, 128, 1024), (va.Fmt.Q8M, 128, 1024), (va.Fmt.Q4M, 128, 1536),
                                       (va.Fmt.Q3M, 128, 1536), (va.Fmt.Q8M, 64, 2048)],
                         ids=lambda x: x.label if isinstance(x, va.Fmt) else str(x))
@pytest.mark.parametrize("less", [0, 1])
def test_one_slot_short_capacities_keep_static_splits(fmt, D, cap, less):
    """One work-group per merge group below the line, whose partial stays in the kernel."""
    wrote = _run(fmt, _ragged(5, 40, 300), 8, 8, D, 32, 64, seed=cap + D, max_seq_len=cap - less)
    assert wrote == 0 if less else wrote > 0, wrote


def test_without_a_ticket_slot():
    """hipStreamPerThread gets none: the splits that were picked for the plan, in two passes."""
    lens = _ragged(2, 40, 900)
    pb = batch_util.PagedBatch(va.Fmt.Q8M, lens, 32, 8, 128, 32, 64, seed=21)
    S = va.pick_splits_paged(va.Fmt.Q8M, pb.shape)
    try:
        got = pb.run(S=S, stream=2)                              # hipStreamPerThread
        assert pb.ws_floats == len(lens) * 32 * S * (128 + 2)
        balanced = pb.run(S=S)
        assert 0 < pb.ws_floats < len(lens) * 32 * S * (128 + 2)
    finally:
        pb.free()
    _check_batch(pb, got)
    _check_batch(pb, balanced)


@pytest.mark.parametrize("S", [1, 2, 3, 7])
def test_small_workspaces(S):
    """S as the caller chose it: 1 leaves no room for the plan's pieces."""
    wrote = _run(va.Fmt.Q8M, _ragged(9, 40, 500), 32, 8, 128, 32, 64, seed=S, S=S)
    assert wrote == 0 if S == 1 else 0 < wrote < 40 * 32 * S * (128 + 2)


@pytest.mark.parametrize("fmt,Hq", [(va.Fmt.Q4M, 32), (va.Fmt.F16M, 8)], ids=lambda x: x.label if isinstance(x, va.Fmt) else f"Hq{x}")
def test_captured_step_follows_the_lengths(fmt, Hq):
    Hkv, D, G, P = 8, 128, 32, 64
    full = _ragged(4, 36, 700)
    pb = batch_util.PagedBatch(fmt, full, Hq, Hkv, D, G, P, seed=77, max_seq_len=2048, max_pages=2048 // P)
    st = va.Stream()
    try:
        B = len(full)
        S = va.pick_splits_paged(fmt, pb.shape)
        out, ws = va.DeviceBuffer(B * Hq * D * 2), va.DeviceBuffer(va.ws_bytes(B * Hq, D, S))
        lens = va.DeviceBuffer.from_array(pb.seq_lens)
        pb.bufs += [out, ws, lens]
        quant = pb.kspool is not None
        b = va.PagedBufs(K=pb._dev(pb.kpool), V=pb._dev(pb.vpool), scK=pb._dev(pb.kspool) if quant else 0,
                         scV=pb._dev(pb.vspool) if quant else 0, block_table=pb._dev(pb.table), seq_lens=lens.ptr,
                         q=pb._dev(pb.q), out=out.ptr, ws=ws.ptr)

        def result():
            va.sync()
            return out.download(np.uint16).copy()

        with va.Graph.capture(st) as cap:
            va.decode_paged(fmt, b, pb.shape, S, stream=st)
        r = np.random.default_rng(8)
        for k in range(4):
            now = pb.seq_lens if k == 0 else np.asarray([int(r.integers(0, L + 1)) for L in full], np.int32)
            lens.upload(now)
            cap.graph.launch(st)
            replayed = result()
            va.decode_paged(fmt, b, pb.shape, S)
            assert np.array_equal(replayed, result()), k
            if k == 0:
                got = replayed.view(np.float16).astype(np.float32).reshape(B, Hq, D)
                for i in range(B):
                    _check(got[i], pb.ref[i], pb.mag[i], i)
        cap.graph.destroy()
    finally:
        pb.free()
        st.destroy()
