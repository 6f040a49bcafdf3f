"""GPU parity of the balanced work split of paged batches (va_balance.hpp): the cut points
move with the lengths, so batches of many shapes are decoded, each against the oracle's
double reference within the fp16 rounding bound widened by 8 fp32 ulps of each output's
terms (tests/numerics.py cond_bound: among 10^5 outputs some cancel far below the terms
summed, where any fp32 sum's rounding is set by those). Covered: merge groups inside one
run, over two and over many (up to the 64 pieces of one merge), more sequences than
one scan of 64 lengths, empty sequences, equal lengths, sub-groups and masked query
slots, every kernel form, S too small for the plan (static splits), and replays of a
captured step whose lengths change on the device."""
import numpy as np
import pytest

import voltattn_amd as va
from tests import batch_util
from tests.numerics import cond_bound

pytestmark = pytest.mark.gpu

TILED = [va.Fmt.F16M, va.Fmt.Q8M, va.Fmt.Q4M, va.Fmt.Q3M]


def _check(got, ref, mag, what):
    err, bound = np.abs(got.astype(np.float64) - ref), cond_bound(ref, mag)
    assert np.all(np.isfinite(got)), what
    assert np.all(err <= bound), (what, int((err > bound).sum()), float((err / bound).max()))


def _run(fmt, lens, Hq, Hkv, D, G, P, seed, S=0, max_seq_len=None):
    print(f"balance {fmt.label} B={len(lens)} Hq={Hq} Hkv={Hkv} D={D} P={P} S={S} longest={max(lens)}", flush=True)
    cap = max_seq_len or max(lens)
    pb = batch_util.PagedBatch(fmt, lens, Hq, Hkv, D, G, P, seed=seed, max_seq_len=cap, max_pages=-(-cap // P))
    try:
        got = pb.run(S=S)
    finally:
        pb.free()
    for b, L in enumerate(lens):
        if L == 0:
            assert np.all(got[b] == 0.0), b
        else:
            _check(got[b], pb.ref[b], pb.mag[b], (fmt.label, b, L))


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
    _run(fmt, lens, Hq, Hkv, 128, 32, 64, seed=Hq)


@pytest.mark.parametrize("fmt", TILED, ids=lambda f: f.label)
@pytest.mark.parametrize("D,G,Hq", [(128, 64, 4), (64, 32, 2), (64, 64, 8)])
def test_few_long_sequences(fmt, D, G, Hq):
    """A capacity far above the lengths: few merge groups in many pieces; one long sequence
    beside short ones takes the most pieces that a merge holds."""
    _run(fmt, [9000, 130, 1, 700], Hq, 2, D, G, 256, seed=D + G + Hq, max_seq_len=1 << 17)
    _run(fmt, [2100] * 4, Hq, 2, D, G, 64, seed=D + G + Hq + 1, max_seq_len=65536)


@pytest.mark.parametrize("S", [1, 2, 3, 7])
def test_small_workspaces(S):
    """S as the caller chose it: 1 and 2 leave no room for the plan's pieces."""
    _run(va.Fmt.Q8M, _ragged(9, 40, 500), 32, 8, 128, 32, 64, seed=S, S=S)


@pytest.mark.parametrize("fmt,Hq", [(va.Fmt.Q4M, 32), (va.Fmt.F16M, 8)], ids=lambda x: x.label if isinstance(x, va.Fmt) else f"Hq{x}")
def test_captured_step_follows_the_lengths(fmt, Hq):
    Hkv, D, G, P = 8, 128, 32, 64
    full = _ragged(4, 36, 700)
    pb = batch_util.PagedBatch(fmt, full, Hq, Hkv, D, G, P, seed=77)
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
