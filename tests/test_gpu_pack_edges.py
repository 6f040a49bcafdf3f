"""GPU: the quantizer, unpacker and cache write path where their lane layouts can go
wrong, bit for bit against the oracle's quantize() and dq() (src/voltattn.cu:705-767):
element counts around a work-group's step, quotients one fp32 step from a rounding
boundary (where a reciprocal cannot decide), non-finite inputs, and appends of row
counts around the span that a work-group takes, at page sizes of any kind."""
import numpy as np
import pytest

import oracle
import voltattn_amd as va

pytestmark = pytest.mark.gpu
LIM = {8: 127, 4: 7, 3: 3}


def _quantize(x, D, G, bits):
    rows = x.size // D
    with va.DeviceBuffer.from_array(x) as dx, va.DeviceBuffer(oracle.packed_bytes(bits, x.size)) as dp, \
            va.DeviceBuffer(rows * (D // G) * 2) as ds:
        va.quantize(bits, G, dx.ptr, rows, D, dp.ptr, ds.ptr)
        va.sync()
        return dp.download(np.uint8), ds.download(np.uint16)


def _near_ties(rng, n, G, lim):
    """Groups whose quotients lie at, and one fp32 step either side of, k + 1/2."""
    x = rng.uniform(-1, 1, (n // G, G)).astype(np.float32)
    s = np.exp2(rng.uniform(-12, 8, n // G)).astype(np.float32)
    x[:, 0] = 1.0
    x *= (s * lim)[:, None]
    sh = np.where(x[:, 0] > 0, x[:, 0] / np.float32(lim), 1).astype(np.float32).astype(np.float16).astype(np.float32)
    k = rng.integers(-lim, lim, (n // G, G)).astype(np.float32) + np.float32(0.5)
    t = (k * sh[:, None]).astype(np.float32)
    t = np.nextafter(t, np.float32(np.inf) * rng.choice([-1, 1], t.shape).astype(np.float32))
    use = (rng.random(x.shape) < 0.6) & (np.abs(t) < np.abs(x[:, :1]))
    use[:, 0] = False
    return np.where(use, t, x).astype(np.float32).ravel()


@pytest.mark.parametrize("bits", [8, 4, 3])
@pytest.mark.parametrize("G,D", [(32, 64), (32, 96), (64, 128)])
@pytest.mark.parametrize("rows", [1, 5, 31, 513])
def test_quantize_edges(bits, G, D, rows):
    rng = np.random.default_rng(bits * 100 + G + rows)
    x = _near_ties(rng, rows * D, G, LIM[bits])
    if rows == 513:
        x[3 * G:3 * G + 4] = [np.inf, -np.inf, np.nan, 1.0]      # scale inf: codes 0
        x[5 * G:6 * G] = 3.0e-9                                  # scale rounds to 0: codes 0
        x[7 * G + 2] = np.nan                                    # ignored by the maximum, code 0
    data, scale = oracle.quantize(x, D, G, bits)
    got, gscale = _quantize(x, D, G, bits)
    assert np.array_equal(gscale, scale)
    assert np.array_equal(got, data)
    with va.DeviceBuffer.from_array(data) as dp, va.DeviceBuffer.from_array(scale) as ds, \
            va.DeviceBuffer(rows * D * 4) as dx:
        va.dequantize(bits, G, dp.ptr, ds.ptr, rows, D, dx.ptr)
        va.sync()
        back = dx.download(np.float32)
    want = oracle.dequant(data, scale, rows, D, G, bits).ravel()
    same = (back.view(np.uint32) == want.view(np.uint32)) | (np.isnan(back) & np.isnan(want))
    assert same.all()


@pytest.mark.parametrize("fmt,G", [(va.Fmt.F16M, 32), (va.Fmt.Q8M, 32), (va.Fmt.Q8M, 64), (va.Fmt.Q4M, 64),
                                   (va.Fmt.Q3M, 32)], ids=lambda x: x.label if isinstance(x, va.Fmt) else str(x))
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("n", [1, 31, 32, 33, 64, 65, 129, 200])
def test_append_spans(fmt, G, D, n):
    """Rows around half a span and whole ones (64 rows at D 128, 128 at D 64), pages of
    48 rows; one sequence starts before position 0, one runs into an invalid page id and
    one past its table: those rows are not written."""
    rng = np.random.default_rng(n * 7 + D + G + int(fmt))
    B, Hkv, P, npg = 4, 3, 48, 5
    start = np.array([0, 47, -3, 230], np.int32)
    table = rng.permutation(B * npg + 1)[:B * npg].reshape(B, npg).astype(np.int32)
    table[1, 1] = -4
    num_pages, bits, quant = B * npg + 1, va.fmt_bits(fmt), va.fmt_bits(fmt) != 16
    pool = np.full((num_pages, Hkv, P, va.row_bytes(fmt, D)), 0xA5, np.uint8)
    spool = np.full((num_pages, Hkv, P, D // G), 0x5A5A, np.uint16)
    x = _near_ties(rng, B * Hkv * n * D, 32, LIM.get(bits, 7)).reshape(B, Hkv, n, D).astype(np.float16)
    print(f"append span {fmt.label} G={G} D={D} n={n}", flush=True)
    shape = va.PagedShape(B, Hkv, Hkv, D, G, P, npg, num_pages, 0)
    bufs = [va.DeviceBuffer.from_array(a) for a in (x.view(np.uint16), start, table, pool, spool)]
    try:
        dx, dst, dtab, dpool, dsp = (b.ptr for b in bufs)
        va.append_kv(fmt, dx, n, dst, dtab, shape, dpool, dsp if quant else 0)
        va.sync()
        got = bufs[3].download(np.uint8).reshape(pool.shape)
        gots = bufs[4].download(np.uint16).reshape(spool.shape)
    finally:
        for b in bufs:
            b.free()
    for b in range(B):
        for r in range(n):
            p = int(start[b]) + r
            if p < 0 or p // P >= npg or not 0 <= table[b, p // P] < num_pages:
                continue
            for h in range(Hkv):
                if quant:
                    d, s = oracle.quantize(x[b, h, r].astype(np.float32), D, G, bits)
                    pool[table[b, p // P], h, p % P], spool[table[b, p // P], h, p % P] = d, s
                else:
                    pool[table[b, p // P], h, p % P] = x[b, h, r].view(np.uint8)
    assert np.array_equal(got, pool)
    assert not quant or np.array_equal(gots, spool)
