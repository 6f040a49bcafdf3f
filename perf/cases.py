"""The work that programs give this library, as measurable cases.

A case names an entry point and its sizes:

* ``mha``: one decode step of a model's attention layers, every query head with
  its own K/V head (``voltattn_amd.launch``), launched call by call or replayed
  from a captured graph as a serving loop would;
* ``gqa``: one grouped-query decode step of one sequence (``decode_gqa``);
* ``paged``: one decode step of a batch of sequences of different lengths over
  a page pool, through the PyTorch op;
* ``step``: what a serving loop does per token and layer: append the new K and
  V rows of every sequence to the pool, then decode (the C ABI's mirror);
* ``append``: the prompt's rows written into the pool (PyTorch op);
* ``quantize`` / ``dequantize``: whole caches packed and unpacked (PyTorch ops).

K, V and q are N(0, 1) draws, as in the tests and the benchmark; quantized caches
come from the per-group symmetric quantizer, restated here in plain torch.
The one-position-per-wave formats (f16, q8, q4 without "+") are kept as the
control that the others are compared with, and are no case of their own.
"""
from __future__ import annotations

import math
import random

import torch

import voltattn_amd as va
import voltattn_amd.torch_ops  # noqa: F401  (registers torch.ops.voltattn)

BITS = {"f16+": 16, "q8+": 8, "q4+": 4, "q3+": 3}
LIMIT = {8: 127, 4: 7, 3: 3}
LARGEST = 950_000_000          # bytes of a drawn case at most: the longest listed context's


def listed():
    return [
        # the smallest call there is in practice: a small model's first tokens; launch latency only
        {"name": "mha q4 tiny", "kind": "mha", "fmt": "q4+", "H": 8, "D": 64, "G": 32, "L": 257, "layers": 1, "graph": False},
        # a chat-length context, four layers of it replayed from one graph: fixed cost per layer
        {"name": "mha q8 4k graph", "kind": "mha", "fmt": "q8+", "H": 32, "D": 128, "G": 32, "L": 4096, "layers": 4, "graph": True},
        # the benchmark's uncompressed shape
        {"name": "mha f16 16k", "kind": "mha", "fmt": "f16+", "H": 32, "D": 128, "G": 64, "L": 16384, "layers": 1, "graph": False},
        # 40 heads do not divide the CUs, and no tile divides the length
        {"name": "mha q4 odd", "kind": "mha", "fmt": "q4+", "H": 40, "D": 128, "G": 64, "L": 10007, "layers": 1, "graph": False},
        # the longest context the benchmark has
        {"name": "mha q3 256k", "kind": "mha", "fmt": "q3+", "H": 32, "D": 128, "G": 32, "L": 262144, "layers": 1, "graph": False},
        # grouped heads over a long context, four query heads to a K/V head
        {"name": "gqa q8 64k", "kind": "gqa", "fmt": "q8+", "Hq": 32, "Hkv": 8, "D": 128, "G": 32, "L": 65536},
        # eight query heads to a K/V head, a ragged length
        {"name": "gqa q4 wide", "kind": "gqa", "fmt": "q4+", "Hq": 64, "Hkv": 8, "D": 128, "G": 32, "L": 20011},
        # a batch in mid-flight: sequences of very different lengths
        {"name": "paged q8 ragged", "kind": "paged", "fmt": "q8+", "B": 48, "Hq": 32, "Hkv": 8, "D": 128, "G": 32, "page": 256, "L": 16384, "mix": 1},
        # many short sequences, one new token each
        {"name": "step q4 many", "kind": "step", "fmt": "q4+", "B": 64, "Hq": 32, "Hkv": 8, "D": 128, "G": 32, "page": 64, "L": 3000, "mix": 2},
        # prompts of four sequences entering the cache
        {"name": "append q8 prompt", "kind": "append", "fmt": "q8+", "B": 4, "Hkv": 8, "D": 128, "G": 32, "page": 256, "n": 8192, "mix": 3},
        # a whole uncompressed cache packed, and one unpacked
        {"name": "quantize q4", "kind": "quantize", "fmt": "q4+", "H": 32, "L": 32768, "D": 128, "G": 32},
        {"name": "dequantize q3", "kind": "dequantize", "fmt": "q3+", "H": 32, "L": 16384, "D": 128, "G": 64},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["mha", "mha", "gqa", "gqa", "paged", "paged", "step", "append", "quantize", "dequantize"])
    while True:
        D = rng.choice([64, 128, 128, 128])
        G = rng.choice([32, 64])
        fmt = rng.choice(["f16+", "q8+", "q8+", "q4+", "q4+", "q3+"])
        hkv = rng.choice([2, 4, 8])
        c = {"kind": kind, "fmt": fmt, "D": D, "G": G}
        if kind == "mha":
            c.update(H=rng.choice([8, 12, 16, 20, 32, 40, 64]), L=_log(rng, 100, 262144),
                     layers=rng.choice([1, 2, 4]), graph=rng.random() < 0.5)
        elif kind == "gqa":
            c.update(Hkv=hkv, Hq=hkv * rng.choice([2, 3, 4, 6, 7, 8]), L=_log(rng, 300, 262144))
        elif kind in ("paged", "step"):
            c.update(B=_log(rng, 1, 96), Hkv=hkv, Hq=hkv * rng.choice([1, 2, 4, 7, 8]),
                     page=rng.choice([64, 128, 256]), L=_log(rng, 300, 32768), mix=rng.randrange(1 << 20))
        else:
            if kind != "append":
                c["fmt"] = rng.choice(["q8+", "q4+", "q3+"])
                c.update(H=rng.choice([8, 12, 32, 40]), L=_log(rng, 500, 65536))
            else:
                c.update(B=_log(rng, 1, 64), Hkv=hkv, page=rng.choice([64, 128, 256]), n=_log(rng, 1, 8192),
                         mix=rng.randrange(1 << 20))
        if work(c)["bytes"] <= LARGEST:
            return c


# ------------------------------------------------------------------- sizes --
def _lens(c):
    """Positions of each sequence: spread over 1/32 .. 1 of the longest, which is there."""
    r = random.Random(c["mix"] * 1009 + c["B"])
    lens = [_log(r, max(1, c["L"] // 32), c["L"]) for _ in range(c["B"])]
    lens[r.randrange(c["B"])] = c["L"]
    return lens


def _starts(c):
    """Positions already in the cache before the appended rows."""
    r = random.Random(c["mix"] * 1009 + c["B"])
    return [r.randrange(0, 2 * c["page"]) for _ in range(c["B"])]


def _row(c):
    """Bytes of one K (or V) row of one head with its scales."""
    b = BITS[c["fmt"]]
    return c["D"] * b // 8 + (0 if b == 16 else 2 * (c["D"] // c["G"]))


def work(case):
    c, D = case, case["D"]
    if c["kind"] == "mha":
        n = c["H"] * c["L"] * c["layers"]
        return {"bytes": 2 * n * _row(c) + 4 * c["layers"] * c["H"] * D, "flops": 4 * n * D}
    if c["kind"] == "gqa":
        return {"bytes": 2 * c["Hkv"] * c["L"] * _row(c) + 4 * c["Hq"] * D, "flops": 4 * c["Hq"] * c["L"] * D}
    if c["kind"] in ("paged", "step"):
        n = sum(_lens(c))
        new = 2 * c["B"] * c["Hkv"] * (2 * D + _row(c)) if c["kind"] == "step" else 0
        return {"bytes": 2 * c["Hkv"] * n * _row(c) + 4 * c["B"] * c["Hq"] * D + new, "flops": 4 * c["Hq"] * n * D}
    if c["kind"] == "append":
        n = c["B"] * c["Hkv"] * c["n"]
        return {"bytes": n * (2 * D + _row(c)), "flops": n * D}
    n = c["H"] * c["L"]
    return {"bytes": n * (4 * D + _row(c)), "flops": n * D}


def tolerance(case):
    # Packing and unpacking are exact by definition. Attention sums in fp32 and rounds to
    # fp16 once, so two correct sums differ only where that rounding goes the other way.
    # Against the float64 result rounded to fp16 the cases were off by 0 .. 2.7e-5 (2-norm),
    # and by one fp16 step (9e-4) at most; an output of few values moves more per step.
    if case["kind"] in ("append", "quantize", "dequantize"):
        return "exact"
    return {"rel": 2e-4, "max": 4e-3}


# ------------------------------------------------------------------ inputs --
def _gen(seed):
    return torch.Generator("cuda").manual_seed(int(seed))


def _normal(shape, gen, dtype=torch.float32):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)


def _pack(x, bits, G):
    """Symmetric per-group codes and fp16 scales of fp32 x [..., D]: packed uint8 [..., D*bits/8]."""
    lim = LIMIT[bits]
    g = x.unflatten(-1, (-1, G))
    amax = g.abs().amax(-1)
    scale = torch.where(amax > 0, amax / lim, torch.ones_like(amax)).half()
    v = (g / scale.float().unsqueeze(-1)).round().clamp(-lim, lim).flatten(-2).to(torch.int32)
    if bits == 8:
        return v.to(torch.int8).view(torch.uint8), scale
    if bits == 4:
        v = (v + 8).unflatten(-1, (-1, 2))
        return (v[..., 0] | (v[..., 1] << 4)).to(torch.uint8), scale
    v = (v + 4).unflatten(-1, (-1, 8))
    w = sum(v[..., i] << (3 * i) for i in range(8))
    return torch.stack([(w >> s) & 255 for s in (0, 8, 16)], -1).flatten(-2).to(torch.uint8), scale


def _unpack(p, scale, bits, G):
    """float64 values of packed rows (fp16 rows when bits is 16)."""
    if bits == 16:
        return p.double()
    if bits == 8:
        v = p.view(torch.int8).to(torch.int32)
    elif bits == 4:
        w = p.to(torch.int32)
        v = torch.stack([w & 15, w >> 4], -1).flatten(-2) - 8
    else:
        w = p.to(torch.int32).unflatten(-1, (-1, 3))
        w = w[..., 0] | (w[..., 1] << 8) | (w[..., 2] << 16)
        v = torch.stack([(w >> (3 * i)) & 7 for i in range(8)], -1).flatten(-2) - 4
    return (v.double().unflatten(-1, (-1, G)) * scale.double().unsqueeze(-1)).flatten(-2)


def _cache(c, lead, gen):
    """K or V rows [*lead, row] (+ scales) of N(0, 1) values, made a block at a time."""
    bits, D, step = BITS[c["fmt"]], c["D"], 1 << 19
    n = math.prod(lead)
    if bits == 16:
        out = torch.empty((n, D), dtype=torch.float16, device="cuda")
        for i in range(0, n, step):
            out[i:i + step] = _normal((min(step, n - i), D), gen)
        return out.view(lead + (D,)), None
    pay = torch.empty((n, D * bits // 8), dtype=torch.uint8, device="cuda")
    sc = torch.empty((n, D // c["G"]), dtype=torch.float16, device="cuda")
    for i in range(0, n, step):
        pay[i:i + step], sc[i:i + step] = _pack(_normal((min(step, n - i), D), gen), bits, c["G"])
    return pay.view(lead + (-1,)), sc.view(lead + (-1,))


def _ptr(t):
    return 0 if t is None else t.data_ptr()


class State:
    """What a program holds between steps; a captured graph is given back with it."""

    graph = stream = None

    def __del__(self):
        if self.graph is not None:
            self.graph.destroy()
            self.stream.destroy()


def _int32(x):
    return torch.tensor(x, dtype=torch.int32, device="cuda")


def _pool(c, s, lens, gen, seed, both=True):
    """A page pool with the sequences' pages scattered over it."""
    P = c["page"]
    need = [-(-n // P) for n in lens]
    s.table_host = [[0] * max(need) for _ in need]
    ids = list(range(sum(need) + 2))
    random.Random(seed).shuffle(ids)
    for row, n in zip(s.table_host, need):
        row[:n] = [ids.pop() for _ in range(n)]
    s.table = _int32(s.table_host)
    lead = (sum(need) + 2, c["Hkv"], P)
    s.k, s.ks = _cache(c, lead, gen)
    if both:
        s.v, s.vs = _cache(c, lead, gen)


def prepare(case, seed):
    c, s = dict(case), State()
    s.c, s.f = c, va.Fmt.parse(c["fmt"])
    gen = _gen(seed)
    kind, D, G = c["kind"], c["D"], c["G"]
    f16 = lambda *shape: torch.empty(shape, dtype=torch.float16, device="cuda")  # noqa: E731
    if kind in ("mha", "gqa"):
        Hq, Hkv = (c["H"], c["H"]) if kind == "mha" else (c["Hq"], c["Hkv"])
        S = va.pick_splits(s.f, Hq, c["L"], D) if kind == "mha" else va.pick_splits_gqa(s.f, Hq, Hkv, c["L"], D)
        s.S, s.layers, s.bufs, s.outs = S, [], [], []
        ws = torch.empty(va.ws_bytes(Hq, D, S) // 4, device="cuda")
        for _ in range(c.get("layers", 1)):
            q = _normal((Hq, D), gen, torch.float16)
            k, ks = _cache(c, (Hkv, c["L"]), gen)
            v, vs = _cache(c, (Hkv, c["L"]), gen)
            s.layers.append((q, k, v, ks, vs, ws))
            s.outs.append(f16(Hq, D))
            s.bufs.append(va.DeviceBufs(K=_ptr(k), V=_ptr(v), scK=_ptr(ks), scV=_ptr(vs), q=_ptr(q),
                                        out=_ptr(s.outs[-1]), ws=_ptr(ws)))
        if c.get("graph"):
            torch.cuda.synchronize()
            s.stream = va.Stream()
            with va.Graph.capture(s.stream) as cap:
                for b in s.bufs:
                    va.launch(s.f, b, Hq, c["L"], D, S, G=G, stream=s.stream)
            s.graph = cap.graph
    elif kind in ("paged", "step"):
        lens = _lens(c)
        _pool(c, s, lens, gen, seed)
        s.lens = _int32(lens)
        s.q = _normal((c["B"], c["Hq"], D), gen, torch.float16)
        if kind == "step":
            s.newk, s.newv = (_normal((c["B"], c["Hkv"], 1, D), gen, torch.float16) for _ in "kv")
            s.start = _int32([n - 1 for n in lens])
            s.out = f16(c["B"], c["Hq"], D)
            s.shape = va.PagedShape(c["B"], c["Hq"], c["Hkv"], D, G, c["page"], s.table.shape[1], s.k.shape[0], c["L"])
            s.S = va.pick_splits_paged(s.f, s.shape)
            s.ws = torch.empty(va.ws_bytes(c["B"] * c["Hq"], D, s.S) // 4, device="cuda")
            s.bufs = va.PagedBufs(K=_ptr(s.k), V=_ptr(s.v), scK=_ptr(s.ks), scV=_ptr(s.vs), block_table=_ptr(s.table),
                                  seq_lens=_ptr(s.lens), q=_ptr(s.q), out=_ptr(s.out), ws=_ptr(s.ws))
    elif kind == "append":
        starts = _starts(c)
        s.x = _normal((c["B"], c["Hkv"], c["n"], D), gen, torch.float16)
        s.start = _int32(starts)
        _pool(c, s, [a + c["n"] for a in starts], gen, seed, both=False)
    else:
        s.x = _normal((c["H"], c["L"], D), gen)
        if kind == "dequantize":
            s.p, s.sc = _cache(c, (c["H"], c["L"]), gen)
            del s.x
    torch.cuda.synchronize()
    return s


# --------------------------------------------------------------------- run --
def run(s):
    c, ops = s.c, torch.ops.voltattn
    kind, D, G = c["kind"], c["D"], c["G"]
    if kind == "mha":
        if s.graph is not None:
            s.graph.launch()
        else:
            for b in s.bufs:
                va.launch(s.f, b, c["H"], c["L"], D, s.S, G=G)
        return s.outs
    if kind == "gqa":
        va.decode_gqa(s.f, s.bufs[0], c["Hq"], c["Hkv"], c["L"], D, S=s.S, G=G)
        return s.outs
    if kind == "paged":
        return ops.decode_paged(s.q, s.k, s.v, s.ks, s.vs, s.table, s.lens, c["fmt"], c["L"], G)
    if kind == "step":
        for x, p, sc in ((s.newk, s.k, s.ks), (s.newv, s.v, s.vs)):
            va.append_kv(s.f, _ptr(x), 1, _ptr(s.start), _ptr(s.table), s.shape, _ptr(p), _ptr(sc))
        va.decode_paged(s.f, s.bufs, s.shape, s.S)
        return s.out, s.k, s.v, s.ks, s.vs
    if kind == "append":
        ops.append_kv(s.x, s.start, s.table, s.k, s.ks, c["fmt"], G)
        return s.k, s.ks
    if kind == "quantize":
        return ops.quantize(s.x, BITS[c["fmt"]], G)
    return ops.dequantize(s.p, s.sc, BITS[c["fmt"]], G)


# ------------------------------------------------------------------- exact --
def _attend(q, k, v):
    """float64 attention of query rows q [n, D] over one head's k, v [L, D]."""
    p = torch.softmax((q.double() @ k.T) / math.sqrt(q.shape[-1]), -1)
    return p @ v


def exact(case, seed):
    c = dict(case)
    if c["kind"] in ("append", "quantize"):
        return None                                   # bytes, compared as they are
    s = prepare(dict(c, graph=False), seed)
    bits, G = BITS[c["fmt"]], c["G"]
    if c["kind"] == "dequantize":
        return torch.cat([_unpack(s.p[h:h + 1], s.sc[h:h + 1], bits, G) for h in range(c["H"])])
    rows = lambda p, sc: _unpack(p, sc, bits, G)      # noqa: E731
    if c["kind"] in ("mha", "gqa"):
        outs = []
        for q, k, v, ks, vs, _ in s.layers:
            n = q.shape[0] // k.shape[0]
            outs.append(torch.cat([_attend(q[h * n:(h + 1) * n], rows(k[h], None if ks is None else ks[h]),
                                           rows(v[h], None if vs is None else vs[h])) for h in range(k.shape[0])]))
        return outs
    lens, n, P = _lens(c), c["Hq"] // c["Hkv"], c["page"]
    out = torch.empty(s.q.shape, dtype=torch.float64, device="cuda")
    for b, L in enumerate(lens):
        pages = torch.tensor(s.table_host[b][:-(-L // P)], device="cuda")
        kb, vb = ((rows(p[pages], None if sc is None else sc[pages])).transpose(0, 1).flatten(1, 2)[:, :L]
                  for p, sc in ((s.k, s.ks), (s.v, s.vs)))
        if c["kind"] == "step":                       # the new row replaces the last position
            for x, t in ((s.newk, kb), (s.newv, vb)):
                new = x[b, :, 0].float()
                t[:, L - 1] = new.double() if bits == 16 else _unpack(*_pack(new, bits, G), bits, G)
        for h in range(c["Hkv"]):
            out[b, h * n:(h + 1) * n] = _attend(s.q[b, h * n:(h + 1) * n], kb[h], vb[h])
    return (out, None, None, None, None) if c["kind"] == "step" else out
