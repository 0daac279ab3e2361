"""The work this library is used for, as measurable cases: trellis-quantized linears from one decode row to a prefill
chunk, routed expert layers at the same widths, and the encoder's search.

A case is a dict of plain values.  `listed()` holds the fixed ones, `draw(rng)` one more of the same ranges;
`prepare(case, seed)` makes what a program holds before the call, `run(state)` is one pass through the public entry
points, `work(case)` the bytes and operations the pass cannot do without, `tolerance(case)` what another correct
implementation may differ by, and `exact(case, seed)` the pass's result in 64-bit torch without the library.
"""
from __future__ import annotations

import math

import torch

from sushi_amd import exl3

DEV = "cuda:0"

# Codebooks by the name a pack's config gives them.
DECODES = {
    "mcg": exl3.MCG,
    "mul1": exl3.MUL1,
    "3inst": exl3.INST3,
    "spec1": exl3.Decode(exl3.Codebook.spec1, exl3.Window(15), exl3.Table.spec1_w15),
}
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}


def _linear(name, rows, fin, fout, n, codebook, dtype, out):
    return dict(name=name, kind="linear", rows=rows, fin=fin, fout=fout, n=n, codebook=codebook, dtype=dtype, out=out)


def _moe(name, kind, rows, experts, hidden, inter, topk, n, codebook, dtype):
    return dict(name=name, kind=kind, rows=rows, experts=experts, hidden=hidden, inter=inter, topk=topk, n=n,
                codebook=codebook, dtype=dtype)


def listed():
    return [
        # one token through a square 4-bit projection: the smallest decode call, latency and launch count
        _linear("decode_1row_4096x4096_k4", 1, 4096, 4096, 64, "3inst", "f16", "f16"),
        # a 7-row speculative verify step through a 3-bit down projection, bf16 activations
        _linear("verify_7rows_14336x4096_k3", 7, 14336, 4096, 48, "mcg", "bf16", "bf16"),
        # one token through a 6-bit output head, f32 logits: the largest single weight of a decode step
        _linear("head_1row_5120x129280_k6", 1, 5120, 129280, 96, "spec1", "f16", "f32"),
        # 40 sequences decoding together through a square 4-bit projection
        _linear("batch_40rows_4096x4096_k4", 40, 4096, 4096, 64, "3inst", "f16", "f16"),
        # a short prompt through a 6-bit fused attention input projection
        _linear("prompt_200rows_2560x16384_k6", 200, 2560, 16384, 96, "mcg", "bf16", "bf16"),
        # a ragged prompt through a 4-bit down projection with f32 activations
        _linear("prompt_777rows_14336x4096_k4", 777, 14336, 4096, 64, "mcg", "f32", "f32"),
        # a 2048-token prefill chunk through a 3-bit up projection
        _linear("prefill_2048rows_4096x14336_k3", 2048, 4096, 14336, 48, "3inst", "f16", "f16"),
        # a routed layer and its shared expert, router included: one token, a decode batch, a prefill chunk
        _moe("moe_1token_e256_k2", "moe_shared", 1, 256, 2048, 768, 8, 32, "mcg", "f16"),
        _moe("moe_32tokens_e256_k2", "moe_shared", 32, 256, 2048, 768, 8, 32, "mcg", "f16"),
        _moe("moe_2048tokens_e256_k2", "moe_shared", 2048, 256, 2048, 768, 8, 32, "mcg", "bf16"),
        # a rate-grouped layer (a quarter of the experts at 1 bit, the rest at 2) at a verify width of 64 rows
        _moe("ragged_64rows_e256_k1_k2", "ragged", 64, 256, 4096, 2048, 8, 32, "spec1", "f16"),
        # the encoder's search over the tiles of a 1024 x 1024 weight at 2 bits and a 12-bit window
        dict(name="encode_4096tiles_k2_w12", kind="encode", tiles=4096, n=32, window=12, codebook="mcg"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the listed ones' ranges: rows 1 .. 2048, 1 to 8 bits, widths of 1280 to 14336 (the head's 129280
    at decode rows), MoE layers of 1 .. 2048 tokens, 64 to 4096 tiles to encode."""
    kind = rng.choice(["linear"] * 7 + ["head"] + ["moe_shared"] * 3 + ["ragged"] + ["encode"])
    if kind == "head":
        return dict(kind="linear", rows=rng.randint(1, 8), fin=128 * rng.randint(16, 40),
                    fout=128 * rng.randint(512, 1010), n=rng.choice([64, 96]), codebook=rng.choice(["spec1", "mcg"]),
                    dtype=rng.choice(["f16", "bf16"]), out=rng.choice(["f32", "f16"]))
    if kind == "linear":
        rows = _log(rng, 1, 2048)
        while True:
            fin, fout = (128 * _log(rng, 10, 112) for _ in range(2))
            if fin * fout <= 4096 * 14336:
                break
        dtype = rng.choice(["f16", "f16", "bf16", "f32"])
        return dict(kind="linear", rows=rows, fin=fin, fout=fout, n=rng.choice([16, 24, 32, 40, 48, 64, 80, 96, 128]),
                    codebook=rng.choice(["mcg", "mcg", "3inst", "spec1", "mul1"]), dtype=dtype, out=dtype)
    if kind == "moe_shared":
        return dict(kind=kind, rows=_log(rng, 1, 2048), experts=rng.choice([64, 128, 256]),
                    hidden=128 * rng.randint(8, 20), inter=128 * rng.randint(4, 8), topk=rng.choice([4, 6, 8]),
                    n=rng.choice([24, 32, 48, 64]), codebook=rng.choice(["mcg", "spec1"]),
                    dtype=rng.choice(["f16", "bf16"]))
    if kind == "ragged":
        return dict(kind=kind, rows=rng.randint(2, 64), experts=rng.choice([64, 128, 256]),
                    hidden=128 * rng.randint(16, 32), inter=128 * rng.randint(8, 16), topk=rng.choice([6, 8]), n=32,
                    codebook="spec1", dtype=rng.choice(["f16", "bf16"]))
    return dict(kind="encode", tiles=_log(rng, 64, 4096), n=rng.choice([32, 48]), window=12,
                codebook=rng.choice(["mcg", "mul1"]))


# ---------------------------------------------------------------------------------------------------------------
# Inputs


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _codes(g, *shape):
    return torch.randint(-32768, 32768, shape, dtype=torch.int16, device=DEV, generator=g)


def _scales(g, *shape):
    """Sign x magnitude, as a pack's suh / svh: +-1 times 0.5 .. 1.5."""
    sign = torch.randint(0, 2, shape, device=DEV, generator=g).float() * 2 - 1
    return (sign * (0.5 + torch.rand(shape, device=DEV, generator=g)))


def _proj(g, experts, fin, fout, n):
    """A bank whose projection keeps unit-variance inputs near unit scale."""
    return exl3.Proj(_codes(g, experts, fin // 16, fout // 16, n), _scales(g, experts, fin).half(),
                     (_scales(g, experts, fout) / math.sqrt(fin)).half())


def _bank(g, experts, hidden, inter, n):
    return exl3.Bank(_proj(g, experts, hidden, inter, n), _proj(g, experts, hidden, inter, n),
                     _proj(g, experts, inter, hidden, n))


def _x(g, rows, width, dtype):
    """Hidden states: N(0, 1) with one channel in 64 eight times as wide (activation outliers)."""
    x = torch.randn(rows, width, device=DEV, generator=g)
    wide = torch.rand(width, device=DEV, generator=g) < 1 / 64
    return (x * torch.where(wide, 8.0, 1.0)).to(DTYPES[dtype])


def _inputs(case, seed):
    g = _gen(seed)
    if case["kind"] == "linear":
        p = _proj(g, 1, case["fin"], case["fout"], case["n"])
        return dict(x=_x(g, case["rows"], case["fin"], case["dtype"]), p=p)
    if case["kind"] == "encode":
        return dict(tiles=torch.randn(case["tiles"], 256, device=DEV, generator=g))
    E, hidden, inter = case["experts"], case["hidden"], case["inter"]
    if case["kind"] == "ragged":
        banks = [_bank(g, E // 4, hidden, inter, 16), _bank(g, E - E // 4, hidden, inter, 32)]
    else:
        banks = [_bank(g, E, hidden, inter, case["n"]), _bank(g, 1, hidden, inter, case["n"])]
    return dict(x=_x(g, case["rows"], hidden, case["dtype"]), banks=banks,
                logits=torch.randn(case["rows"], E, device=DEV, generator=g))


def prepare(case, seed):
    s = _inputs(case, seed)
    s["case"] = dict(case)
    if case["kind"] == "ragged":
        s["ragged"] = exl3.Ragged.init(s.pop("banks"))
    return s


def run(s):
    c = s["case"]
    if c["kind"] == "encode":
        return exl3.encode_tiles(s["tiles"], c["n"], exl3.Decode(DECODES[c["codebook"]].codebook,
                                                                 exl3.Window(c["window"])))
    dec = DECODES[c["codebook"]]
    if c["kind"] == "linear":
        return exl3.linear(s["x"], s["p"], dec, DTYPES[c["out"]])
    inds, scores = exl3.moe_routing_chain(s["logits"], c["topk"])
    if c["kind"] == "ragged":
        y = exl3.moe_ragged(s["x"], s["ragged"], inds, scores, dec, verify_rows=True)
    else:
        y = exl3.moe_with_shared_bank(s["x"], s["banks"][0], s["banks"][1], inds, scores, dec)
    return y, inds, scores


# ---------------------------------------------------------------------------------------------------------------
# What a pass cannot do without


def work(case):
    size = {"f16": 2, "bf16": 2, "f32": 4}
    if case["kind"] == "linear":
        fin, fout, rows = case["fin"], case["fout"], case["rows"]
        by = fin * fout * case["n"] // 128 + 2 * (fin + fout) + rows * (fin * size[case["dtype"]] +
                                                                         fout * size[case["out"]])
        return {"bytes": by, "flops": 2 * rows * fin * fout}
    if case["kind"] == "encode":
        # every step scores all 2^window codewords against the predecessors (multiply-add and compare), twice round
        return {"bytes": case["tiles"] * (1024 + 2 * case["n"] + 8),
                "flops": case["tiles"] * 2 * 256 * (1 << case["window"]) * 3}
    E, hidden, inter, rows, topk = (case[k] for k in ("experts", "hidden", "inter", "rows", "topk"))
    hit = E * (1 - (1 - topk / E) ** rows)  # experts a uniform routing is expected to touch
    shared = 0 if case["kind"] == "ragged" else 1
    bits = 16 * (0.25 * 1 + 0.75 * 2) if case["kind"] == "ragged" else case["n"]
    per_expert = 3 * (hidden * inter * bits / 128 + 2 * (hidden + inter))
    return {"bytes": int((hit + shared) * per_expert + 2 * rows * hidden * 2 + rows * (4 * E + 8 * topk)),
            "flops": 6 * rows * (topk + shared) * hidden * inter}


def tolerance(case):
    if case["kind"] == "encode":
        return "exact"
    if case["kind"] == "linear":
        # one rounding of the output (f16 2.1e-4, bf16 1.7e-3 in the 2-norm against 64 bits); f32 outputs see only the
        # sums' order and the prepared inputs that round to the neighbouring f16 (up to 7e-6)
        return {"f16": {"rel": 8e-4, "max": 4e-3}, "bf16": {"rel": 7e-3, "max": 3e-2},
                "f32": {"rel": 3e-5, "max": 3e-4}}[case["out"]]
    # the routed and the shared sum are each rounded, then their sum (f16 3e-4, bf16 2.4e-3); expert ids are whole
    return {"f16": {"rel": 1.2e-3, "max": 8e-3, "differ": 1e-3}, "bf16": {"rel": 1e-2, "max": 5e-2, "differ": 1e-3}}[
        case["dtype"]]


# ---------------------------------------------------------------------------------------------------------------
# The same pass in 64 bits: weights decoded by the format's definition, then plain matrix products

# spec1-w15's (multiplier, mask) at the rates the cases use
_SPEC1 = {16: (0x84D1CF89, 0x8FE08947), 24: (0x84C1CF49, 0x8FE08B47), 32: (0x846C1FA7, 0x8FE08C80),
          40: (0x843C1FA7, 0x8FFE8E40), 48: (0x84181FB5, 0x8FE08F80), 64: (0x3FED4CEF, 0x8FF08FF0),
          80: (0x8000387B, 0x8FE08FF7), 96: (0xD0003751, 0x8FF98FFF), 128: (0x80003811, 0x8FFC8FFC)}


def _f16_bits(b):
    return torch.where(b >= 32768, b - 65536, b).to(torch.int16).view(torch.float16)


def _decode(cw, codebook, n):
    """Weights (f64) of masked codewords (int64), each rounded to f16 where the format rounds."""
    m32 = 0xFFFFFFFF
    if codebook == "mul1":
        p = (cw * 0x83DCD12D) & m32
        s = (p & 255) + ((p >> 8) & 255) + ((p >> 16) & 255) + (p >> 24)
        lo, hi = (_f16_bits(torch.tensor([b], device=DEV)).double() for b in (0x1EEE, 0xC931))
        return (_f16_bits(0x6400 + s).double() * lo + hi).half().double()
    if codebook == "spec1":
        mult, mask = _SPEC1[n]
        p = ((cw * mult) & m32) & mask
        scale = 4096.0
    else:
        p = (cw * 89226354 + 64248484) & m32 if codebook == "3inst" else (cw * 0xCBAC1FED) & m32
        p = (p & 0x8FFF8FFF) ^ 0x3B603B60
        scale = 1.0
    return (_f16_bits(p & 65535).double() + _f16_bits(p >> 16).double()).half().double() * scale


def _weights(trellis, codebook, n):
    """The inner weight [in, out] of one expert's trellis [in/16, out/16, n]."""
    it, ot = trellis.shape[0], trellis.shape[1]
    window = DECODES[codebook].window.bits
    hw = trellis.reshape(it * ot, n // 2, 2).long() & 65535
    words = hw[..., 0] | (hw[..., 1] << 16)
    t = torch.arange(256, device=DEV)
    last = (((t + 1) * n) // 16 - 1) % (16 * n)  # the codeword's last bit
    wl = last >> 5
    two = (words[:, (wl - 1) % (n // 2)] << 32) | words[:, wl]
    w = _decode((two >> (31 - (last & 31))) & ((1 << window) - 1), codebook, n)
    lane, i = t >> 3, t & 7
    q, col = lane & 3, (lane >> 2) + 8 * (i >= 4)
    row = 2 * q + (i & 1) + 8 * ((i >> 1) & 1)
    tile = torch.empty(it * ot, 256, dtype=torch.float64, device=DEV)
    tile[:, row * 16 + col] = w
    return tile.reshape(it, ot, 16, 16).transpose(1, 2).reshape(it * 16, ot * 16)


def _had128(v):
    h = torch.ones(1, 1, dtype=torch.float64, device=DEV)
    for _ in range(7):
        h = torch.cat([torch.cat([h, h], 1), torch.cat([h, -h], 1)])
    return (v.reshape(*v.shape[:-1], -1, 128) @ h).reshape(v.shape) / math.sqrt(128)


def _project(x, p, e, codebook):
    """x [rows, in] (f64) through expert e of a bank: f16 prepared input, f64 sums, no rounding of the result."""
    xp = _had128(x.half().double() * p.suh[e].double()).half().double()
    it, ot = p.trellis.shape[1], p.trellis.shape[2]
    step = max(8, (1 << 17) // it // 8 * 8)  # output tiles decoded at a time
    inner = torch.cat([xp @ _weights(p.trellis[e, :, o:o + step], codebook, p.n) for o in range(0, ot, step)], 1)
    return _had128(inner) * p.svh[e].double()


def _swiglu(x, bank, e, codebook):
    gate, up = _project(x, bank.gate, e, codebook), _project(x, bank.up, e, codebook)
    mid = gate / (1 + torch.exp(-gate)) * up
    p = bank.down  # the down input is prepared from the f64 product
    xp = _had128(mid * p.suh[e].double()).half().double()
    return _had128(xp @ _weights(p.trellis[e], codebook, p.n)) * p.svh[e].double()


def exact(case, seed):
    if case["kind"] == "encode":
        return None  # codes are whole numbers, held to equality
    s = _inputs(case, seed)
    x, cb = s["x"].double(), case["codebook"]
    if case["kind"] == "linear":
        return _project(x, s["p"], 0, cb)
    top, inds = torch.topk(s["logits"].double(), case["topk"], dim=-1)
    scores = torch.softmax(top, -1)
    y = torch.zeros_like(x)
    first = 0
    for bank in s["banks"] if case["kind"] == "ragged" else s["banks"][:1]:
        for e in range(bank.gate.experts):
            tok, slot = torch.nonzero(inds == first + e, as_tuple=True)
            if tok.numel():
                y[tok] += scores[tok, slot, None] * _swiglu(x[tok], bank, e, cb)
        first += bank.gate.experts
    if case["kind"] != "ragged":
        y += _swiglu(x, s["banks"][1], 0, cb)
    return y, inds.int(), scores
