"""The work the library is measured on: what an engine has it do in one pass over attention layers.

A case is one call pattern of a serving engine at the public interface (``HipKvCache``):

``attend``   the attention of one step over ``layers`` layers, Q given.
``layer``    a layer's whole share of the library: QK-norm, RoPE and the K/V store of the new rows
             (``qk_rope_store``), then their attention on the Q it wrote.
``park``     a sequence restored from a snapshot held in device memory and parked again
             (``read_seq``, ``write_seq``).

The batch of a step is ``rows`` sequences that each append ``row_new`` tokens (1: decode; 2 and more:
a run of drafted tokens being verified), with contexts spread over ``ctx_lo .. ctx_hi`` (their
logarithm), then ``chunks`` sequences that append ``chunk_lo .. chunk_hi`` prompt tokens after
``prior`` cached ones. ``lens`` seeds these lengths, so they belong to the case; everything else comes
from the seed given to ``prepare``. ``q_exact``: Q already rounded to the pages' 16-bit type, as
activations held in that type are; without it Q has all its f32 bits, as ``qk_rope_store`` writes it.
"""

from __future__ import annotations

import math
import random

import torch

from llmario_amd.kv import HipKvCache, Layer, Segments

_BASE = {"kind": "attend", "kv": "f16", "heads": 32, "kv_heads": 8, "hd": 128, "hdv": 128, "layers": 1,
         "rows": 0, "row_new": 1, "ctx_lo": 1, "ctx_hi": 1, "chunks": 0, "chunk_lo": 0, "chunk_hi": 0, "prior": 0,
         "window": 0, "q_exact": False, "neox": True, "qk_norm": True, "block": 16, "lens": 0}


def _case(name, **kw):
    return {"name": name, **_BASE, **kw}


def listed():
    return [
        # one short chat turn on f32 pages, one token: the smallest call, all launch latency
        _case("decode_one_f32", kv="f32", heads=8, kv_heads=8, hd=64, hdv=64, rows=1, ctx_lo=256, ctx_hi=256),
        # one user's decode step through four layers: store the token, attend, the next layer
        _case("layers_one_f16", kind="layer", layers=4, rows=1, ctx_lo=2987, ctx_hi=2987, block=32),
        # a full decode batch of mixed context lengths, three layers of a step, pages from HBM
        _case("decode_batch_f16", layers=3, rows=32, ctx_lo=512, ctx_hi=4096, lens=2),
        # few very long contexts on quantised pages: split over the whole device
        _case("decode_long_q8", kv="q8_0", heads=64, rows=8, ctx_lo=32768, ctx_hi=32768, q_exact=True),
        # speculative decoding: every sequence verifies a run of four drafted tokens
        _case("verify_batch_bf16", kv="bf16", rows=24, row_new=4, ctx_lo=512, ctx_hi=4096, lens=5),
        # four whole prompts at once, activations held in bf16
        _case("prefill_bf16", kv="bf16", chunks=4, chunk_lo=2048, chunk_hi=2048, q_exact=True),
        # ragged prompts on quantised pages, the whole layer (norm, RoPE, store, attention)
        _case("layer_prompts_q8", kind="layer", kv="q8_0", chunks=3, chunk_lo=401, chunk_hi=2047, lens=7),
        # continuous batching: decode rows beside two prompt chunks in one call
        _case("mixed_f16", heads=40, rows=16, ctx_lo=1024, ctx_hi=8192, chunks=2, chunk_lo=512, chunk_hi=512,
              prior=4096, lens=5),
        # wide heads with a sliding window: prompts beside decode rows
        _case("window_wide_bf16", kv="bf16", heads=16, kv_heads=4, hd=256, hdv=256, rows=4, ctx_lo=700, ctx_hi=3000,
              chunks=2, chunk_lo=600, chunk_hi=1100, window=1024, lens=9),
        # a prompt on f32 pages (full-precision cache)
        _case("prompt_f32", kv="f32", heads=16, kv_heads=4, hd=64, hdv=64, chunks=2, chunk_lo=250, chunk_hi=700,
              lens=10),
        # a head width off the matrix instructions' multiples, every head its own K/V: decode rows
        # and a prompt chunk
        _case("step_hd80_f16", heads=32, kv_heads=32, hd=80, hdv=80, rows=8, ctx_lo=200, ctx_hi=3000, chunks=1,
              chunk_lo=120, chunk_hi=120, prior=300, lens=11),
        # a parked conversation brought back into the cache and parked again, eight layers
        _case("park_q8", kind="park", kv="q8_0", layers=8, rows=1, ctx_lo=9999, ctx_hi=9999),
    ]


# (heads, kv_heads, hd, hdv) by use: grouped heads of the usual widths, every head its own K/V, wide
# heads, a value width of its own, a width off the matrix instructions' multiples
_GEOMS = [(32, 8, 128, 128), (40, 8, 128, 128), (64, 8, 128, 128), (16, 4, 64, 64), (8, 8, 64, 64), (32, 32, 64, 64),
          (16, 4, 256, 256), (32, 8, 192, 128), (12, 4, 96, 96), (32, 32, 80, 80)]


def _log(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))))


def _bounds(c):
    """The listed work of the same kind of path that a drawn case stays within: (bytes, flops)."""
    if c["kv"] == "f32" or c["hd"] % 32 or c["hd"] != c["hdv"] or c["hd"] > 128:
        return 250e6, 6e9
    return 600e6, 90e9


def draw(rng):
    while True:
        c = dict(_BASE)
        kind = rng.choice(["decode", "decode", "verify", "prompt", "prompt", "mixed", "layer", "layer", "park"])
        c["kv"] = rng.choice(["f16", "bf16", "q8_0", "f16", "bf16", "q8_0", "f32"])
        c["heads"], c["kv_heads"], c["hd"], c["hdv"] = rng.choice(_GEOMS)
        if c["kv"] == "q8_0" and (c["hd"] % 32 or c["hdv"] % 32):
            c["kv"] = "f16"
        c["block"] = rng.choice([16, 32])
        c["lens"] = rng.randrange(1 << 30)
        c["q_exact"] = rng.random() < 0.3
        if kind in ("decode", "verify", "mixed"):
            c["rows"] = _log(rng, 1, 48)
            c["ctx_lo"] = _log(rng, 16, 8192)
            c["ctx_hi"] = min(32768, c["ctx_lo"] * rng.choice([1, 2, 4, 8]))
            c["row_new"] = rng.randint(2, 7) if kind == "verify" else 1
            c["window"] = rng.choice([0, 0, 0, 1024, 4096])
        if kind in ("prompt", "mixed", "layer"):
            c["chunks"] = rng.randint(1, 4)
            c["chunk_lo"] = _log(rng, 8, 2048)
            c["chunk_hi"] = min(2048, c["chunk_lo"] * rng.choice([1, 1, 2, 4]))
            c["prior"] = rng.choice([0, 0, _log(rng, 16, 8192)])
            c["window"] = rng.choice([0, 0, 0, 1024, 4096])
        if kind == "layer":
            c["kind"] = "layer"
            c["hdv"] = c["hd"]   # the fused store takes one width
            c["neox"], c["qk_norm"] = rng.random() < 0.7, rng.random() < 0.6
            if rng.random() < 0.5:   # decode rows alone, through several layers
                c["chunks"] = c["chunk_lo"] = c["chunk_hi"] = c["prior"] = 0
                c["rows"], c["layers"] = _log(rng, 1, 48), rng.randint(1, 4)
                c["ctx_lo"] = _log(rng, 16, 4096)
                c["ctx_hi"] = min(8192, c["ctx_lo"] * rng.choice([1, 4]))
        if kind == "park":
            c.update(kind="park", rows=1, layers=rng.randint(1, 8), q_exact=False, ctx_lo=_log(rng, 40, 12000))
            c["ctx_hi"] = c["ctx_lo"]
        w, (b, f) = work(c), _bounds(c)
        if w["bytes"] <= b and w["flops"] <= f:
            return c


# ---- the batch of a case --------------------------------------------------------------------------


def _batch(c):
    """[(cached tokens, new tokens)] per sequence."""
    rng = random.Random(c["lens"])
    out = [(max(_log(rng, c["ctx_lo"], c["ctx_hi"]) - c["row_new"], 0), c["row_new"]) for _ in range(c["rows"])]
    return out + [(c["prior"], _log(rng, c["chunk_lo"], c["chunk_hi"])) for _ in range(c["chunks"])]


def _elem_bytes(c):
    return {"f32": 4.0, "f16": 2.0, "bf16": 2.0, "q8_0": 34.0 / 32.0}[c["kv"]]


def work(c):
    kv_row = c["kv_heads"] * (c["hd"] + c["hdv"])
    n_bytes = flops = 0.0
    for prior, new in _batch(c):
        if c["kind"] == "park":   # each byte of the snapshot in and out of the pages, both ways
            tokens = -(-(prior + new) // c["block"]) * c["block"]
            n_bytes += 4 * tokens * kv_row * _elem_bytes(c)
            continue
        first = max(0, prior + 1 - c["window"]) if c["window"] else 0
        keys = prior + new - first
        pairs = sum(min(p + 1, c["window"] or p + 1) for p in range(prior, prior + new))
        n_bytes += keys * kv_row * _elem_bytes(c) + new * c["heads"] * (c["hd"] + c["hdv"]) * 4.0
        if c["kind"] == "layer":   # Q read once more before it is rotated, the new K/V rows read
            n_bytes += new * (c["heads"] * c["hd"] + kv_row) * 4.0
        flops += 2.0 * (c["hd"] + c["hdv"]) * pairs * c["heads"]
    return {"bytes": c["layers"] * n_bytes, "flops": c["layers"] * flops}


# ---- inputs, made from (case, seed) alone ---------------------------------------------------------


def _rand(c, seed, tag, shape):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + tag * 7919 + 1) & 0x7FFFFFFFFFFF)
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)


def _to_page(x, kv):
    """The f32 values a row has once it is held in the pages' type."""
    if kv == "f16":
        return x.half().float()
    if kv == "bf16":
        return x.bfloat16().float()
    if kv == "q8_0":
        b = x.float().reshape(-1, 32)
        d = b.abs().amax(dim=1, keepdim=True) / 127.0
        codes = torch.round(b * torch.where(d != 0, 1.0 / d, torch.zeros_like(d)))
        return (codes * d.half().float()).reshape(x.shape)
    return x.float()


def _seq_kv(c, seed, layer, s, tokens):
    """K and V of a sequence's cached positions, representable in the pages' type."""
    t = 2 * (layer * 4096 + s)
    return (_to_page(_rand(c, seed, t, (tokens, c["kv_heads"] * c["hd"])), c["kv"]),
            _to_page(_rand(c, seed, t + 1, (tokens, c["kv_heads"] * c["hdv"])), c["kv"]))


def _step_in(c, seed, layer, n_rows):
    """What the projections hand over for the step's rows: q, k, v."""
    t = 100000 + 4 * layer
    return (_rand(c, seed, t, (n_rows, c["heads"], c["hd"])), _rand(c, seed, t + 1, (n_rows, c["kv_heads"], c["hd"])),
            _rand(c, seed, t + 2, (n_rows, c["kv_heads"], c["hdv"])))


def _norms(c, seed, layer):
    if not c["qk_norm"]:
        return None, None
    w = 1.0 + 0.1 * _rand(c, seed, 200000 + layer, (2, c["hd"]))
    return w[0].contiguous(), w[1].contiguous()


def _scale(c):
    return 1.0 / math.sqrt(c["hd"])


_THETA, _EPS = 10000.0, 1e-6


# ---- the measured passes --------------------------------------------------------------------------


def prepare(case, seed):
    c, batch = case, _batch(case)
    n_rows, n_seqs = sum(n for _, n in batch), len(batch)
    totals = [p + n for p, n in batch]
    if c["kind"] == "park":
        n_seqs, totals = 2, totals + totals
    hc = HipKvCache([Layer(c["heads"], c["kv_heads"], c["hd"], c["hdv"])] * c["layers"], max_ctx=max(totals),
                    n_seqs=n_seqs, kv_type=c["kv"], block_tokens=c["block"], pool_tokens=sum(totals) + c["block"] * n_seqs)
    # block ids as a long-running cache has them: scattered over the pool
    order = list(range(hc.layout()["pool_blocks"]))
    random.Random(seed).shuffle(order)
    at = 0
    for s, (prior, new) in enumerate(batch):
        need = -(-(prior + new) // c["block"])
        hc.adopt_blocks(s, order[at:at + need])
        at += need
        held = prior if c["kind"] == "layer" else prior + new
        for layer in range(c["layers"] if held else 0):
            k, v = _seq_kv(c, seed, layer, s, held)
            hc.store(layer, [(s, 0, held, 0)], k, v)
        hc.set_len(s, prior + new if c["kind"] == "park" else prior)
    st = {"case": c, "hc": hc, "scale": _scale(c)}
    if c["kind"] == "park":
        length = totals[0]
        src = hc.write_seq(0)
        hc.clear(0)
        st.update(length=length, src=src, dst=torch.empty_like(src))
    else:
        start, segs = 0, []
        for s, (prior, new) in enumerate(batch):
            segs.append((s, start, new, prior))
            start += new
        st["segs"] = Segments(segs)
        st["out"] = [torch.empty(n_rows, c["heads"], c["hdv"], device="cuda") for _ in range(c["layers"])]
        ins = [_step_in(c, seed, layer, n_rows) for layer in range(c["layers"])]
        st["q"] = [_q_held(c, q) for q, _, _ in ins]
        if c["kind"] == "layer":
            st["k"], st["v"] = [i[1] for i in ins], [i[2] for i in ins]
            st["norms"] = [_norms(c, seed, layer) for layer in range(c["layers"])]
            st["q_out"] = [torch.empty_like(q) for q in st["q"]]
    torch.cuda.synchronize()
    return st


def _q_held(c, q):
    """Q as the caller holds it: all f32 bits, or rounded to the pages' 16-bit type."""
    if c["q_exact"] and c["kind"] == "attend" and c["kv"] != "f32":
        return _to_page(q, "bf16" if c["kv"] == "bf16" else "f16")
    return q


def run(st):
    c, hc = st["case"], st["hc"]
    if c["kind"] == "park":
        hc.read_seq(0, st["length"], st["src"])
        return hc.write_seq(0, st["dst"])
    if c["kind"] == "attend":
        for layer in range(c["layers"]):
            hc.attend(layer, st["segs"], st["q"][layer], st["out"][layer], st["scale"], c["window"])
        return st["out"]
    for layer in range(c["layers"]):
        q_norm, k_norm = st["norms"][layer]
        hc.qk_rope_store(layer, st["segs"], st["q"][layer], st["k"][layer], st["v"][layer], st["q_out"][layer],
                         theta=_THETA, neox=c["neox"], q_norm=q_norm, k_norm=k_norm, eps=_EPS)
        hc.attend(layer, st["segs"], st["q_out"][layer], st["out"][layer], st["scale"], c["window"])
    return st["q_out"] + st["out"]


# ---- the same in 64 bits --------------------------------------------------------------------------


def _norm_rope64(c, x, w, pos):
    """RMS norm and rotation of x [rows, heads, hd] at positions pos, in 64 bits. The angles are part
    of the path's definition: position times frequency, both in f32."""
    x = x.double()
    if w is not None:
        x = x / torch.sqrt((x * x).mean(dim=-1, keepdim=True) + _EPS) * w.double()
    half = c["hd"] // 2
    expo = -(2.0 * torch.arange(half, dtype=torch.float32)) / float(c["hd"])
    freq = (_THETA ** expo.double()).float().cuda()
    ang = (pos.float()[:, None] * freq[None, :]).double()[:, None, :]
    cos, sin = torch.cos(ang), torch.sin(ang)
    out = torch.empty_like(x)
    a, b = (slice(0, half), slice(half, None)) if c["neox"] else (slice(0, None, 2), slice(1, None, 2))
    out[..., a] = x[..., a] * cos - x[..., b] * sin
    out[..., b] = x[..., a] * sin + x[..., b] * cos
    return out


def _attend64(c, q, k, v, prior):
    """q [new, heads, hd] over k, v [prior + new, kv_heads * width], causal and windowed."""
    new, group = q.shape[0], c["heads"] // c["kv_heads"]
    first = max(0, prior + 1 - c["window"]) if c["window"] else 0
    k = k[first:].double().reshape(-1, c["kv_heads"], c["hd"])
    v = v[first:].double().reshape(-1, c["kv_heads"], c["hdv"])
    key = torch.arange(first, first + k.shape[0], device="cuda")
    out = torch.empty(new, c["heads"], c["hdv"], dtype=torch.float64, device="cuda")
    step = max(1, int(1.5e8) // (group * k.shape[0]))
    for h in range(c["kv_heads"]):
        kt, vh = k[:, h].t().contiguous(), v[:, h].contiguous()
        for t in range(0, new, step):
            qh = q[t:t + step, h * group:(h + 1) * group].reshape(-1, c["hd"]).contiguous()
            pos = prior + t + torch.arange(qh.shape[0], device="cuda") // group
            s = torch.mm(qh, kt) * _scale(c)
            hide = key[None, :] > pos[:, None]
            if c["window"]:
                hide |= key[None, :] <= pos[:, None] - c["window"]
            p = torch.softmax(s.masked_fill_(hide, -math.inf), dim=1)
            out[t:t + step, h * group:(h + 1) * group] = torch.mm(p, vh).reshape(-1, group, c["hdv"])
    return out


def exact(case, seed):
    c, batch = case, _batch(case)
    if c["kind"] == "park":
        return None   # bytes: the start's are the standard
    n_rows = sum(n for _, n in batch)
    pos = torch.cat([torch.arange(p, p + n) for p, n in batch]).cuda()
    qs, outs = [], []
    for layer in range(c["layers"]):
        q, k, v = _step_in(c, seed, layer, n_rows)
        if c["kind"] == "layer":
            wq, wk = _norms(c, seed, layer)
            q = _norm_rope64(c, q, wq, pos)
            k = _to_page(_norm_rope64(c, k, wk, pos).float(), c["kv"]).reshape(n_rows, -1)
            v = _to_page(v, c["kv"]).reshape(n_rows, -1)
            qs.append(q)
        else:
            q = _q_held(c, q).double()
        out, start = [], 0
        for s, (prior, new) in enumerate(batch):
            held = prior if c["kind"] == "layer" else prior + new
            ks, vs = _seq_kv(c, seed, layer, s, held)
            if c["kind"] == "layer":
                ks, vs = torch.cat([ks, k[start:start + new]]), torch.cat([vs, v[start:start + new]])
            out.append(_attend64(c, q[start:start + new], ks, vs, prior))
            start += new
        outs.append(torch.cat(out))
    return qs + outs


# Four times the largest error against exact() seen over the listed cases and 160 drawn ones, by page
# type: (rel, max). The weights and Q keep what two parts of the pages' 16-bit type hold.
_ATTEND_TOL = {"f32": (3e-6, 4e-5), "f16": (3e-6, 4e-5), "bf16": (1.2e-5, 2e-4), "q8_0": (1.2e-5, 2.5e-4)}
# A layer's own K rows are rounded to the page type after a norm and a rotation in 32 bits: a value
# next to a rounding boundary lands on either side, one key among few for the first prompt tokens.
_LAYER_TOL = {"f32": (3e-6, 4e-5), "f16": (3e-5, 3e-3), "bf16": (1.2e-4, 1.2e-2), "q8_0": (1.3e-4, 3e-2)}


def tolerance(case):
    if case["kind"] == "park":
        return "exact"
    rel, most = (_LAYER_TOL if case["kind"] == "layer" else _ATTEND_TOL)[case["kv"]]
    return {"rel": rel, "max": most}
