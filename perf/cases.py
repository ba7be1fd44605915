"""The calls that a program built on this framework makes in earnest, with their sizes.

``listed()`` holds the named cases, ``draw(rng)`` gives more of the same ranges. A case says which
part of the path runs (``kind``) and how large it is; ``prepare`` makes what the program has in hand
before the call (weights, caches, tables, inputs), ``run`` is one pass through the public entry
points, ``work`` the bytes and operations that such a pass cannot do without, and ``exact`` the same
pass in 64 bits with plain torch.

The two decoders are those of the 0.6B (hidden 1024, FFN 3072) and 1.7B (2048, 6144) models: 28
layers, 16 query and 8 key/value heads of 128, vocabulary 151936, INT8 weights with a scale per row.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from qwenasr_amd import kernels as K
from qwenasr_amd.decoder import DecoderInt8, DecoderInt8Batched

NQ, NK, HD = 16, 8, 128
QD, KV = NQ * HD, NK * HD
VOCAB = 151936
EPS, THETA = 1e-6, 1e6
F = 4  # bytes of a float
F32, F64, I8 = torch.float32, torch.float64, torch.int8


def listed() -> list[dict]:
    return [
        # the per-token elementwise ops of one decoder layer, one token: the smallest calls there are
        {"name": "layer_ops_0.6b_1_token", "kind": "ops", "hidden": 1024, "tokens": 1},
        # one generated token of a 30 s utterance, whole 0.6B decoder: logits
        {"name": "decode_0.6b_whole", "kind": "decode", "hidden": 1024, "layers": 28, "pos": 403},
        # one generated token late in a long recording, four layers of the 1.7B decoder and its lm_head
        {"name": "decode_1.7b_4_layers", "kind": "decode", "hidden": 2048, "layers": 4, "pos": 1801},
        # the prompt and audio rows of an utterance through the whole 0.6B decoder
        {"name": "prefill_0.6b_whole", "kind": "prefill", "hidden": 1024, "layers": 28, "tokens": 512, "start": 0},
        # a long recording's rows through a layer of the 1.7B decoder
        {"name": "prefill_1.7b_long", "kind": "prefill", "hidden": 2048, "layers": 1, "tokens": 1473, "start": 0},
        # streaming: the next few seconds of audio after what is cached already, two layers
        {"name": "prefill_0.6b_chunk", "kind": "prefill", "hidden": 1024, "layers": 2, "tokens": 77, "start": 610},
        # a full server: 256 streams with their own positions, int8 activations, two layers and the lm_head
        {"name": "streams_1.7b_w8a8_256", "kind": "streams", "hidden": 2048, "layers": 2, "batch": 256,
         "rows": 2048, "w8a8": True},
        # a half-full server with the reference's fp32 activations, two layers and the lm_head
        {"name": "streams_1.7b_w8a32_64", "kind": "streams", "hidden": 2048, "layers": 2, "batch": 64,
         "rows": 1024, "w8a8": False},
        # a few streams on the small model, four layers and the lm_head
        {"name": "streams_0.6b_w8a32_11", "kind": "streams", "hidden": 1024, "layers": 4, "batch": 11,
         "rows": 768, "w8a8": False},
        # the audio encoder's row ops on 3000 frames
        {"name": "encoder_rows_3000", "kind": "encoder", "rows": 3000, "dim": 896, "positions": 104},
        # logits and greedy token of one stream
        {"name": "lm_head_0.6b", "kind": "lm_head", "hidden": 1024, "rows": 1},
        # the int8 gate/up half of a 1.7B layer for 256 streams: norm + quantize, head norms + RoPE, GEMM + SwiGLU
        {"name": "w8a8_chain_1.7b_256", "kind": "w8a8_chain", "hidden": 2048, "batch": 256},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng) -> dict:
    kind = rng.choice(["ops", "decode", "prefill", "prefill", "streams", "streams", "encoder", "lm_head", "w8a8_chain"])
    hidden = rng.choice([1024, 2048])
    if kind == "ops":
        return {"kind": kind, "hidden": hidden, "tokens": _log_int(rng, 1, 2048)}
    if kind == "decode":
        return {"kind": kind, "hidden": hidden, "layers": rng.randint(1, 6), "pos": _log_int(rng, 20, 2047)}
    if kind == "prefill":
        return {"kind": kind, "hidden": hidden, "layers": rng.randint(1, 2), "tokens": _log_int(rng, 8, 1500),
                "start": rng.choice([0, 0, rng.randint(1, 500)])}
    if kind == "streams":
        return {"kind": kind, "hidden": hidden, "layers": rng.randint(1, 2), "batch": _log_int(rng, 2, 256),
                "rows": rng.randint(200, 1536), "w8a8": rng.choice([True, False])}
    if kind == "encoder":
        return {"kind": kind, "rows": _log_int(rng, 50, 3000), "dim": rng.choice([896, 1024]),
                "positions": rng.randint(13, 104)}
    if kind == "lm_head":
        return {"kind": kind, "hidden": hidden, "rows": rng.choice([1, 1, _log_int(rng, 2, 32)])}
    return {"kind": kind, "hidden": hidden, "batch": _log_int(rng, 2, 256)}


# ---------------------------------------------------------------------------
# What the program has in hand
# ---------------------------------------------------------------------------
class _Maker:
    """Seeded tensors on the GPU."""

    def __init__(self, seed: int):
        self.dev = torch.device("cuda")
        self.gen = torch.Generator(device=self.dev)
        self.gen.manual_seed(seed)

    def randn(self, n: int, scale: float = 1.0, mean: float = 0.0) -> torch.Tensor:
        t = torch.empty(n, dtype=F32, device=self.dev).normal_(generator=self.gen)
        return t.mul_(scale).add_(mean)

    def weight(self, out_dim: int, in_dim: int) -> K.QuantWeight:
        """What the quantizer gives for normal rows: int8 with the row's largest value near 127, and a
        scale that makes the rows' values those of a trained projection."""
        q = torch.empty(out_dim * in_dim, dtype=torch.float16, device=self.dev).normal_(generator=self.gen)
        q = q.mul_(36.0).round_().clamp_(-127, 127).to(I8)
        return K.QuantWeight(q, self.randn(out_dim, 0.1, 1.0).abs_().mul_(0.7 / 36.0 / math.sqrt(in_dim)),
                             out_dim, in_dim)

    def gain(self, n: int) -> torch.Tensor:
        return self.randn(n, 0.1, 1.0)

    def ints(self, lo: int, hi: int, n: int) -> torch.Tensor:
        return torch.randint(lo, hi, (n,), generator=self.gen, device=self.dev, dtype=torch.int32)


def _decoder_weights(m: _Maker, hidden: int, layers: int, lm_head: bool) -> dict:
    inter = 3 * hidden
    made = [{"wq": m.weight(QD, hidden), "wk": m.weight(KV, hidden), "wv": m.weight(KV, hidden),
             "wo": m.weight(hidden, QD), "gate_up": m.weight(2 * inter, hidden), "down": m.weight(hidden, inter),
             "q_norm": m.gain(HD), "k_norm": m.gain(HD), "input_norm": m.gain(hidden),
             "post_attn_norm": m.gain(hidden)} for _ in range(layers)]
    lm = m.weight(VOCAB if lm_head else 1024, hidden)  # a prefill does not reach the lm_head
    return {"layers": made, "norm": m.gain(hidden), "lm_head": lm, "tok_embeddings": lm}


def prepare(case: dict, seed: int) -> dict:
    m = _Maker(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "ops":
        h, t = case["hidden"], case["tokens"]
        s.update(x=m.randn(t * h), delta=m.randn(t * h, 0.3), w=m.gain(h), out=torch.empty(t * h, device=m.dev),
                 q=m.randn(t * QD), k=m.randn(t * KV), qw=m.gain(HD), kw=m.gain(HD), rope=K.RopeCache(m.dev),
                 pos=m.ints(0, 2048, t), gate_up=m.randn(t * 6 * h), act=torch.empty(t * 3 * h, device=m.dev))
        s["rope"].ensure(2048, HD, THETA)
    elif kind in ("decode", "prefill"):
        h, layers = case["hidden"], case["layers"]
        w = _decoder_weights(m, h, layers, kind == "decode")
        start = case["pos"] if kind == "decode" else case["start"]
        t = 1 if kind == "decode" else case["tokens"]
        d = DecoderInt8(w, h, 3 * h, layers, NQ, NK, HD, EPS, THETA, max_seq=start + t, device=m.dev)
        for l in range(layers):  # the rows of what came before
            d.kv.k_layer_block(l)[:start * KV].copy_(m.randn(start * KV))
            d.kv.v_layer_block(l)[:start * KV].copy_(m.randn(start * KV, 0.7))
        d.kv.len = start
        s.update(w=w, d=d, start=start)
        if kind == "decode":
            s.update(token=m.ints(0, VOCAB, 1), embed=torch.empty(h, device=m.dev))
            d.prepare()
        else:
            s["embeds"] = m.randn(t * h, 0.5)
            d.prepare_prefill(None, t)
    elif kind == "streams":
        h, layers, b, rows = case["hidden"], case["layers"], case["batch"], case["rows"]
        w = _decoder_weights(m, h, layers, True)
        d = DecoderInt8Batched(w, h, 3 * h, layers, b, rows, NQ, NK, HD, EPS, THETA, device=m.dev, w8a8=case["w8a8"])
        for l in range(layers):
            d.k[l].normal_(generator=m.gen)
            d.v[l].normal_(generator=m.gen).mul_(0.7)
        d.positions.copy_(m.ints(0, rows, b))
        s.update(w=w, d=d, tokens=m.ints(0, VOCAB, b), embeds=torch.empty(b * h, device=m.dev))
    elif kind == "encoder":
        r, dim, n = case["rows"], case["dim"], case["positions"]
        pe = torch.empty(n * dim, device=m.dev)
        K.sinusoidal_pe(pe, n, dim)
        s.update(x=m.randn(r * dim), pe=pe, out=torch.empty(r * dim, device=m.dev), w=m.gain(dim),
                 b=m.randn(dim, 0.1), ffn=m.randn(4 * r * dim), act=torch.empty(4 * r * dim, device=m.dev),
                 delta=m.randn(r * dim, 0.3), w2=m.gain(dim), b2=m.randn(dim, 0.1),
                 out2=torch.empty(r * dim, device=m.dev))
    elif kind == "lm_head":
        h, r = case["hidden"], case["rows"]
        s.update(w=m.weight(VOCAB, h), x=m.randn(r * h), idx=torch.empty(r, dtype=torch.int32, device=m.dev),
                 logits=torch.empty(r * VOCAB, device=m.dev), ws=K.lm_head_workspace(VOCAB, m.dev))
    else:  # w8a8_chain
        h, b = case["hidden"], case["batch"]
        packed = K.pack_w8a8_tiles(m.weight(6 * h, h))
        s.update(x=m.randn(b * h), delta=m.randn(b * h, 0.3), w=m.gain(h),
                 xq=torch.empty(b * h, dtype=I8, device=m.dev), xs=torch.empty(b, device=m.dev),
                 q=m.randn(b * QD), k=m.randn(b * KV), qw=m.gain(HD), kw=m.gain(HD), rope=K.RopeCache(m.dev),
                 pos=m.ints(0, 2048, b), packed=packed, out=torch.empty(b * 3 * h, device=m.dev))
        s["rope"].ensure(2048, HD, THETA)
    return s


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------
def run(s: dict):
    c = s["case"]
    kind = c["kind"]
    if kind == "ops":
        h, t = c["hidden"], c["tokens"]
        K.add_rms_norm(s["x"], s["delta"], s["w"], s["out"], t, h, EPS)
        K.head_rms_norm_rope(s["q"], s["k"], s["qw"], s["kw"], s["rope"].cos, s["rope"].sin, s["pos"], t, NQ, NK, HD,
                             EPS)
        K.swiglu_multiply(s["act"], s["gate_up"], t, 3 * h)
        return {"x": s["x"], "out": s["out"], "q": s["q"], "k": s["k"], "act": s["act"]}
    if kind == "decode":
        d = s["d"]
        d.kv.len = s["start"]  # the same token again: the cache holds rows 0..start-1
        K.embed_gather_i8(s["embed"], s["w"]["tok_embeddings"], s["token"], 1, c["hidden"])
        d.prepare()
        d.decode(s["embed"])
        d.finish()
        return {"logits": d.logits, "x_norm": d.x_norm, "k": d.kv.k, "v": d.kv.v}
    if kind == "prefill":
        d, t = s["d"], c["tokens"]
        d.kv.len = s["start"]
        d.prepare_prefill(None, t)
        d.prefill(s["embeds"], t)
        return {"x": d.px[:t * c["hidden"]], "k": d.kv.k, "v": d.kv.v}
    if kind == "streams":
        d = s["d"]
        K.embed_gather_i8(s["embeds"], s["w"]["tok_embeddings"], s["tokens"], c["batch"], c["hidden"])
        d.decode(s["embeds"])
        return {"logits": d.logits, "x_norm": d.x_norm, "k": d.k, "v": d.v}
    if kind == "encoder":
        r, dim, n = c["rows"], c["dim"], c["positions"]
        K.pe_add_layer_norm(s["x"], s["pe"], s["out"], s["w"], s["b"], r, dim, n, 1e-5)
        s["act"].copy_(s["ffn"])  # the FFN's first projection writes its rows anew for each pass
        K.gelu_erf(s["act"], 4 * r * dim)
        K.add_layer_norm(s["x"], s["delta"], s["w2"], s["b2"], s["out2"], r, dim, 1e-5)
        return {"x": s["x"], "out": s["out"], "act": s["act"], "out2": s["out2"]}
    if kind == "lm_head":
        K.lm_head_int8_argmax(s["idx"], s["logits"], s["x"], s["w"], c["rows"], c["hidden"], VOCAB, s["ws"])
        return {"idx": s["idx"], "logits": s["logits"]}
    h, b = c["hidden"], c["batch"]
    K.add_rms_norm_quant(s["x"], s["delta"], s["w"], None, s["xq"], s["xs"], b, h, EPS)
    K.head_rms_norm_rope(s["q"], s["k"], s["qw"], s["kw"], s["rope"].cos, s["rope"].sin, s["pos"], b, NQ, NK, HD, EPS)
    K.gate_up_swiglu_w8a8_packed(s["out"], s["packed"], s["xq"], s["xs"], b, h, 3 * h)
    return {"x": s["x"], "xq": s["xq"], "xs": s["xs"], "q": s["q"], "k": s["k"], "out": s["out"]}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "ops":
        h, t = case["hidden"], case["tokens"]
        return {"bytes": F * (t * (4 * h + 2 * (QD + KV) + 9 * h + 2 * HD + 1) + h + 2 * HD), "flops": 60 * t * h}
    if kind in ("decode", "prefill", "streams"):
        h, layers = case["hidden"], case["layers"]
        inter = 3 * h
        weights = (QD + 2 * KV) * h + h * QD + 2 * inter * h + h * inter
        scales = F * (QD + 2 * KV + h + 2 * inter + h)
        if kind == "decode":
            t, keys = 1, case["pos"] + 1
        elif kind == "prefill":
            t, keys = case["tokens"], case["start"] + case["tokens"]
        else:
            t, keys = case["batch"], case["batch"] * (case["rows"] + 1) / 2  # mean of the drawn positions
        if kind == "prefill":
            pairs = t * case["start"] + t * (t + 1) / 2
        else:
            pairs = keys
        per_layer = weights + scales + F * (2 * keys * KV + 2 * h + 2 * HD)
        flops = layers * (2 * t * weights + 4 * pairs * QD)
        total = layers * per_layer + F * 2 * t * h
        if kind != "prefill":  # final norm, lm_head, logits
            total += VOCAB * h + F * VOCAB + F * t * VOCAB + F * h
            flops += 2 * t * VOCAB * h
        return {"bytes": total, "flops": flops}
    if kind == "encoder":
        n = case["rows"] * case["dim"]
        return {"bytes": F * (n * (4 + 3 * 4 - 4 + 4) + case["positions"] * case["dim"] + 4 * case["dim"]),
                "flops": 150 * n}
    if kind == "lm_head":
        h, r = case["hidden"], case["rows"]
        return {"bytes": VOCAB * h + F * VOCAB + F * r * (h + VOCAB + 1), "flops": 2 * r * VOCAB * h}
    h, b = case["hidden"], case["batch"]
    return {"bytes": 6 * h * h + F * 6 * h + b * (F * 3 * h + h + F + F * 2 * (QD + KV) + F * 3 * h + F * 2 * HD),
            "flops": 2 * b * 6 * h * h}


def tolerance(case: dict) -> dict:
    """About four times what a last-bit change of the inputs and gains (relative 1e-7) moves the outputs."""
    kind = case["kind"]
    if kind in ("ops", "encoder", "lm_head"):
        return {"rel": 1e-6, "max": 5e-6}
    if kind == "prefill":
        return {"rel": 5e-6, "max": 4e-5} if case["layers"] > 6 else {"rel": 2e-6, "max": 1.5e-5}
    if kind == "decode":
        return {"rel": 1.5e-5, "max": 7e-5} if case["layers"] > 6 else {"rel": 5e-6, "max": 3e-5}
    if kind == "streams":
        # w8a8: a last bit decides between two int8 values of an activation, and a stream's row follows from them
        return {"rel": 3e-2, "max": 0.9} if case["w8a8"] else {"rel": 5e-6, "max": 3e-5}
    return {"rel": 2e-3, "max": 4e-2, "differ": 1e-3}  # as w8a8 streams, one layer's half


# ---------------------------------------------------------------------------
# The same pass in 64 bits
# ---------------------------------------------------------------------------
def _rms(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def _ln(x: torch.Tensor, w: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    x = x - x.mean(-1, keepdim=True)
    return x / (x.square().mean(-1, keepdim=True) + 1e-5).sqrt() * w.double() + b.double()


def _rope(x: torch.Tensor, pos: torch.Tensor) -> torch.Tensor:
    """x [t, heads, HD] rotated at pos [t]. The model's angles are float32 by definition:
    (float32) position times the float32 inverse frequency."""
    inv = np.array([np.float32(1.0) / np.float32(math.pow(THETA, float(np.float32(2 * d) / np.float32(HD))))
                    for d in range(HD // 2)], np.float32)
    angle = (pos.to(F32)[:, None] * torch.from_numpy(inv).to(x.device)[None, :]).double()[:, None, :]
    a, b = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], -1)


def _linear(x: torch.Tensor, w: K.QuantWeight) -> torch.Tensor:
    parts = []
    for o in range(0, w.out_dim, 8192):
        e = min(w.out_dim, o + 8192)
        q = w.data[o * w.in_dim:e * w.in_dim].view(e - o, w.in_dim).double()
        parts.append((x @ q.t().contiguous()) * w.scales[o:e].double())
    return torch.cat(parts, -1)


def _swiglu(gate_up: torch.Tensor) -> torch.Tensor:
    g, u = gate_up[..., 0::2], gate_up[..., 1::2]
    return g / (1 + (-g).exp()) * u


def _attend(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, offset: int) -> torch.Tensor:
    """q [t, NQ, HD] at positions offset.. over k, v [n, NK, HD]."""
    t, n = q.shape[0], k.shape[0]
    late = torch.arange(n, device=q.device)[None, :] > torch.arange(offset, offset + t, device=q.device)[:, None]
    out = torch.empty_like(q)
    for h in range(NQ):
        kk, vv = k[:, h // (NQ // NK)].contiguous(), v[:, h // (NQ // NK)].contiguous()
        p = (q[:, h].contiguous() @ kk.t().contiguous()) / math.sqrt(HD)
        out[:, h] = p.masked_fill_(late, -math.inf).softmax(-1) @ vv
    return out


def _layers(x: torch.Tensor, w: dict, pos: torch.Tensor, attend) -> torch.Tensor:
    """The decoder's layers on rows x [t, hidden]; attend(layer, q, k, v) stores the rows and attends."""
    t = x.shape[0]
    for l, lw in enumerate(w["layers"]):
        n = _rms(x, lw["input_norm"])
        q = _rope(_rms(_linear(n, lw["wq"]).view(t, NQ, HD), lw["q_norm"]), pos)
        k = _rope(_rms(_linear(n, lw["wk"]).view(t, NK, HD), lw["k_norm"]), pos)
        a = attend(l, q, k, _linear(n, lw["wv"]).view(t, NK, HD))
        x = x + _linear(a.reshape(t, QD), lw["wo"])
        x = x + _linear(_swiglu(_linear(_rms(x, lw["post_attn_norm"]), lw["gate_up"])), lw["down"])
    return x


def _embed(w: K.QuantWeight, ids: torch.Tensor) -> torch.Tensor:
    i = ids.long()
    return w.data.view(w.out_dim, w.in_dim)[i].double() * w.scales[i].double()[:, None]


def exact(case: dict, seed: int):
    kind = case["kind"]
    if case.get("w8a8"):
        return None  # activations rounded to int8 inside: a last bit decides a whole step there
    s = prepare(case, seed)
    if kind == "ops":
        h, t = case["hidden"], case["tokens"]
        x = (s["x"].double() + s["delta"].double()).view(t, h)
        q, k = (_rope(_rms(s[n].double().view(t, -1, HD), s[n + "w"]), s["pos"]) for n in "qk")
        return {"x": x.view(-1), "out": _rms(x, s["w"]).view(-1), "q": q.reshape(-1), "k": k.reshape(-1),
                "act": _swiglu(s["gate_up"].double().view(t, -1)).reshape(-1)}
    if kind in ("decode", "prefill"):
        d, w, start, h = s["d"], s["w"], s["start"], case["hidden"]
        t = 1 if kind == "decode" else case["tokens"]
        kc, vc = (c.double().view(case["layers"], -1, NK, HD) for c in (d.kv.k, d.kv.v))

        def attend(l, q, k, v):
            kc[l, start:start + t], vc[l, start:start + t] = k, v
            return _attend(q, kc[l, :start + t], vc[l, :start + t], start)

        x = _embed(w["tok_embeddings"], s["token"]) if kind == "decode" else s["embeds"].double().view(t, h)
        x = _layers(x, w, torch.arange(start, start + t, device=x.device), attend)
        if kind == "prefill":
            return {"x": x.view(-1), "k": kc.view(-1), "v": vc.view(-1)}
        n = _rms(x, w["norm"])
        return {"logits": _linear(n, w["lm_head"]).view(-1), "x_norm": n.view(-1), "k": kc.view(-1), "v": vc.view(-1)}
    if kind == "streams":
        d, w, b, rows = s["d"], s["w"], case["batch"], case["rows"]
        kc, vc = d.k.clone().view(case["layers"], b, rows, NK, HD), d.v.clone().view(case["layers"], b, rows, NK, HD)
        at = d.positions.tolist()

        def attend(l, q, k, v):
            out = torch.empty_like(q)
            for i, p in enumerate(at):
                kk = torch.cat([kc[l, i, :p].double(), k[i:i + 1]])
                vv = torch.cat([vc[l, i, :p].double(), v[i:i + 1]])
                out[i:i + 1] = _attend(q[i:i + 1], kk, vv, p)
                kc[l, i, p], vc[l, i, p] = k[i].to(F32), v[i].to(F32)
            return out

        n = _rms(_layers(_embed(w["tok_embeddings"], s["tokens"]), w, d.positions, attend), w["norm"])
        return {"logits": _linear(n, w["lm_head"]).view(-1), "x_norm": n.view(-1), "k": kc.view(d.k.shape),
                "v": vc.view(d.v.shape)}
    if kind == "encoder":
        r, dim = case["rows"], case["dim"]
        pe = s["pe"].double().view(-1, dim)
        x = s["x"].double().view(r, dim) + pe[torch.arange(r, device=pe.device) % pe.shape[0]]
        x2, f = x + s["delta"].double().view(r, dim), s["ffn"].double()
        return {"x": x2.view(-1), "out": _ln(x, s["w"], s["b"]).view(-1),
                "act": f * 0.5 * (1 + torch.erf(f / math.sqrt(2.0))), "out2": _ln(x2, s["w2"], s["b2"]).view(-1)}
    if kind == "lm_head":
        return {"idx": None, "logits": _linear(s["x"].double().view(case["rows"], -1), s["w"]).view(-1)}
    h, b = case["hidden"], case["batch"]
    x = (s["x"].double() + s["delta"].double()).view(b, h)
    q, k = (_rope(_rms(s[n].double().view(b, -1, HD), s[n + "w"]), s["pos"]) for n in "qk")
    n = _rms(x, s["w"])  # its int8 values, and what follows from them, hang on last bits
    return {"x": x.view(-1), "xq": None, "xs": n.abs().amax(-1) / 127, "q": q.reshape(-1), "k": k.reshape(-1),
            "out": None}
