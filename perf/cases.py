"""Workloads of the TinyLlama device path: what a serving program calls, over
the sizes it meets.

A case is a dict of plain values whose "kind" names the call:

    decode   Engine.decode: RoPE + cache append + attention, one new token for
             each of n_seq sequences, `layers` layers per call
    prefill  Engine.prefill: RoPE + append + causal attention of n_tok prompt
             tokens at positions pos0 ..
    matmul   Engine.matmul (one vector) / Engine.matmul_batch: one weight matrix
    layer    attn_qkv, decode, attn_out, ffn_block: one transformer layer of a
             decode step over n_seq sequences
    forward  Engine.forward: one token through the whole model, to logits
    prompt   Engine.prefill_forward: a prompt through the whole model as one
             batch, to the last token's logits

Shapes are TinyLlama's (22 layers, n_embd 2048, 32 / 4 heads of 64, n_ff 5632,
vocabulary 32000) and, for attention, other head counts the engine takes.
Weights are Gaussian, quantised to the GGUF formats on the device.

listed() are the named cases, draw(rng) another of the same ranges;
prepare / run / work / tolerance / exact serve one case.
"""
from __future__ import annotations

import importlib
import math

import numpy as np
import torch

tla = importlib.import_module("tinyllama-engine_amd")

DEV = "cuda"
HEAD_DIM = 64
N_LAYERS, N_EMBD, N_HEAD, N_HEAD_KV, N_FF, N_VOCAB = 22, 2048, 32, 4, 5632, 32000
EPS = 1e-5
FREQ_BASE = 10000.0
TYPES = {"f32": tla.W_F32, "f16": tla.W_F16, "q4_0": tla.W_Q4_0, "q8_0": tla.W_Q8_0, "q6_k": tla.W_Q6_K}
ROW_BYTES = {"f32": lambda c: 4 * c, "f16": lambda c: 2 * c, "q8_0": lambda c: c // 32 * 34,
             "q4_0": lambda c: c // 32 * 18, "q6_k": lambda c: c // 256 * 210}


def listed():
    return [
        # one layer's attention block for one short conversation: pure latency
        {"name": "decode_single", "kind": "decode", "n_seq": 1, "layers": 1, "n_head": 32, "n_head_kv": 4,
         "ctx": 128, "ragged": False},
        # the attention of one decode step at TinyLlama's full context
        {"name": "decode_model", "kind": "decode", "n_seq": 1, "layers": 22, "n_head": 32, "n_head_kv": 4,
         "ctx": 2048, "ragged": False},
        # a serving batch of conversations of all lengths
        {"name": "decode_ragged", "kind": "decode", "n_seq": 64, "layers": 8, "n_head": 32, "n_head_kv": 4,
         "ctx": 2048, "ragged": True},
        # long documents, a small batch
        {"name": "decode_long", "kind": "decode", "n_seq": 8, "layers": 4, "n_head": 32, "n_head_kv": 4,
         "ctx": 16384, "ragged": False},
        # the attention of a 512-token prompt, all layers in one call
        {"name": "prefill_512", "kind": "prefill", "n_tok": 512, "pos0": 0, "layers": 22, "n_head": 32,
         "n_head_kv": 4},
        # the next chunk of a longer prompt, one layer
        {"name": "prefill_chunk", "kind": "prefill", "n_tok": 333, "pos0": 1500, "layers": 1, "n_head": 32,
         "n_head_kv": 4},
        # the classifier of a decode step (TinyLlama files keep it in Q6_K)
        {"name": "head_q6_k", "kind": "matmul", "type": "q6_k", "rows": 32000, "cols": 2048, "n_tok": 1},
        # one projection of a prompt
        {"name": "gate_q8_0_200", "kind": "matmul", "type": "q8_0", "rows": 5632, "cols": 2048, "n_tok": 200},
        # one layer of a decode step over a small and a large serving batch
        {"name": "layer_q8_0_12", "kind": "layer", "type": "q8_0", "n_seq": 12, "ctx": 512},
        {"name": "layer_f16_64", "kind": "layer", "type": "f16", "n_seq": 64, "ctx": 1024},
        # one token of a chat through the whole model
        {"name": "forward_q4_0", "kind": "forward", "type": "q4_0", "pos": 100},
        # a prompt through the whole model
        {"name": "prompt_q4_0_512", "kind": "prompt", "type": "q4_0", "n_tok": 512},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "matmul", "matmul", "layer", "layer", "forward", "prompt"])
    if kind == "decode":
        n_head, n_head_kv = rng.choice([(32, 4), (32, 4), (32, 8), (16, 2), (8, 8)])
        ctx = _log(rng, 16, 16384)
        layers = rng.choice([1, 2, 4, 8, 22])
        # at most the positions of the largest listed batch
        n_seq = _log(rng, 1, max(1, min(96, 500000 // (ctx * layers))))
        return {"kind": kind, "n_seq": n_seq, "layers": layers, "n_head": n_head, "n_head_kv": n_head_kv,
                "ctx": ctx, "ragged": n_seq > 1 and rng.random() < 0.6}
    if kind == "prefill":
        n_head, n_head_kv = rng.choice([(32, 4), (32, 4), (32, 8), (16, 2), (8, 8)])
        n_tok = _log(rng, 2, 1500)
        return {"kind": kind, "n_tok": n_tok, "pos0": rng.choice([0, 0, rng.randrange(0, 1500)]),
                "layers": rng.choice([1, 2, 22] if n_tok <= 512 else [1, 2]), "n_head": n_head,
                "n_head_kv": n_head_kv}
    if kind == "matmul":
        rows, cols = rng.choice([(2560, 2048), (2048, 2048), (11264, 2048), (2048, 5632), (32000, 2048),
                                 (rng.randrange(50, 3000), 256 * rng.randrange(1, 17))])
        n_tok = rng.choice([1, _log(rng, 2, 64), _log(rng, 16, 512)])
        if rows == 32000:
            n_tok = min(n_tok, 8)
        return {"kind": kind, "type": rng.choice(sorted(TYPES)), "rows": rows, "cols": cols, "n_tok": n_tok}
    if kind == "layer":
        return {"kind": kind, "type": rng.choice(["q4_0", "q8_0", "f16"]), "n_seq": _log(rng, 1, 128),
                "ctx": _log(rng, 64, 1024)}
    if kind == "forward":
        return {"kind": kind, "type": rng.choice(["q4_0", "q8_0", "f16"]), "pos": _log(rng, 1, 2047)}
    return {"kind": "prompt", "type": rng.choice(["q4_0", "q8_0", "f16"]), "n_tok": _log(rng, 2, 512)}


# ---- inputs ---------------------------------------------------------------------

class Gen:
    """Seeded inputs on the device."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return torch.randn(*shape, generator=self.g, device=DEV).mul_(std)

    def uniform(self, *shape, lo=0.0, hi=1.0):
        return torch.rand(*shape, generator=self.g, device=DEV).mul_(hi - lo).add_(lo)

    def ints(self, lo, hi, n):
        return torch.randint(lo, hi, (n,), generator=self.g, device=DEV).cpu().tolist()

    def weights(self, rows, cols, wtype, std=0.02):
        return quantise(self.normal(rows, cols, std=std), wtype)


def _bytes(t):
    return t.contiguous().view(torch.uint8).reshape(*t.shape[:-1], -1)


def quantise(w, wtype):
    """w [rows][cols] as GGUF bytes, uint8 [rows * row bytes]."""
    rows, cols = w.shape
    if wtype == "f32":
        return _bytes(w).reshape(-1)
    if wtype == "f16":
        return _bytes(w.half()).reshape(-1)
    if wtype == "q8_0":
        b = w.view(rows, cols // 32, 32)
        d = (b.abs().amax(-1, keepdim=True) / 127).half()
        q = (b / d.float().clamp_min(1e-12)).round_().clamp_(-127, 127).to(torch.int8)
        return torch.cat([_bytes(d), _bytes(q)], -1).reshape(-1)
    if wtype == "q4_0":
        b = w.view(rows, cols // 32, 32)
        at = b.abs().argmax(-1, keepdim=True)
        d = (b.gather(-1, at) / -8).half()
        df = d.float()
        q = torch.where(df == 0, torch.full_like(b, 8.0), (b / torch.where(df == 0, torch.ones_like(df), df) + 8.5).floor_())
        q = q.clamp_(0, 15).to(torch.uint8)
        return torch.cat([_bytes(d), q[..., :16] | (q[..., 16:] << 4)], -1).reshape(-1)
    if wtype == "q6_k":
        b = w.view(rows, cols // 256, 16, 16)
        sub = b.abs().amax(-1) / 31
        d = (sub.amax(-1, keepdim=True) / 127).half()
        sc = (sub / d.float().clamp_min(1e-12)).round_().clamp_(1, 127).to(torch.int8)
        scale = (d.float() * sc.float()).clamp_min(1e-12).unsqueeze(-1)
        q = ((b / scale).round_().clamp_(-32, 31) + 32).to(torch.uint8).view(rows, cols // 256, 2, 4, 32)
        # value 128 h + 32 k + i: low nibbles of byte 64 h + 32 (k % 2) + i
        # (k < 2) or its high ones, bits 2k of byte 32 h + i of the high part
        ql = torch.stack([(q[:, :, :, 0] & 15) | ((q[:, :, :, 2] & 15) << 4),
                          (q[:, :, :, 1] & 15) | ((q[:, :, :, 3] & 15) << 4)], 3)
        qh = (q[:, :, :, 0] >> 4) | ((q[:, :, :, 1] >> 4) << 2) | ((q[:, :, :, 2] >> 4) << 4) | ((q[:, :, :, 3] >> 4) << 6)
        return torch.cat([ql.reshape(rows, cols // 256, 128), qh.reshape(rows, cols // 256, 64), _bytes(sc), _bytes(d)],
                         -1).reshape(-1)
    raise ValueError(wtype)


def dequantise(raw, rows, cols, wtype):
    """The values of GGUF bytes in 64 bits, [rows][cols]."""
    f64 = torch.float64
    if wtype == "f32":
        return raw.view(torch.float32).view(rows, cols).to(f64)
    if wtype == "f16":
        return raw.view(torch.float16).view(rows, cols).to(f64)
    if wtype == "q8_0":
        b = raw.view(rows, cols // 32, 34)
        return (b[..., 2:].contiguous().view(torch.int8).to(f64) * b[..., :2].contiguous().view(torch.float16).to(f64)).view(rows, cols)
    if wtype == "q4_0":
        b = raw.view(rows, cols // 32, 18)
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], -1).to(f64) - 8
        return (q * b[..., :2].contiguous().view(torch.float16).to(f64)).view(rows, cols)
    b = raw.view(rows, cols // 256, 210)
    ql = b[..., :128].reshape(rows, -1, 2, 2, 32)
    qh = b[..., 128:192].reshape(rows, -1, 2, 1, 32)
    lo = torch.cat([ql & 15, ql >> 4], 3)
    hi = torch.cat([qh >> s & 3 for s in (0, 2, 4, 6)], 3)
    q = (lo | (hi << 4)).to(f64) - 32
    sc = b[..., 192:208].contiguous().view(torch.int8).to(f64)
    d = b[..., 208:210].contiguous().view(torch.float16).to(f64)
    return (q.reshape(rows, -1, 16, 16) * (sc * d).unsqueeze(-1)).reshape(rows, cols)


_engines: dict = {}


def engine(layers=N_LAYERS, n_ctx=2048, n_head=N_HEAD, n_head_kv=N_HEAD_KV):
    """The process's engine for one configuration (a server keeps one)."""
    n_ctx = max(128, 1 << (n_ctx - 1).bit_length())
    key = (layers, n_ctx, n_head, n_head_kv)
    if key not in _engines:
        _engines[key] = tla.Engine(tla.Config(layers, n_head * HEAD_DIM, n_head, n_head_kv, n_ctx, FREQ_BASE))
    return _engines[key]


class DeviceWeights:
    """A whole model's weights in device tensors, described as a tla.Model."""

    def __init__(self, gen, wtype):
        kv = N_HEAD_KV * HEAD_DIM
        ty = TYPES[wtype]
        self.wtype = wtype
        self.embd = gen.weights(N_VOCAB, N_EMBD, wtype, std=1.0)
        self.layers = []
        for _ in range(N_LAYERS):
            self.layers.append({
                "attn_norm": gen.uniform(N_EMBD, lo=0.5, hi=1.5), "wq": gen.weights(N_EMBD, N_EMBD, wtype),
                "wk": gen.weights(kv, N_EMBD, wtype), "wv": gen.weights(kv, N_EMBD, wtype),
                "wo": gen.weights(N_EMBD, N_EMBD, wtype), "ffn_norm": gen.uniform(N_EMBD, lo=0.5, hi=1.5),
                "w_gate": gen.weights(N_FF, N_EMBD, wtype), "w_up": gen.weights(N_FF, N_EMBD, wtype),
                "w_down": gen.weights(N_EMBD, N_FF, wtype)})
        self.norm = gen.uniform(N_EMBD, lo=0.5, hi=1.5)
        self.head = gen.weights(N_VOCAB, N_EMBD, "q6_k")
        p = lambda d, k: d[k].data_ptr()  # noqa: E731
        self.table = (tla.LayerWeights * N_LAYERS)(*[
            tla.LayerWeights(p(d, "attn_norm"), p(d, "wq"), p(d, "wk"), p(d, "wv"), p(d, "wo"), ty, ty, ty, ty,
                             p(d, "ffn_norm"), p(d, "w_gate"), p(d, "w_up"), p(d, "w_down"), ty) for d in self.layers])
        self.c = tla.Model(N_FF, N_VOCAB, EPS, self.embd.data_ptr(), ty, self.norm.data_ptr(), self.head.data_ptr(),
                           TYPES["q6_k"], self.table)


def lengths(case, gen):
    """Positions of the new tokens: ctx - 1, or uniform in [ctx / 8, ctx)."""
    n, ctx = case["n_seq"], case["ctx"]
    if case["ragged"]:
        return np.array(gen.ints(ctx // 8, ctx, n), np.int32)
    return np.full(n, ctx - 1, np.int32)


def caches(gen, n_seq, layers, n_ctx, kv_dim):
    """Key and value caches with every row filled (rows past a sequence's
    position hold an earlier request's)."""
    return gen.normal(n_seq, layers, n_ctx, kv_dim), gen.normal(n_seq, layers, n_ctx, kv_dim)


def prepare(case, seed):
    kind, gen, s = case["kind"], Gen(seed), {"kind": case["kind"]}
    if kind == "decode":
        h, hkv, nl, ns = case["n_head"], case["n_head_kv"], case["layers"], case["n_seq"]
        e = s["e"] = engine(nl, case["ctx"], h, hkv)
        s["pos"] = lengths(case, gen)
        s["q"], s["k"], s["v"] = (gen.normal(ns, nl, n * HEAD_DIM) for n in (h, hkv, hkv))
        s["kc"], s["vc"] = caches(gen, ns, nl, e.cfg.n_ctx, hkv * HEAD_DIM)
        s["out"] = torch.zeros_like(s["q"])
        s["stride"] = nl * e.cfg.n_ctx * hkv * HEAD_DIM
    elif kind == "prefill":
        h, hkv, nl, nt = case["n_head"], case["n_head_kv"], case["layers"], case["n_tok"]
        e = s["e"] = engine(nl, case["pos0"] + nt, h, hkv)
        s["q"], s["k"], s["v"] = (gen.normal(nl, nt, n * HEAD_DIM) for n in (h, hkv, hkv))
        s["kc"], s["vc"] = caches(gen, 1, nl, e.cfg.n_ctx, hkv * HEAD_DIM)
        s["out"] = torch.zeros_like(s["q"])
    elif kind == "matmul":
        s["e"] = engine()
        s["w"] = gen.weights(case["rows"], case["cols"], case["type"])
        s["x"] = gen.normal(case["n_tok"], case["cols"])
        s["out"] = torch.zeros(case["n_tok"], case["rows"], device=DEV)
    elif kind == "layer":
        ns, ty = case["n_seq"], case["type"]
        e = s["e"] = engine(1, case["ctx"])
        s["pos"] = lengths(dict(case, ragged=ns > 1), gen)
        kv = N_HEAD_KV * HEAD_DIM
        s["w"] = {"attn_norm": gen.uniform(N_EMBD, lo=0.5, hi=1.5), "wq": gen.weights(N_EMBD, N_EMBD, ty),
                  "wk": gen.weights(kv, N_EMBD, ty), "wv": gen.weights(kv, N_EMBD, ty),
                  "wo": gen.weights(N_EMBD, N_EMBD, ty), "ffn_norm": gen.uniform(N_EMBD, lo=0.5, hi=1.5),
                  "w_gate": gen.weights(N_FF, N_EMBD, ty), "w_up": gen.weights(N_FF, N_EMBD, ty),
                  "w_down": gen.weights(N_EMBD, N_FF, ty)}
        s["x0"] = gen.normal(ns, N_EMBD)
        s["x"] = torch.zeros_like(s["x0"])
        s["q"], s["att"] = torch.zeros_like(s["x0"]), torch.zeros_like(s["x0"])
        s["k"], s["v"] = (torch.zeros(ns, kv, device=DEV) for _ in range(2))
        s["hb"] = torch.zeros(ns, 2, N_FF, device=DEV)
        s["kc"], s["vc"] = caches(gen, ns, 1, e.cfg.n_ctx, kv)
        s["stride"] = e.cfg.n_ctx * kv
    else:
        s["e"] = engine()
        s["model"] = DeviceWeights(gen, case["type"])
        s["tokens"] = gen.ints(0, N_VOCAB, case.get("n_tok", 1))
        s["kc"], s["vc"] = caches(gen, 1, N_LAYERS, s["e"].cfg.n_ctx, N_HEAD_KV * HEAD_DIM)
        s["logits"] = torch.zeros(N_VOCAB, device=DEV)
    s["case"] = dict(case)
    torch.cuda.synchronize()  # the engine has a stream of its own
    return s


# ---- one pass -------------------------------------------------------------------

def run(s):
    kind, e, c = s["kind"], s["e"], s["case"]
    if kind == "decode":
        e.decode(s["pos"], 0, c["layers"], s["out"].data_ptr(), s["q"].data_ptr(), s["k"].data_ptr(),
                 s["v"].data_ptr(), s["kc"].data_ptr(), s["vc"].data_ptr(), s["stride"])
        return s["out"], s["kc"], s["vc"]
    if kind == "prefill":
        e.prefill(c["pos0"], c["n_tok"], 0, c["layers"], s["out"].data_ptr(), s["q"].data_ptr(), s["k"].data_ptr(),
                  s["v"].data_ptr(), s["kc"].data_ptr(), s["vc"].data_ptr())
        return s["out"], s["kc"], s["vc"]
    if kind == "matmul":
        args = s["out"].data_ptr(), s["w"].data_ptr(), s["x"].data_ptr(), c["rows"], c["cols"]
        if c["n_tok"] == 1:
            e.matmul(*args, TYPES[c["type"]])
        else:
            e.matmul_batch(*args, c["n_tok"], TYPES[c["type"]])
        return s["out"]
    if kind == "layer":
        n, ty, x = c["n_seq"], TYPES[c["type"]], s["x"].data_ptr()
        w = {k: t.data_ptr() for k, t in s["w"].items()}
        e.copy(x, s["x0"].data_ptr(), s["x0"].numel() * 4)
        e.attn_qkv(n, s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), x, w["attn_norm"], EPS, w["wq"],
                   w["wk"], w["wv"], ty)
        e.decode(s["pos"], 0, 1, s["att"].data_ptr(), s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                 s["kc"].data_ptr(), s["vc"].data_ptr(), s["stride"])
        e.attn_out(n, x, w["wo"], s["att"].data_ptr(), ty)
        e.ffn_block(n, x, w["ffn_norm"], EPS, w["w_gate"], w["w_up"], w["w_down"], N_FF, ty, s["hb"].data_ptr())
        return s["x"], s["kc"], s["vc"]
    if kind == "forward":
        e.forward(s["model"], s["kc"].data_ptr(), s["vc"].data_ptr(), s["tokens"][0], c["pos"], s["logits"].data_ptr())
    else:
        e.prefill_forward(s["model"], s["kc"].data_ptr(), s["vc"].data_ptr(), s["tokens"], 0, s["logits"].data_ptr())
    return s["logits"], s["kc"], s["vc"]


# ---- what a pass cannot do without -----------------------------------------------

def _attention_work(n_head, n_head_kv, new, keys, query_keys):
    """Bytes and flops of one layer: `new` tokens appended, `keys` cache rows of
    each cache read, query_keys (query, key) pairs per head."""
    kv = n_head_kv * HEAD_DIM * 4
    return (2 * keys * kv + new * (2 * n_head * HEAD_DIM * 4 + 4 * kv), 4 * n_head * HEAD_DIM * query_keys)


def _layer_weights(wtype):
    rows = [(N_EMBD, N_EMBD), (512, N_EMBD), (N_EMBD, N_EMBD), (2 * N_FF, N_EMBD), (N_EMBD, N_FF)]
    return sum(r * ROW_BYTES[wtype](c) for r, c in rows), sum(r * c for r, c in rows)


def work(case):
    kind = case["kind"]
    if kind == "decode":
        # a ragged batch's mean length
        ln = case["ctx"] if not case["ragged"] else (case["ctx"] // 8 + case["ctx"]) // 2
        n = case["n_seq"] * case["layers"]
        b, f = _attention_work(case["n_head"], case["n_head_kv"], 1, ln - 1, ln)
        return {"bytes": n * b, "flops": n * f}
    if kind == "prefill":
        t, p = case["n_tok"], case["pos0"]
        b, f = _attention_work(case["n_head"], case["n_head_kv"], t, p, t * p + t * (t + 1) // 2)
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    if kind == "matmul":
        r, c, t = case["rows"], case["cols"], case["n_tok"]
        return {"bytes": r * ROW_BYTES[case["type"]](c) + 4 * t * (r + c), "flops": 2 * r * c * t}
    wb, wn = _layer_weights(case["type"])
    if kind == "layer":
        n = case["n_seq"]
        ln = case["ctx"] if n == 1 else (case["ctx"] // 8 + case["ctx"]) // 2
        b, f = _attention_work(N_HEAD, N_HEAD_KV, 1, ln - 1, ln)
        # the residual in and out; q, k, v and the attention's output stay inside the layer
        return {"bytes": wb + n * (b + 8 * N_EMBD), "flops": n * (f + 2 * wn)}
    t = case.get("n_tok", 1)
    p = case.get("pos", 0)
    b, f = _attention_work(N_HEAD, N_HEAD_KV, t, p, t * p + t * (t + 1) // 2)
    head = N_VOCAB * ROW_BYTES["q6_k"](N_EMBD)
    return {"bytes": N_LAYERS * (wb + b) + head + t * ROW_BYTES[case["type"]](N_EMBD) + 4 * N_VOCAB,
            "flops": t * N_LAYERS * 2 * wn + N_LAYERS * f + 2 * N_VOCAB * N_EMBD}


# About four times the error against 64 bits of the 32-bit sums, over the
# ranges: attention 1e-7 to 7e-7, a product 1e-7 to 3e-7, a layer 1.5e-7 to
# 3e-7; a whole model's last logits 0.9e-6 to 2.3e-6, since a rounding in one
# layer travels through those that follow.
TOLERANCE = {"decode": 3e-6, "prefill": 3e-6, "matmul": 1.5e-6, "layer": 2e-6, "forward": 1e-5, "prompt": 1e-5}


def tolerance(case):
    return {"rel": TOLERANCE[case["kind"]]}


# ---- the same in 64 bits ----------------------------------------------------------

F64 = torch.float64


def _rotate(x, pos):
    """RoPE of x [n][heads * 64] at positions pos [n]: consecutive pairs; the
    angle is the engine's (32-bit position times 32-bit frequency)."""
    i = np.arange(HEAD_DIM // 2)
    expo = (2 * i).astype(np.float32) / np.float32(HEAD_DIM)
    freq = np.float32(1) / np.power(np.float64(np.float32(FREQ_BASE)), expo.astype(np.float64)).astype(np.float32)
    angle = np.asarray(pos, np.float32)[:, None] * freq[None, :]
    a = torch.from_numpy(angle).to(x.device).to(F64)[:, None, :]
    c, s = a.cos(), a.sin()
    y = x.to(F64).view(x.shape[0], -1, HEAD_DIM // 2, 2)
    return torch.stack([y[..., 0] * c - y[..., 1] * s, y[..., 0] * s + y[..., 1] * c], -1).view(x.shape[0], -1)


def _attend(q, k, v, pos0):
    """Causal attention of q [t][H * 64] at pos0 .. over k, v [n][Hkv * 64]."""
    t, n = q.shape[0], k.shape[0]
    h, hkv = q.shape[1] // HEAD_DIM, k.shape[1] // HEAD_DIM
    out = torch.empty(t, h, HEAD_DIM, dtype=F64, device=q.device)
    mask = torch.arange(n, device=q.device)[None, :] > pos0 + torch.arange(t, device=q.device)[:, None]
    for g in range(hkv):
        kg = k[:, g * HEAD_DIM:(g + 1) * HEAD_DIM].to(F64)
        vg = v[:, g * HEAD_DIM:(g + 1) * HEAD_DIM].to(F64)
        r = h // hkv
        qg = q.to(F64).view(t, h, HEAD_DIM)[:, g * r:(g + 1) * r].reshape(t * r, HEAD_DIM)
        sc = (qg @ kg.t()).view(t, r, n) / math.sqrt(HEAD_DIM)
        sc.masked_fill_(mask[:, None, :], -math.inf)
        out[:, g * r:(g + 1) * r] = (torch.softmax(sc, -1).view(t * r, n) @ vg).view(t, r, HEAD_DIM)
    return out.view(t, h * HEAD_DIM)


def _norm(x, w):
    return x / (x.square().mean(-1, keepdim=True) + float(np.float32(EPS))).sqrt() * w.to(F64)


def _product(x, raw, rows, wtype):
    return x.to(F64) @ dequantise(raw, rows, x.shape[-1], wtype).t()


def _layer(x, w, wtype, attend):
    """One layer over x [t][n_embd]; attend(q, k, v) is its attention block."""
    kv = N_HEAD_KV * HEAD_DIM
    h = _norm(x, w["attn_norm"])
    a = attend(_product(h, w["wq"], N_EMBD, wtype), _product(h, w["wk"], kv, wtype), _product(h, w["wv"], kv, wtype))
    x = x + _product(a, w["wo"], N_EMBD, wtype)
    h = _norm(x, w["ffn_norm"])
    g = _product(h, w["w_gate"], N_FF, wtype)
    u = _product(h, w["w_up"], N_FF, wtype)
    return x + _product(g * torch.sigmoid(g) * u, w["w_down"], N_EMBD, wtype)


def exact(case, seed):
    kind = case["kind"]
    s = prepare(case, seed)
    if kind == "matmul":
        return _product(s["x"], s["w"], case["rows"], case["type"])
    kc, vc = s["kc"].to(F64), s["vc"].to(F64)

    def step(q, k, v, seq, layer, pos0):
        """Append k, v [t] at pos0 .. and attend."""
        n = q.shape[0]
        at = np.arange(pos0, pos0 + n)
        kc[seq, layer, pos0:pos0 + n] = _rotate(k, at)
        vc[seq, layer, pos0:pos0 + n] = v.to(F64)
        return _attend(_rotate(q, at), kc[seq, layer, :pos0 + n], vc[seq, layer, :pos0 + n], pos0)

    if kind == "decode":
        out = torch.empty_like(s["q"], dtype=F64)
        for i, p in enumerate(s["pos"].tolist()):
            for l in range(case["layers"]):
                out[i, l] = step(s["q"][i, l][None], s["k"][i, l][None], s["v"][i, l][None], i, l, p)[0]
        return out, kc, vc
    if kind == "prefill":
        return torch.stack([step(s["q"][l], s["k"][l], s["v"][l], 0, l, case["pos0"])
                            for l in range(case["layers"])]), kc, vc
    if kind == "layer":
        pos = s["pos"].tolist()
        batch = lambda q, k, v: torch.cat([step(q[i:i + 1], k[i:i + 1], v[i:i + 1], i, 0, p)  # noqa: E731
                                           for i, p in enumerate(pos)])
        return _layer(s["x0"].to(F64), s["w"], case["type"], batch), kc, vc
    m = s["model"]
    rb = ROW_BYTES[m.wtype](N_EMBD)
    rows = m.embd.view(N_VOCAB, rb)[torch.tensor(s["tokens"], device=DEV)]
    x = dequantise(rows.reshape(-1).contiguous(), len(s["tokens"]), N_EMBD, m.wtype)
    pos0 = case.get("pos", 0)
    for l, w in enumerate(m.layers):
        x = _layer(x, w, m.wtype, lambda q, k, v: step(q, k, v, 0, l, pos0))
    return _product(_norm(x[-1:], m.norm), m.head, N_VOCAB, "q6_k")[0], kc, vc
