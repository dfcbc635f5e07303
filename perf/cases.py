"""The workloads whose speed is tracked: Qwen2.5-1.5B-shape Q4_0 inference as a program using this framework runs it.

Whole calls run an 8-layer model of the full width with the full tied head (345 MB of weights, more than the
256 MB Infinity Cache, so a pass streams its weights from HBM as the 28-layer model does): the graph-replayed
decode step at batch 1 and in batches over the paged KV cache, and the prefill of a prompt. The other cases are single
layers, products, attention and the Q6_K head, each through an entry point that a program can call.

A case is a dict of plain values:
  kind "decode"   one greedy token at batch 1 at position `pos` (Decoder.capture, one graph replay)
  kind "batched"  one step of B sequences, contexts U[256, 2047] (BatchedDecoder.capture), `act` "q8" or "f16"
  kind "prefill"  Prefill.chunk of P prompt tokens at positions pos0 ..
  kind "layer"    Prefill.layer: one decoder layer for P tokens at positions pos0 ..
  kind "product"  q355_mmq_q4_0_q8_1 of T tokens with one of the model's matrices; gate_up with SwiGLU -> Q8_1
  kind "attn"     q355_attn_prefill of P queries at positions pos0 .., fp32 output
  kind "head"     the Q6_K LM head for T tokens (T = 1: q355_head_logits_q6k, else q355_mmq_q6k_logits)
"""
from __future__ import annotations

import functools
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parents[1] / "3080lab_amd"))

from lab import qwen_batched as QB  # noqa: E402
from lab import qwen_model as QM  # noqa: E402
from lab.hip import call, ptr  # noqa: E402

DEV = "cuda"
LAYERS, MAXLEN, PAGE = 8, 2048, 64
CFG = QM.Config(L=LAYERS)
H, FFN, HD, NH, NKV, V = 1536, 8960, 128, 12, 2, 151936
SCALE = 1.0 / math.sqrt(HD)
FIX = 2.0 ** 48                                            # residual stream: int64, value * 2^48
# the layer's matrices: rows, columns
MATS = {"qkv": ((NH + 2 * NKV) * HD, H), "o": (H, NH * HD), "gate_up": (2 * FFN, H), "down": (H, FFN)}


def listed():
    return [
        # a chat reply's tokens just after a short prompt: the batch-1 step, all launches and latency
        {"name": "decode_b1_pos140", "kind": "decode", "pos": 140},
        # the same deep into a long conversation, where the attention has 29 pages to read
        {"name": "decode_b1_pos1811", "kind": "decode", "pos": 1811},
        # a small serving batch
        {"name": "batched_q8_b8", "kind": "batched", "B": 8, "act": "q8"},
        # a full serving batch
        {"name": "batched_q8_b32", "kind": "batched", "B": 32, "act": "q8"},
        # a partly filled batch in the reference's fp16 arithmetic
        {"name": "batched_f16_b24", "kind": "batched", "B": 24, "act": "f16"},
        # a long prompt in one chunk, the largest call
        {"name": "prefill_2048", "kind": "prefill", "P": 2048, "pos0": 0},
        # a short question of odd length
        {"name": "prefill_77", "kind": "prefill", "P": 77, "pos0": 0},
        # the last chunk of a prompt prefilled in pieces of 512
        {"name": "layer_512_at_1536", "kind": "layer", "P": 512, "pos0": 1536},
        # a medium prompt of odd length
        {"name": "layer_333", "kind": "layer", "P": 333, "pos0": 0},
        # the largest product of the model alone, with its SwiGLU and Q8_1 epilogue
        {"name": "gate_up_2048", "kind": "product", "mat": "gate_up", "T": 2048},
        # the attention of a follow-up turn behind a 500-token history
        {"name": "attn_1500_at_500", "kind": "attn", "P": 1500, "pos0": 500},
        # llama.cpp's Q6_K output head for a small batch
        {"name": "head_q6k_b8", "kind": "head", "T": 8},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["decode", "batched", "prefill", "layer", "product", "attn", "head"])
    if kind == "decode":
        return {"kind": kind, "pos": rng.randint(1, 2046)}
    if kind == "batched":
        return {"kind": kind, "B": _log_int(rng, 2, 32), "act": rng.choice(["q8", "q8", "f16"])}
    if kind == "head":
        return {"kind": kind, "T": _log_int(rng, 1, 32)}
    if kind == "product":
        return {"kind": kind, "mat": rng.choice(sorted(MATS)), "T": _log_int(rng, 24, 2048)}
    n = _log_int(rng, 8, 2048)
    return {"kind": kind, "P": n, "pos0": rng.choice([0, rng.randint(0, 2048 - n)])}


# ---- inputs ----------------------------------------------------------------------------------------

def _gen(*seed):
    s = 0
    for v in seed:
        s = (s * 1000003 + int(v) + 12345) % (2 ** 62)
    return torch.Generator(device=DEV).manual_seed(s)


def _q4(g, n, k, std=0.02):
    """A Gaussian matrix [n, k] by the Q4_0 rule -> (q uint8 [n, k/32, 32] 0..15, d fp16 [n, k/32])."""
    x = torch.randn(n, k // 32, 32, generator=g, device=DEV) * std
    m = x.gather(2, x.abs().argmax(2, keepdim=True))
    d = m / -8.0
    q = torch.clamp(torch.floor(x / d + 8.5), 0, 15).to(torch.uint8)
    return q, d[..., 0].to(torch.float16)


def _gguf_bytes(q, d):
    """GGUF Q4_0 blocks [n * k/32, 18] as a numpy array (host), the form weights arrive in."""
    b = torch.empty(*q.shape[:2], 18, dtype=torch.uint8, device=DEV)
    b[..., :2] = d.view(torch.uint8).reshape(*d.shape, 2)
    b[..., 2:] = q[..., :16] | (q[..., 16:] << 4)
    return b.reshape(-1, 18).cpu().numpy()


def _planes(q, d):
    """The library's Q4_0 planes: qs uint8 [n/16][k/32][16][16], d fp16 [n/16][k/32][16]."""
    n, nb = d.shape
    qs = (q[..., :16] | (q[..., 16:] << 4)).reshape(n // 16, 16, nb, 16).transpose(1, 2).contiguous()
    return qs, d.reshape(n // 16, 16, nb).transpose(1, 2).contiguous()


def _q8(x):
    """Q8_1 of fp32 x [t, k]: codes int8 [t, k], stored blocks half2 [t, k/32, 2] = (d, d * sum q)."""
    x = x.to(torch.float32).reshape(x.shape[0], -1, 32)
    d = x.abs().amax(2, keepdim=True)
    d = d / torch.full_like(d, 127.0)                       # a division: by a Python number torch multiplies by 1/127
    q = torch.where(d != 0, torch.round(x / torch.where(d != 0, d, torch.ones_like(d))), torch.zeros_like(x))
    ds = torch.stack([d[..., 0], d[..., 0] * q.sum(2)], -1).to(torch.float16)
    return q.to(torch.int8).reshape(x.shape[0], -1), ds


@functools.lru_cache(maxsize=1)
def _model():
    """The 8-layer model: GGUF bytes on the host, its device form, loaded once as a serving program loads it."""
    g = _gen(7)
    vec = lambda n, std, mean=0.0: (torch.randn(n, generator=g, device=DEV) * std + mean).cpu().numpy()  # noqa: E731
    w = {"embed": _gguf_bytes(*_q4(g, V, H)), "norm": vec(H, 0.01, 1.0), "layers": []}
    for _ in range(LAYERS):
        L = {name: _gguf_bytes(*_q4(g, n, k)) for name, n, k in
             (("wq", NH * HD, H), ("wk", NKV * HD, H), ("wv", NKV * HD, H), ("wo", H, NH * HD), ("wg", FFN, H),
              ("wu", FFN, H), ("wd", H, FFN))}
        L.update(bq=vec(NH * HD, 0.02), bk=vec(NKV * HD, 0.02), bv=vec(NKV * HD, 0.02), ln1=vec(H, 0.01, 1.0),
                 ln2=vec(H, 0.01, 1.0))
        w["layers"].append(L)
    return w, QM.DeviceModel(w, CFG, maxlen=MAXLEN)


def _context(seed, layer, B):
    """K and V fp16 [B, NKV, MAXLEN, HD] of `layer`: what earlier tokens left in the cache."""
    g = _gen(seed, 100 + layer)
    return [torch.randn(B, NKV, MAXLEN, HD, generator=g, device=DEV).to(torch.float16) for _ in range(2)]


def _fill(cache, table, ctx):
    """Contiguous [B, NKV, MAXLEN, HD] -> the pages of `cache` that block table [B, pages] names."""
    B, pages = table.shape
    cache[table.reshape(-1).long()] = ctx.reshape(B, NKV, pages, PAGE, HD).transpose(1, 2).reshape(-1, NKV, PAGE, HD)


def _tokens(seed, n):
    return np.random.default_rng([int(seed), 5]).integers(0, V, n).astype(np.int32)


def _positions(seed, B):
    return np.random.default_rng([int(seed), 6]).integers(256, MAXLEN, B).astype(np.int32)


def _residual(seed, n):
    """A residual stream [n, H] as it stands between layers, int64 fixed point."""
    x = torch.randn(n, H, generator=_gen(seed, 11), device=DEV, dtype=torch.float64)
    return torch.round(x * FIX).to(torch.int64)


def _activations(seed, n, k):
    """Activations with a heavier tail than a Gaussian, as they come out of a norm or a SwiGLU."""
    g = _gen(seed, 12)
    return torch.randn(n, k, generator=g, device=DEV) * torch.exp(0.5 * torch.randn(n, k, generator=g, device=DEV))


def _q6(seed):
    """The Q6_K head: v uint8 [V, H] 0..63, sub-block scales int8 [V, H/16], super-block scales fp16 [V, H/256]."""
    g = _gen(3)
    v = torch.clamp(torch.round(torch.randn(V, H, generator=g, device=DEV) * 10) + 32, 0, 63).to(torch.uint8)
    sc = torch.randint(40, 128, (V, H // 16), generator=g, device=DEV, dtype=torch.int32).to(torch.int8)
    d = (torch.rand(V, H // 256, generator=g, device=DEV) * 4e-5 + 3e-5).to(torch.float16)
    return v, sc, d


@functools.lru_cache(maxsize=1)
def _q6_planes():
    v, sc, d = _q6(0)
    v = v.reshape(V, H // 32, 32)
    lo = (v[..., :16] & 15) | ((v[..., 16:] & 15) << 4)
    hv = v >> 4
    hi = hv[..., :8] | (hv[..., 8:16] << 2) | (hv[..., 16:24] << 4) | (hv[..., 24:] << 6)
    t = lambda a: a.reshape(V // 16, 16, *a.shape[1:]).transpose(1, 2).contiguous()  # noqa: E731
    return t(lo), t(hi), t(sc.reshape(V, H // 32, 2)), t(d)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        w, m = _model()
        dec = QM.Decoder(m, T=1, max_ctx=MAXLEN)
        for i in range(LAYERS):
            k, v = _context(seed, i, 1)
            _fill(dec.kc[i], dec.block_table, k)
            _fill(dec.vc[i], dec.block_table, v)
        tok = torch.from_numpy(_tokens(seed, 1)).to(DEV)
        pos = torch.full((1,), case["pos"], dtype=torch.int32, device=DEV)
        dec.tok.copy_(tok)
        dec.pos.copy_(pos)
        dec.capture()
        return {"kind": kind, "dec": dec, "tok": tok, "pos": pos}
    if kind == "batched":
        w, m = _model()
        B = case["B"]
        dec = QB.BatchedDecoder(m, B, MAXLEN, page_seed=int(seed) % 1000, act=case["act"], keep_logits=True)
        for i in range(LAYERS):
            k, v = _context(seed, i, B)
            _fill(dec.kc[i], dec.block_table, k)
            _fill(dec.vc[i], dec.block_table, v)
        tok = torch.from_numpy(_tokens(seed, B)).to(DEV)
        pos = torch.from_numpy(_positions(seed, B)).to(DEV)
        dec.tok.copy_(tok)
        dec.pos.copy_(pos)
        dec.capture()
        return {"kind": kind, "dec": dec, "tok": tok, "pos": pos}
    if kind in ("prefill", "layer"):
        w, m = _model()
        P, pos0 = case["P"], case["pos0"]
        dec = QM.Decoder(m, T=1, max_ctx=MAXLEN)
        pf = QB.Prefill(dec, max_chunk=MAXLEN)
        if pos0:
            for i in range(LAYERS if kind == "prefill" else 1):
                k, v = _context(seed, i, 1)
                k[:, :, pos0:] = 0
                v[:, :, pos0:] = 0
                _fill(dec.kc[i], dec.block_table, k)
                _fill(dec.vc[i], dec.block_table, v)
        s = {"kind": kind, "dec": dec, "pf": pf, "P": P, "pos0": pos0}
        if kind == "prefill":
            s["ids"] = _tokens(seed, P)
        else:
            s["h"] = _residual(seed, P)
            pf.pos[:P].copy_(torch.arange(pos0, pos0 + P, dtype=torch.int32))
        return s
    if kind == "product":
        n, k = MATS[case["mat"]]
        T = case["T"]
        qs, d = _planes(*_q4(_gen(seed, 2), n, k))
        xq, xds = _q8(_activations(seed, T, k))
        s = {"kind": kind, "swiglu": case["mat"] == "gate_up", "n": n, "k": k, "T": T, "qs": qs, "d": d, "xq": xq,
             "xds": xds}
        if s["swiglu"]:
            s["oq"] = torch.zeros(T, n // 2, dtype=torch.int8, device=DEV)
            s["ods"] = torch.zeros(T, n // 64, 2, dtype=torch.float16, device=DEV)
        else:
            s["y"] = torch.zeros(T, n, dtype=torch.float32, device=DEV)
        return s
    if kind == "attn":
        P, pos0 = case["P"], case["pos0"]
        k, v = _context(seed, 0, 1)
        table = torch.from_numpy(np.random.default_rng([int(seed), 9]).permutation(MAXLEN // PAGE).astype(np.int32)).to(DEV)
        kc = torch.zeros(MAXLEN // PAGE, NKV, PAGE, HD, dtype=torch.float16, device=DEV)
        vc = torch.zeros_like(kc)
        _fill(kc, table[None], k)
        _fill(vc, table[None], v)
        nbytes = call("q355_attn_prefill_ws_bytes", P, MAXLEN, NH, NKV)
        return {"kind": kind, "P": P, "pos0": pos0, "kc": kc, "vc": vc, "table": table, "q": _queries(seed, P),
                "ws": torch.zeros((nbytes + 3) // 4, dtype=torch.float32, device=DEV),
                "out": torch.zeros(P, NH * HD, dtype=torch.float32, device=DEV)}
    assert kind == "head"
    T = case["T"]
    s = {"kind": kind, "T": T, "planes": _q6_planes(), "y": torch.zeros(T, V, dtype=torch.float32, device=DEV)}
    if T == 1:
        s["h"] = _residual(seed, 1)
        s["norm"] = torch.ones(H, dtype=torch.float32, device=DEV)
        parts = call("q355_head_nparts", V)
    else:
        s["xq"], s["xds"] = _q8(_activations(seed, T, H))
        parts = call("q355_mmq_nparts", V)
    s["pmax"] = torch.zeros(T, parts, dtype=torch.float32, device=DEV)
    s["pidx"] = torch.zeros(T, parts, dtype=torch.int32, device=DEV)
    return s


def _queries(seed, P):
    return torch.randn(P, NH * HD, generator=_gen(seed, 13), device=DEV).to(torch.float16)


# ---- one pass --------------------------------------------------------------------------------------

def run(s):
    kind = s["kind"]
    if kind in ("decode", "batched"):
        dec = s["dec"]
        dec.tok.copy_(s["tok"])                             # the step feeds its own token and position back
        dec.pos.copy_(s["pos"])
        dec.graph.replay()
        return {"logits": dec.logits}
    if kind == "prefill":
        s["pf"].chunk(s["ids"], s["pos0"])
        dec = s["dec"]
        return {"logits": dec.logits, "k": dec.kc, "v": dec.vc}
    if kind == "layer":
        pf, P = s["pf"], s["P"]
        pf.h[:P].copy_(s["h"])
        pf.layer(0, P, s["pos0"])
        return {"h": pf.hidden_f64(P), "k": s["dec"].kc[0], "v": s["dec"].vc[0]}
    if kind == "product":
        sw = s["swiglu"]
        call("q355_mmq_q4_0_q8_1", ptr(s["qs"]), ptr(s["d"]), s["n"], s["k"], ptr(s["xq"]), ptr(s["xds"]), s["T"],
             7 if sw else 0, None if sw else ptr(s["y"]), None, ptr(s["oq"]) if sw else None,
             ptr(s["ods"]) if sw else None, None, None)
        return {"q": s["oq"], "ds": s["ods"]} if sw else {"y": s["y"]}
    if kind == "attn":
        call("q355_attn_prefill", ptr(s["q"]), ptr(s["kc"]), ptr(s["vc"]), ptr(s["table"]), s["pos0"], s["P"], NH, NKV,
             SCALE, ptr(s["out"]), ptr(s["ws"]), s["ws"].numel() * 4)
        return {"out": s["out"]}
    lo, hi, sc, d = s["planes"]
    if s["T"] == 1:
        call("q355_head_logits_q6k", ptr(lo), ptr(hi), ptr(sc), ptr(d), V, H, ptr(s["h"]), ptr(s["norm"]), 1e-6,
             ptr(s["y"]), ptr(s["pmax"]), ptr(s["pidx"]), 1)
    else:
        call("q355_mmq_q6k_logits", ptr(lo), ptr(hi), ptr(sc), ptr(d), V, H, ptr(s["xq"]), ptr(s["xds"]), s["T"],
             ptr(s["y"]), ptr(s["pmax"]), ptr(s["pidx"]))
    return {"logits": s["y"], "pmax": s["pmax"]}


# ---- what a pass cannot do without -------------------------------------------------------------------

def _layer_work(T, keys, kv_bytes):
    """One layer for T tokens that attend to `keys` keys in all, reading kv_bytes of K and V."""
    wts = sum(n * k for n, k in MATS.values())
    return wts * 0.5625 + kv_bytes + T * NKV * HD * 4, 2 * wts * T + 4 * HD * NH * keys


def work(case):
    kind = case["kind"]
    kv = NKV * HD * 2 * 2                                   # K and V of one position, bytes
    if kind == "decode":
        n = case["pos"] + 1
        b, f = _layer_work(1, n, n * kv)
        return {"bytes": LAYERS * b + V * H * 0.5625 + V * 4, "flops": LAYERS * f + 2 * V * H}
    if kind == "batched":
        B = case["B"]
        n = B * (256 + MAXLEN) // 2
        b, f = _layer_work(B, n, n * kv)
        return {"bytes": LAYERS * b + V * H * 0.5625 + B * V * 4, "flops": LAYERS * f + 2 * V * H * B}
    if kind in ("prefill", "layer", "attn"):
        P, pos0 = case["P"], case["pos0"]
        keys = P * pos0 + P * (P + 1) // 2
        if kind == "attn":
            return {"bytes": (pos0 + P) * kv + P * NH * HD * (2 + 4), "flops": 4 * HD * NH * keys}
        b, f = _layer_work(P, keys, pos0 * kv)
        if kind == "layer":
            return {"bytes": b + P * H * (8 + 8), "flops": f}
        return {"bytes": LAYERS * b + V * H * 0.5625 + V * 4 + P * 4, "flops": LAYERS * f + 2 * V * H}
    if kind == "product":
        n, k = MATS[case["mat"]]
        T = case["T"]
        out = n // 2 * 1.125 if case["mat"] == "gate_up" else n * 4
        return {"bytes": n * k * 0.5625 + T * k * 1.125 + T * out, "flops": 2 * n * k * T}
    T = case["T"]
    return {"bytes": V * H * 0.8203125 + T * H * 1.125 + T * V * 4, "flops": 2 * V * H * T}


def tolerance(case):
    # A Q8_1 code of a layer input that falls on the other side of a rounding step moves what follows by 1/127 of its
    # block's largest value; last-bit differences of the fp32 sums and the fp16 probabilities of the prefill
    # attention bring such flips, and each layer adds its own. Each bound is about four times the distance from the
    # 64-bit result that was measured over several seeds (in brackets).
    kind = case["kind"]
    if kind == "decode":
        return {"rel": 1e-7}                                # f64 throughout: fp32 rounding of the logits (2.5e-8)
    if kind == "batched":
        return {"rel": 2.5e-2} if case["act"] == "q8" else {"rel": 2e-2}       # (6.3e-3: one sequence flips; 5e-3)
    if kind == "prefill":
        return {"rel": 1.2e-1}                              # eight layers of flips (3.4e-2)
    if kind == "layer":
        return {"rel": 1.5e-2}                              # (3.9e-3)
    if kind == "product":
        # (scales 5.4e-5, 5e-6 of the codes, a few of a small call's; sums 3e-7)
        return {"rel": 2e-4, "differ": 5e-5} if case["mat"] == "gate_up" else {"rel": 1.2e-6}
    if kind == "attn":
        return {"rel": 8e-4}                                # fp16 probabilities (1.9e-4)
    return {"rel": 5e-7}                                    # fp32 rounding of the logits (1.3e-7)


# ---- the same in 64 bits, from the definitions -------------------------------------------------------

def _dense(b, n, k, act="q8"):
    """GGUF Q4_0 bytes -> float64 [n, k] on the GPU; act "f16": the fp16 values d (q - 8) of that arithmetic."""
    b = torch.from_numpy(b).to(DEV).reshape(n, k // 32, 18)
    d = b[..., :2].contiguous().view(torch.float16).to(torch.float64)
    q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], 2).to(torch.float64) - 8
    w = (d * q).reshape(n, k)
    return w.to(torch.float16).to(torch.float64) if act == "f16" else w


def _deq8(q, ds):
    return (q.to(torch.float64).reshape(q.shape[0], -1, 32) * ds[..., :1].to(torch.float64)).reshape(q.shape[0], -1)


def _operand(x, act):
    return x.to(torch.float16).to(torch.float64) if act == "f16" else _deq8(*_q8(x))


def _rms(h, w):
    return h / torch.sqrt((h * h).mean(1, keepdim=True) + 1e-6) * torch.as_tensor(w, device=DEV, dtype=torch.float64)


def _rope(x, pos):
    inv = 1.0 / (1e6 ** (np.arange(0, HD, 2, dtype=np.float64) / HD))
    ang = pos.cpu().numpy().astype(np.float64)[:, None] * inv[None]
    c, s = (torch.from_numpy(f(ang).astype(np.float32)).to(DEV).to(torch.float64)[:, None] for f in (np.cos, np.sin))
    a, b = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _attend(q, K, Vv, last):
    """q [t, NH, HD], K and Vv [NKV, n, HD]; query t attends to keys 0 .. last[t] -> [t, NH * HD]."""
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    n = int(last.max()) + 1
    mask = torch.arange(n, device=DEV)[None] > last[:, None]
    for h in range(NH):
        k, v = (c[h // (NH // NKV), :n].to(torch.float64) for c in (K, Vv))
        p = torch.softmax((q[:, h] @ k.T * SCALE).masked_fill(mask, -math.inf), 1)
        out[:, h] = p @ v
    return out.reshape(q.shape[0], -1)


def _exact_layer(L, h, pos, K, Vv, seqs, act):
    """h [t, H] float64 at positions pos of sequences seqs (one each, or all of sequence 0); K, Vv [B, NKV, MAXLEN, HD]."""
    t = h.shape[0]
    b64 = lambda a: torch.as_tensor(a, device=DEV, dtype=torch.float64)  # noqa: E731
    x = _operand(_rms(h, L["ln1"]), act)
    q, k, v = (x @ _dense(L["w" + c], n * HD, H, act).T + b64(L["b" + c]) for c, n in (("q", NH), ("k", NKV), ("v", NKV)))
    f16 = lambda a: a.to(torch.float16)                     # one rounding to the cache's type  # noqa: E731
    q = f16(_rope(q.reshape(t, NH, HD), pos)).to(torch.float64)
    K[seqs, :, pos] = f16(_rope(k.reshape(t, NKV, HD), pos))
    Vv[seqs, :, pos] = f16(v.reshape(t, NKV, HD))
    if K.shape[0] == 1:
        att = _attend(q, K[0], Vv[0], pos)
    else:
        att = torch.cat([_attend(q[j:j + 1], K[j], Vv[j], pos[j:j + 1]) for j in range(t)])
    h = h + _operand(att, act) @ _dense(L["wo"], H, NH * HD, act).T
    x = _operand(_rms(h, L["ln2"]), act)
    g, u = (x @ _dense(L[n], FFN, H, act).T for n in ("wg", "wu"))
    return h + _operand(g / (1 + torch.exp(-g)) * u, act) @ _dense(L["wd"], H, FFN, act).T


def _logits(w, h):
    x = _operand(_rms(h, w["norm"]), "q8")
    rows = V // 8
    e = w["embed"].reshape(V, -1)
    return torch.cat([x @ _dense(e[i * rows:(i + 1) * rows].reshape(-1, 18), rows, H).T for i in range(8)], 1)


def _pages(c):
    """[1, NKV, MAXLEN, HD] -> the cache pages of a sequence that owns pages 0, 1, .."""
    return c[0].reshape(NKV, MAXLEN // PAGE, PAGE, HD).transpose(0, 1).contiguous()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("decode", "batched", "prefill", "layer"):
        w, _ = _model()
        act = case.get("act", "q8")
        if kind in ("decode", "batched"):
            B = case.get("B", 1)
            toks = _tokens(seed, B)
            pos = torch.from_numpy(_positions(seed, B) if kind == "batched" else np.array([case["pos"]])).to(DEV).long()
            seqs = torch.arange(B, device=DEV)
        else:
            B, P, pos0 = 1, case["P"], case["pos0"]
            toks = _tokens(seed, P)
            pos = torch.arange(pos0, pos0 + P, device=DEV)
            seqs = torch.zeros(P, dtype=torch.long, device=DEV)
        if kind == "layer":
            h = _residual(seed, P).to(torch.float64) / FIX
        else:
            e = w["embed"].reshape(V, -1)[toks].reshape(-1, 18)
            h = _dense(e, len(toks), H)
        ks, vs = [], []
        for i in range(1 if kind == "layer" else LAYERS):
            K, Vv = _context(seed, i, B)
            if kind in ("prefill", "layer"):
                K[:, :, pos0:] = 0
                Vv[:, :, pos0:] = 0
            h = _exact_layer(w["layers"][i], h, pos, K, Vv, seqs, act)
            if kind in ("prefill", "layer"):
                ks.append(_pages(K))
                vs.append(_pages(Vv))
        if kind == "layer":
            return {"h": h, "k": ks[0], "v": vs[0]}
        if kind == "prefill":
            return {"logits": _logits(w, h[-1:]), "k": ks, "v": vs}
        return {"logits": _logits(w, h)}
    if kind == "product":
        n, k = MATS[case["mat"]]
        q, d = _q4(_gen(seed, 2), n, k)
        W = ((q.to(torch.float64) - 8) * d.to(torch.float64)[..., None]).reshape(n, k)
        y = _deq8(*_q8(_activations(seed, case["T"], k))) @ W.T
        if case["mat"] != "gate_up":
            return {"y": y}
        g, u = y[:, 0::2], y[:, 1::2]                       # rows interleaved gate, up
        oq, ods = _q8(g / (1 + torch.exp(-g)) * u)
        return {"q": oq, "ds": ods}
    if kind == "attn":
        P, pos0 = case["P"], case["pos0"]
        K, Vv = _context(seed, 0, 1)
        q = _queries(seed, P).reshape(P, NH, HD).to(torch.float64)
        return {"out": _attend(q, K[0], Vv[0], torch.arange(pos0, pos0 + P, device=DEV))}
    T = case["T"]
    x = _operand(_rms(_residual(seed, 1).to(torch.float64) / FIX, np.ones(H)), "q8") if T == 1 else _deq8(*_q8(_activations(seed, T, H)))
    v, sc, d = _q6(0)
    y = []
    for i in range(0, V, V // 8):
        r = slice(i, i + V // 8)
        W = (v[r].reshape(-1, H // 16, 16).to(torch.float64) - 32) * sc[r].to(torch.float64)[..., None]
        W = W.reshape(-1, H // 256, 256) * d[r].to(torch.float64)[..., None]
        y.append(x @ W.reshape(-1, H).T)
    y = torch.cat(y, 1)
    if T == 1:
        return {"logits": y, "pmax": None}
    return {"logits": y, "pmax": y.reshape(T, V // 64, 64).amax(2)}
