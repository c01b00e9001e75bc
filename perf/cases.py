"""The work a program has this library do, as cases that can be timed.

Each case is one pass through the public entry points of rustyllm_amd.hip, with
host arrays where the entry point takes host arrays and device tensors where it
takes device addresses:

  matvec     one weight matrix times one activation (Weight::matvec_into)
  ffn        the fused Q4_K/Q4_K/Q6_K feed-forward block
  moe        the routed gpt-oss feed-forward block
  attention  decode attention on device buffers
  experts    the routed expert product of a prefill, on device buffers
  batch      one K-quant matrix times a batch of activations
  prefill    the resident decoder takes a prompt and returns its first token
  decode     the resident decoder generates tokens after a cached prefix

Shapes are this repository's own model configurations (rustyllm_amd.synth);
weights are its synthetic N(0, 0.02) tensors.  The resident models hold fewer
layers than the full configurations, and every second layer shares its host
bytes with an earlier one (the decoder keeps a device copy of its own per
layer).  The weights and the decoder are what a program keeps; activations,
prompts, queries and caches come from the seed.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from rustyllm_amd import hip, synth

Q8_0, Q4_K, Q6_K, MXFP4 = 8, 12, 14, 39
BLOCK = {Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210), MXFP4: (32, 17)}
DEV = "cuda:0"

# layers kept of each configuration, and the positions its cache holds
MODELS = {
    "llama3-8b-q4km": (6, 8192),
    "qwen2.5-14b-q4km": (4, 8192),
    "tinyllama-1.1b-q8_0": (6, 2304),
    "gpt-oss-20b": (4, 8192),
}
# (query heads, kv heads, head dim) of the configurations
HEADS = {"llama3-8b": (32, 8, 128), "qwen2.5-14b": (40, 8, 128), "tinyllama": (32, 4, 64), "gpt-oss": (64, 8, 64)}
WINDOW = 128


# ---- the cases ---------------------------------------------------------------------
def listed():
    return [
        # the smallest projection of a small model: launches and copies
        dict(name="matvec-q8_0-256x2048", kind="matvec", type=Q8_0, rows=256, cols=2048),
        # the largest single matrix of a decode step, an 8B model's output head
        dict(name="matvec-q6k-head", kind="matvec", type=Q6_K, rows=128256, cols=4096),
        # a whole feed-forward block of an 8B model in one call
        dict(name="ffn-8b", kind="ffn", dim=4096, hidden=14336),
        # the routed feed-forward block of gpt-oss-20b
        dict(name="moe-20b", kind="moe", dim=2880, hidden=2880, experts=32, top_k=4),
        # decode attention of an 8B model at its usual context, an odd length
        dict(name="attn-8b-ctx4097", kind="attention", heads="llama3-8b", ctx=4097, ring=False),
        # gpt-oss's sliding-window layers: sinks and a wrapped ring
        dict(name="attn-20b-window", kind="attention", heads="gpt-oss", ctx=5000, ring=True),
        # a short prompt's tokens through one projection
        dict(name="batch-q4k-37", kind="batch", type=Q4_K, rows=14336, cols=4096, tokens=37),
        # 250 prompt tokens through one expert tensor of gpt-oss-20b
        dict(name="experts-20b-1000", kind="experts", experts=32, top_k=4, rows=2880, cols=2880, tokens=250,
             per_pair=False, mfma=False),
        # time to first token of a 512-token prompt, 8B shape
        dict(name="prefill-8b-512", kind="prefill", model="llama3-8b-q4km", tokens=512),
        # ... and of a longer, ragged one through the gpt-oss-20b shape
        dict(name="prefill-20b-1001", kind="prefill", model="gpt-oss-20b", tokens=1001),
        # greedy generation at the context the throughput benchmark uses
        dict(name="decode-8b-ctx4096", kind="decode", model="llama3-8b-q4km", ctx=4096, tokens=16, bf16=False),
        dict(name="decode-20b-ctx4096", kind="decode", model="gpt-oss-20b", ctx=4096, tokens=16, bf16=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "ffn", "moe", "attention", "attention", "experts", "batch", "prefill",
                       "prefill", "prefill", "decode", "decode"])
    if kind == "matvec":
        t = rng.choice([Q8_0, Q4_K, Q6_K, MXFP4])
        cols = max(1, _log(rng, 256, 14336) // BLOCK[t][0]) * BLOCK[t][0]
        return dict(kind=kind, type=t, rows=_log(rng, 64, min(131072, 128256 * 4096 // cols)), cols=cols)
    if kind == "ffn":
        dim = 256 * _log(rng, 2, 24)
        return dict(kind=kind, dim=dim, hidden=256 * rng.randint(dim // 256, 3 * dim // 256))
    if kind == "moe":
        dim = 32 * rng.randint(5, 90)
        return dict(kind=kind, dim=dim, hidden=32 * rng.randint(3, 90), experts=rng.randint(6, 32),
                    top_k=rng.randint(2, 4))
    if kind == "attention":
        heads = rng.choice(sorted(HEADS))
        return dict(kind=kind, heads=heads, ctx=_log(rng, 16, 28000), ring=heads == "gpt-oss" and rng.random() < 0.6)
    if kind == "experts":
        return dict(kind=kind, experts=rng.randint(6, 32), top_k=rng.randint(2, 4), rows=rng.randint(96, 2880),
                    cols=32 * rng.randint(3, 90), tokens=_log(rng, 3, 256), per_pair=rng.random() < 0.5,
                    mfma=rng.random() < 0.25)
    if kind == "batch":
        t = rng.choice([Q4_K, Q6_K])
        return dict(kind=kind, type=t, rows=_log(rng, 256, 14336), cols=256 * _log(rng, 2, 56),
                    tokens=_log(rng, 2, 300))
    if kind == "prefill":
        model = rng.choice(["llama3-8b-q4km", "qwen2.5-14b-q4km", "gpt-oss-20b"])
        return dict(kind=kind, model=model, tokens=_log(rng, 4, 1000 if model == "gpt-oss-20b" else 2000))
    model = rng.choice(sorted(MODELS))
    return dict(kind=kind, model=model, ctx=_log(rng, 16, MODELS[model][1] - 64), tokens=rng.randint(4, 16),
                bf16=model in ("llama3-8b-q4km", "qwen2.5-14b-q4km") and rng.random() < 0.3)


# ---- weights and the resident decoder, kept between passes --------------------------
_KEPT = {}  # the weights of the case in hand
_MODEL = {}  # host model by name (one at a time)
_LIVE = {}  # the configured decoder: "key", "res", "prefix" (positions cached), "ring" (its cached slots)


def _kept(key, make):
    if _KEPT.get("key") != key:
        # device copies are cached by host address: drop them before the memory goes
        hip.weight_cache_clear()
        _KEPT.clear()
        _KEPT.update(key=key, value=make())
    return _KEPT["value"]


def _rows(t, seed, rows, cols):
    return synth.normal_quantized(t, seed, rows, cols, 0.02)


def _model(name):
    if name not in _MODEL:
        _MODEL.clear()
        layers = MODELS[name][0]
        if name == "gpt-oss-20b":
            cfg = dict(synth.GPTOSS_CONFIGS[name], n_layers=1, vocab=256)
            m = synth.make_gptoss(cfg, seed=1234)
            vocab, emb_t, out_t = synth.GPTOSS_CONFIGS[name]["vocab"], Q8_0, Q8_0
        else:
            cfg = dict(synth.CONFIGS[name], n_layers=2, vocab=256)
            m = synth.make_model(cfg, seed=1234)
            vocab = synth.CONFIGS[name]["vocab"]
            emb_t, out_t = (Q8_0, Q8_0) if cfg["quant"] == "q8_0" else (Q4_K, Q6_K)
        dim = m["config"]["dim"]
        m["config"].update(n_layers=layers, vocab=vocab)
        m["layers"] = [m["layers"][i % len(m["layers"])] for i in range(layers)]
        emb = _rows(emb_t, 77, 8192, dim).reshape(8192, -1)
        m["token_embd"] = (np.resize(emb, (vocab, emb.shape[1])).reshape(-1), emb_t)
        m["output"] = (_rows(out_t, 78, vocab, dim), out_t)
        _MODEL[name] = m
    return _MODEL[name]


def _resident(name, bf16=False):
    if _LIVE.get("key") != (name, bf16):
        _LIVE.clear()
        m = _model(name)
        if name == "gpt-oss-20b":
            res = hip.ResidentGptOss(m, MODELS[name][1])
        else:
            res = hip.Resident(m, MODELS[name][1], kv_bf16=bf16)
        _LIVE.update(key=(name, bf16), res=res, prefix=0, ring=None)
    return _LIVE["res"]


def _cached_prefix(res, model, ctx):
    """A shared prefix in the cache at positions 0..ctx-2 (a ring cache's slots
    are put back, since generated tokens overwrite them)."""
    if ctx < 2:
        return
    ring = "window" in model["config"]
    if _LIVE["prefix"] != ctx:
        toks = synth.token_ids(4321, ctx - 1, model["config"]["vocab"]).astype(np.int32)
        res.generate(toks, 0, want_logits=False)
        _LIVE["prefix"] = ctx
        if ring:
            _LIVE["ring"] = [(l, w, res.kv_read(l, w, 0, res.slots)) for l in range(model["config"]["n_layers"])
                             for w in (0, 1)]
    elif ring:
        for l, w, data in _LIVE["ring"]:
            res.kv_write(l, w, 0, data)


def _need(ok):
    if not ok:
        raise RuntimeError("the call was not handled")


def prepare(case, seed):
    k = case["kind"]
    rng = np.random.default_rng(seed)
    if k == "matvec":
        w = _kept((k, case["type"], case["rows"], case["cols"]), lambda: _rows(case["type"], 11, case["rows"], case["cols"]))
        return dict(case, w=w, x=rng.standard_normal(case["cols"], np.float32), out=np.zeros(case["rows"], np.float32))
    if k == "ffn":
        d, h = case["dim"], case["hidden"]
        w = _kept((k, d, h), lambda: (_rows(Q4_K, 21, h, d), _rows(Q4_K, 22, h, d), _rows(Q6_K, 23, d, h)))
        return dict(case, w=w, x=rng.standard_normal(d, np.float32), out=np.zeros(d, np.float32))
    if k == "moe":
        return dict(case, w=_kept((k, case["dim"], case["hidden"], case["experts"]), lambda: _moe_weights(case)),
                    x=rng.standard_normal(case["dim"], np.float32))
    if k == "attention":
        nh, nkv, hd = HEADS[case["heads"]]
        slots = min(WINDOW, case["ctx"]) if case["ring"] else case["ctx"]
        g = torch.Generator(DEV).manual_seed(seed)
        s = dict(case, q=torch.randn(nh * hd, generator=g, device=DEV), k=torch.randn(slots, nkv * hd, generator=g, device=DEV),
                 v=torch.randn(slots, nkv * hd, generator=g, device=DEV), out=torch.zeros(nh * hd, device=DEV), sinks=None)
        if case["heads"] == "gpt-oss":
            s["sinks"] = torch.randn(nh, generator=g, device=DEV)
        return s
    if k == "experts":
        e, rows, cols, T, top = case["experts"], case["rows"], case["cols"], case["tokens"], case["top_k"]
        w, stride = _kept((k, e, rows, cols), lambda: _expert_tensor(e, rows, cols))
        g = torch.Generator(DEV).manual_seed(seed)
        x = torch.randn(T * top if case["per_pair"] else T, cols, generator=g, device=DEV)
        sel = np.stack([rng.choice(e, size=top, replace=False) for _ in range(T)]).astype(np.int32).reshape(-1)
        return dict(case, w=w, stride=stride, x=x, sel=torch.from_numpy(sel).to(DEV),
                    y=torch.zeros(T * top, rows, device=DEV))
    if k == "batch":
        w = _kept((k, case["type"], case["rows"], case["cols"]), lambda: _rows(case["type"], 31, case["rows"], case["cols"]))
        return dict(case, w=w, x=rng.standard_normal((case["tokens"], case["cols"]), np.float32),
                    out=np.zeros((case["tokens"], case["rows"]), np.float32))
    model = _model(case["model"])
    vocab = model["config"]["vocab"]
    if k == "prefill":
        res = _resident(case["model"])
        _LIVE["prefix"] = 0
        return dict(case, res=res, prompt=synth.token_ids(seed, case["tokens"], vocab).astype(np.int32))
    res = _resident(case["model"], case["bf16"])
    _cached_prefix(res, model, case["ctx"])
    return dict(case, res=res, prompt=synth.token_ids(seed, 1, vocab).astype(np.int32))


def _moe_weights(case):
    d, h, e = case["dim"], case["hidden"], case["experts"]
    vec = lambda s, r, c: synth.normal_f32(s, r, c, 0.02)  # noqa: E731
    return dict(router=_rows(Q8_0, 41, e, d), router_bias=vec(42, 1, e).reshape(-1),
                experts=(_rows(MXFP4, 43, e * h, d), _rows(MXFP4, 44, e * h, d), _rows(MXFP4, 45, e * d, h)),
                biases=(vec(46, e, h), vec(47, e, h), vec(48, e, d)))


def _expert_tensor(e, rows, cols):
    rb = cols // 32 * 17
    stride = (rb + 15) // 16 * 16
    w = np.zeros((e * rows, stride), np.uint8)
    w[:, :rb] = _rows(MXFP4, 51, e * rows, cols).reshape(e * rows, rb)
    return torch.from_numpy(w).to(DEV), stride


# ---- one pass -----------------------------------------------------------------------
def run(s):
    k = s["kind"]
    if k == "matvec":
        _need(hip.matvec_into(s["type"], s["w"], s["x"], s["rows"], s["cols"], s["out"]))
        return s["out"]
    if k == "ffn":
        _need(hip.q4k_q4k_q6k_ffn_into(*s["w"], s["x"], s["dim"], s["hidden"], s["dim"], s["hidden"], s["out"]))
        return s["out"]
    if k == "moe":
        w = s["w"]
        got = hip.moe_ffn(s["x"], w["router"], Q8_0, w["router_bias"], w["experts"], MXFP4, s["hidden"], w["biases"],
                          s["top_k"])
        _need(got is not None)
        return got
    if k == "attention":
        nh, nkv, hd = HEADS[s["heads"]]
        start = max(0, s["ctx"] - WINDOW) if s["ring"] else 0
        sinks = s["sinks"].data_ptr() if s["sinks"] is not None else 0
        _need(hip.attention_noalloc_dev(s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(), sinks,
                                        s["out"].data_ptr(), nh, nh // nkv, hd, hd, nkv * hd, nkv * hd,
                                        s["k"].shape[0], start, s["ctx"] - 1, 1.0 / math.sqrt(hd)))
        return s["out"]
    if k == "experts":
        _need(hip.mxfp4_experts_dev(s["w"].data_ptr(), s["stride"], s["rows"] * s["stride"], s["experts"], s["rows"],
                                    s["cols"], s["x"].data_ptr(), s["cols"], s["per_pair"], s["top_k"],
                                    s["sel"].data_ptr(), s["sel"].numel(), s["y"].data_ptr(), s["rows"], s["mfma"]))
        return s["y"]
    if k == "batch":
        _need(hip.kquant_matvec_batch_into(s["type"], s["w"], s["rows"], s["cols"], s["x"], s["out"]))
        return s["out"]
    if k == "prefill":
        toks, logits = s["res"].generate(s["prompt"], 1)
        return {"token": toks, "logits": logits}
    toks, logits = s["res"].generate(s["prompt"], s["tokens"], start_pos=s["ctx"] - 1)
    return {"tokens": toks, "logits": logits}


# ---- what a pass cannot do without --------------------------------------------------
def _bytes(t, rows, cols):
    return rows * (cols // BLOCK[t][0]) * BLOCK[t][1]


def _model_work(name):
    """Weight bytes and multiply-adds of one token per layer and of the head;
    for gpt-oss the routed part of a layer apart."""
    c = synth.GPTOSS_CONFIGS[name] if name == "gpt-oss-20b" else synth.CONFIGS[name]
    dim, hd, nh, nkv, hid = c["dim"], c["head_dim"], c["n_heads"], c["n_kv_heads"], c["hidden_dim"]
    attn = [((nh + 2 * nkv) * hd, dim), (dim, nh * hd)]
    kv = 2 * nkv * hd * 4
    if name == "gpt-oss-20b":
        dense = sum(_bytes(Q8_0, r, k) for r, k in attn) + _bytes(Q8_0, c["n_experts"], dim)
        one = 3 * _bytes(MXFP4, hid, dim)
        macs = sum(r * k for r, k in attn) + c["n_experts"] * dim + c["top_k"] * 3 * hid * dim
        return c, dense, one, macs, kv, _bytes(Q8_0, c["vocab"], dim)
    dense = 0
    for l in (0, 1):
        tq, tk, tv, to, tg, tu, td = synth.layer_types(c["quant"], l)
        dense += (_bytes(tq, nh * hd, dim) + _bytes(tk, nkv * hd, dim) + _bytes(tv, nkv * hd, dim) +
                  _bytes(to, dim, nh * hd) + _bytes(tg, hid, dim) + _bytes(tu, hid, dim) + _bytes(td, dim, hid)) / 2
    macs = sum(r * k for r, k in attn) + 3 * hid * dim
    return c, dense, 0, macs, kv, _bytes(Q8_0 if c["quant"] == "q8_0" else Q6_K, c["vocab"], dim)


def work(case):
    k = case["kind"]
    if k in ("matvec", "batch"):
        T, r, c = case.get("tokens", 1), case["rows"], case["cols"]
        return {"bytes": _bytes(case["type"], r, c) + 4 * T * (r + c), "flops": 2 * T * r * c}
    if k == "ffn":
        d, h = case["dim"], case["hidden"]
        return {"bytes": 2 * _bytes(Q4_K, h, d) + _bytes(Q6_K, d, h) + 8 * d, "flops": 6 * d * h}
    if k == "moe":
        d, h, e, top = case["dim"], case["hidden"], case["experts"], case["top_k"]
        return {"bytes": _bytes(Q8_0, e, d) + top * (2 * _bytes(MXFP4, h, d) + _bytes(MXFP4, d, h) + 4 * (2 * h + d)) + 8 * d,
                "flops": 2 * (e * d + top * 3 * d * h)}
    if k == "attention":
        nh, nkv, hd = HEADS[case["heads"]]
        n = min(WINDOW, case["ctx"]) if case["ring"] else case["ctx"]
        return {"bytes": 8 * n * nkv * hd + 8 * nh * hd, "flops": 4 * n * nh * hd}
    if k == "experts":
        T, top, r, c = case["tokens"], case["top_k"], case["rows"], case["cols"]
        used = min(case["experts"], T * top)
        return {"bytes": used * _bytes(MXFP4, r, c) + 4 * T * (top if case["per_pair"] else 1) * c + 4 * T * top * r,
                "flops": 2 * T * top * r * c}
    c, dense, one, macs, kv, head = _model_work(case["model"])
    L, T = MODELS[case["model"]][0], case["tokens"]
    nh, hd, win = c["n_heads"], c["head_dim"], c.get("window", 0)

    def seen(pos):  # positions attended at pos, summed over the layers; bytes of their K and V
        full = sum(pos + 1 if not win or l % 2 else min(pos + 1, win) for l in range(L))
        rows = L * (min(pos + 1, win) if win else pos + 1)
        return full, rows * kv

    esize = 2 if case.get("bf16") else 4
    if k == "prefill":
        used = min(c["n_experts"], T * c["top_k"]) if one else 0
        att = sum(seen(p)[0] for p in range(T))
        return {"bytes": L * (dense + used * one + T * kv) + head + 4 * c["vocab"],
                "flops": 2 * L * macs * T + 4 * att * nh * hd + 2 * c["vocab"] * c["dim"]}
    att = [seen(case["ctx"] - 1 + i) for i in range(T)]
    return {"bytes": T * (L * (dense + (c["top_k"] * one if one else 0)) + head) + sum(b for _, b in att) * esize / 4 + 4 * c["vocab"],
            "flops": 2 * T * (L * macs + c["vocab"] * c["dim"]) + 4 * sum(a for a, _ in att) * nh * hd}


def tolerance(case):
    # Whole models: each product quantizes its activation to int8, so a last-bit
    # change becomes whole quantization steps, and routing flips, a few layers
    # on; against 64 bits the logits are 2 to 8% off.  Single products and
    # attention are 1e-7 to 1.5e-6 off.
    if case["kind"] in ("prefill", "decode"):
        return {"rel": 3e-2, "max": 0.99, "differ": 0.0}
    return {"rel": 6e-6, "max": 3e-4, "differ": 0.0}


# ---- the same results in 64 bits ----------------------------------------------------
def _dequant(t, raw, cols, lead):
    """Rows of quantized blocks (uint8 on the GPU) as float64 [*lead, cols]."""
    b = raw.reshape(-1, BLOCK[t][1])
    half = lambda lo: b[:, lo:lo + 2].contiguous().view(torch.float16).to(torch.float64)  # noqa: E731
    if t == Q8_0:
        v = half(0) * b[:, 2:].contiguous().view(torch.int8).to(torch.float64)
    elif t == MXFP4:
        lut = torch.tensor([0, .5, 1, 1.5, 2, 3, 4, 6, 0, -.5, -1, -1.5, -2, -3, -4, -6], dtype=torch.float64, device=b.device)
        nib = torch.stack([b[:, :16] & 15, b[:, :16] >> 4], 2).reshape(-1, 32)
        v = lut[nib.long()] * torch.exp2(b[:, 16:17].to(torch.float64) - 127)
    elif t == Q4_K:
        s = b[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1).to(torch.float64)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).to(torch.float64)
        qs = b[:, 16:].reshape(-1, 4, 32)
        nib = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).to(torch.float64)
        v = (half(0) * sc)[:, :, None] * nib - (half(2) * mn)[:, :, None]
    else:
        ql, qh = b[:, 0:128].reshape(-1, 2, 64).to(torch.int32), b[:, 128:192].reshape(-1, 2, 32).to(torch.int32)
        q = torch.cat([(ql[:, :, :32] & 15) | ((qh & 3) << 4), (ql[:, :, 32:] & 15) | ((qh >> 2 & 3) << 4),
                       (ql[:, :, :32] >> 4) | ((qh >> 4 & 3) << 4), (ql[:, :, 32:] >> 4) | ((qh >> 6 & 3) << 4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64)
        v = (half(208) * sc)[:, :, None] * (q.reshape(-1, 16, 16) - 32).to(torch.float64)
    return v.reshape(*lead, cols)


def _activation(x, t, cols):
    """What a product of type t multiplies with: the block-quantized int8 form
    (256 elements per scale, in the 32-bit steps that define it) or x itself."""
    if t == MXFP4 or cols % 256:
        return x
    f = x.to(torch.float32).reshape(*x.shape[:-1], -1, 256)
    amax = f.abs().amax(-1, keepdim=True)
    inv = torch.where(amax > 0, torch.tensor(127.0, device=x.device) / amax, torch.zeros_like(amax))
    q = torch.clamp(torch.round(f * inv), -128, 127).to(torch.float64)
    return (q * (amax * np.float32(1.0 / 127.0)).to(torch.float64)).reshape(x.shape)


def _times(x, t, raw, rows, cols):
    """x [T, cols] times the quantized matrix, in pieces of its rows."""
    raw = torch.from_numpy(np.ascontiguousarray(raw)) if isinstance(raw, np.ndarray) else raw
    raw, a, out = raw.reshape(rows, -1), _activation(x, t, cols), []
    for r in range(0, rows, 16384):
        part = raw[r:r + 16384].to(DEV)
        out.append(a @ _dequant(t, part, cols, (part.shape[0],)).T)
    return torch.cat(out, -1)


def _f64(a):
    return torch.from_numpy(np.ascontiguousarray(a)).to(DEV).to(torch.float64)


def _swiglu_oss(g, u):
    g, u = g.clamp(max=7.0), u.clamp(-7.0, 7.0)
    return g / (1 + torch.exp(-1.702 * g)) * (u + 1)


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * _f64(w)


def _rope(x, n, hd, inv, neox, conc=1.0):
    T = x.shape[0]
    x = x.reshape(T, n, hd)
    ang = (torch.arange(T, device=DEV, dtype=torch.float32)[:, None] * torch.from_numpy(inv).to(DEV)).to(torch.float64)
    c, s = (torch.cos(ang) * conc)[:, None], (torch.sin(ang) * conc)[:, None]
    a, b = (x[..., :hd // 2], x[..., hd // 2:]) if neox else (x[..., 0::2], x[..., 1::2])
    y = (a * c - b * s, a * s + b * c)
    return torch.cat(y, -1) if neox else torch.stack(y, -1).reshape(T, n, hd)


def _attend(q, k, v, hd, bias, sinks=None):
    """Causal attention [T, n, hd]; bias [T, T] is added to the scores."""
    T, nh, out = q.shape[0], q.shape[1], []
    for h in range(nh):
        kv = h * k.shape[1] // nh
        s = q[:, h] @ k[:, kv].T.contiguous() / math.sqrt(hd) + bias
        if sinks is not None:
            s = torch.cat([s, sinks[h].expand(T, 1)], 1)
        p = torch.softmax(s, -1)
        out.append((p[:, :T] if sinks is not None else p) @ v[:, kv])
    return torch.stack(out, 1).reshape(T, -1)


def _moe(x, w, types, dim, hidden, top_k):
    """The routed block on [T, dim]; types: (router, experts)."""
    e = len(w["router_bias"])
    r = _times(x, types[0], w["router"], e, dim) + _f64(w["router_bias"])
    val, sel = torch.topk(r, top_k, dim=-1)
    p, out = torch.softmax(val, -1), torch.zeros_like(x)
    gate, up, down = (np.asarray(a).reshape(e, -1) for a in w["experts"])
    gb, ub, db = (_f64(b) for b in w["biases"])
    for i in range(e):
        tok, slot = torch.nonzero(sel == i, as_tuple=True)
        if tok.numel():
            h = _swiglu_oss(_times(x[tok], types[1], gate[i], hidden, dim) + gb[i],
                            _times(x[tok], types[1], up[i], hidden, dim) + ub[i])
            out.index_add_(0, tok, (_times(h, types[1], down[i], dim, hidden) + db[i]) * p[tok, slot][:, None])
    return out, sel, p


def _prompt_logits(name, prompt):
    m = _model(name)
    c, inv = m["config"], np.asarray(m["inv_freq"], np.float32)
    dim, hd, nh, nkv, hid, T = c["dim"], c["head_dim"], c["n_heads"], c["n_kv_heads"], c["hidden_dim"], len(prompt)
    emb, t = m["token_embd"]
    x = _dequant(t, torch.from_numpy(emb.reshape(c["vocab"], -1)[prompt]).to(DEV), dim, (T,))
    pos = torch.arange(T, device=DEV)
    far = pos[:, None] - pos[None, :]
    causal = torch.zeros(T, T, dtype=torch.float64, device=DEV).masked_fill(far < 0, -math.inf)
    for l, L in enumerate(m["layers"]):
        oss = name == "gpt-oss-20b"
        w = [(L[n][0], L[n][1]) for n in ("wq", "wk", "wv", "wo")] if oss else [(a, ty) for a, ty, _ in L["w"]]
        xn = _rms(x, L["attn_norm"], c["eps"])
        q, k, v = (_times(xn, w[i][1], w[i][0], n * hd, dim) for i, n in enumerate((nh, nkv, nkv)))
        if L.get("bq") is not None:
            q, k, v = q + _f64(L["bq"]), k + _f64(L["bk"]), v + _f64(L["bv"])
        conc = float(m.get("concentration", 1.0))
        q, k = _rope(q, nh, hd, inv, c.get("neox", False), conc), _rope(k, nkv, hd, inv, c.get("neox", False), conc)
        bias, sinks = causal, None
        if oss:
            # a ring of `window` slots: odd layers walk it once per pass over the
            # slots, so the position p kept in a slot counts p // window + 1 times
            bias, sinks = causal.masked_fill(far >= c["window"], -math.inf), _f64(L["sinks"])
            if l % 2:
                bias = bias + torch.log((pos // c["window"] + 1).to(torch.float64))[None, :]
        att = _attend(q, k, v.reshape(T, nkv, hd), hd, bias, sinks)
        x = x + _times(att, w[3][1], w[3][0], dim, nh * hd) + (_f64(L["bo"]) if oss else 0)
        if oss:
            xn = _rms(x, L["post_attn_norm"], c["eps"])
            parts = dict(router=L["router"], router_bias=L["router_bias"],
                         experts=(L["gate_exps"], L["up_exps"], L["down_exps"]),
                         biases=(L["gate_exps_bias"], L["up_exps_bias"], L["down_exps_bias"]))
            x = x + _moe(xn, parts, (Q8_0, MXFP4), dim, hid, c["top_k"])[0]
        else:
            xn = _rms(x, L["ffn_norm"], c["eps"])
            h = torch.nn.functional.silu(_times(xn, w[4][1], w[4][0], hid, dim)) * _times(xn, w[5][1], w[5][0], hid, dim)
            x = x + _times(h, w[6][1], w[6][0], dim, hid)
    out, t = m["output"]
    return _times(_rms(x[-1:], m["output_norm"], c["eps"]), t, out, c["vocab"], dim)[0]


def exact(case, seed):
    k = case["kind"]
    if k == "decode":
        return None  # each token depends on the one picked before it
    s = dict(case) if k == "prefill" else prepare(case, seed)
    if k == "matvec":
        return _times(_f64(s["x"])[None], s["type"], s["w"], s["rows"], s["cols"])[0]
    if k == "batch":
        return _times(_f64(s["x"]), s["type"], s["w"], s["rows"], s["cols"])
    if k == "ffn":
        d, h = s["dim"], s["hidden"]
        x = _f64(s["x"])[None]
        hid = torch.nn.functional.silu(_times(x, Q4_K, s["w"][0], h, d)) * _times(x, Q4_K, s["w"][1], h, d)
        return _times(hid, Q6_K, s["w"][2], d, h)[0]
    if k == "moe":
        out, _, p = _moe(_f64(s["x"])[None], s["w"], (Q8_0, MXFP4), s["dim"], s["hidden"], s["top_k"])
        return out[0], None, p[0]
    if k == "attention":
        nh, nkv, hd = HEADS[s["heads"]]
        q, K, V = s["q"].double().reshape(nh, hd), s["k"].double(), s["v"].double()
        K, V = (a.reshape(-1, nkv, hd).transpose(0, 1).repeat_interleave(nh // nkv, 0) for a in (K, V))
        sc = (K * q[:, None]).sum(-1) / math.sqrt(hd)
        if s["sinks"] is not None:
            sc = torch.cat([sc, s["sinks"].double()[:, None]], 1)
        p = torch.softmax(sc, -1)[:, :K.shape[1]]
        return (p[:, :, None] * V).sum(1).reshape(-1)
    if k == "experts":
        raw = s["w"].reshape(s["experts"], s["rows"], -1)[:, :, :s["cols"] // 32 * 17]
        sel, out = s["sel"].long(), torch.zeros(s["y"].shape, dtype=torch.float64, device=DEV)
        for e in range(s["experts"]):
            p = torch.nonzero(sel == e)[:, 0]
            if p.numel():
                x = s["x"][p if s["per_pair"] else p // s["top_k"]].double()
                out[p] = _times(x, MXFP4, raw[e].contiguous(), s["rows"], s["cols"])
        return out
    prompt = synth.token_ids(seed, case["tokens"], _model(case["model"])["config"]["vocab"]).astype(np.int64)
    return {"token": None, "logits": _prompt_logits(case["model"], prompt)}
