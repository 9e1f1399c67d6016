"""The work that users of this framework have it do, as cases that can be timed.

Three kinds, each through the entry point that a program calls:

* ``moe``: one MoE layer forward (``MoeLayer.forward``: RmsNorm, router, top-k, experts, combine, residual) on a batch of
  tokens, at the GPT-OSS-20B shape (32 experts), the 120B one (128 experts) and small generic ones; bf16 activations as the
  models run them, f32 activations as the reference's layer takes them.
* ``decoder``: a prompt's cache rows taken over (``cache_load``, what a prefill leaves) and a few decode steps with given
  tokens (scoring, speculative checks, the steady state of generation), logits returned at each step.  The model holds 2 of
  GPT-OSS-20B's 24 layers (one with full attention, one windowed) and a twelfth of its vocabulary, so that every part keeps
  its share of the step.
* ``dequant``: MXFP4 expert matrices unpacked to bf16 or f32 (``mxfp4_dequant``), as a loader for dense use does.

Weights follow the distributions of ``burnext_amd.synth``; the norm scales are not all ones, as in a real checkpoint.
"""
from __future__ import annotations

import math
import pathlib
import sys

import numpy as np
import torch

sys.path.insert(0, str(pathlib.Path(__file__).resolve().parents[1] / "burn-extended_amd"))

DEV = "cuda:0"
ALPHA, LIMIT, EPS = 1.702, 7.0, 1e-5
VOCAB, LAYERS, HEADS, KV_HEADS, HEAD_DIM, CACHE = 16384, 2, 64, 8, 64, 8192
WINDOW, THETA, YARN_FACTOR, YARN_CTX, YARN_ALPHA, YARN_BETA = 128, 150000.0, 32.0, 4096.0, 1.0, 32.0
FP4 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _moe(name, d, f, e, k, tokens, dtype, zipf=False):
    return {"name": name, "kind": "moe", "d": d, "f": f, "experts": e, "topk": k, "tokens": tokens, "dtype": dtype,
            "zipf": zipf}


def _decoder(name, batch, context, steps, kv_bf16=False, experts_bf16=False):
    return {"name": name, "kind": "decoder", "batch": batch, "context": context, "steps": steps, "kv_bf16": kv_bf16,
            "experts_bf16": experts_bf16}


def _dequant(name, experts, rows, cols, dtype, ue8):
    return {"name": name, "kind": "dequant", "experts": experts, "rows": rows, "cols": cols, "dtype": dtype, "ue8": ue8}


def listed():
    return [
        # a small model's layer, the smallest call: launches and latency are all of it
        _moe("tiny_f32_t16", 256, 256, 2, 2, 16, "f32"),
        # one user's next token
        _moe("20b_bf16_t1", 2880, 2880, 32, 4, 1, "bf16"),
        # a small decode batch
        _moe("20b_bf16_t8", 2880, 2880, 32, 4, 8, "bf16"),
        # a server's decode batch, an odd number of users
        _moe("20b_bf16_t45", 2880, 2880, 32, 4, 45, "bf16"),
        # a long prompt with popular and rare experts
        _moe("20b_bf16_t4096_zipf", 2880, 2880, 32, 4, 4096, "bf16", zipf=True),
        # a prompt through a model that keeps its activations in f32, as the reference does
        _moe("20b_f32_t523", 2880, 2880, 32, 4, 523, "f32"),
        # the large model: a server's decode batch, and a chunk of a prompt
        _moe("120b_bf16_t64", 2880, 2880, 128, 4, 64, "bf16"),
        _moe("120b_bf16_t1021", 2880, 2880, 128, 4, 1021, "bf16"),
        # generation: one user with a short context; a batch over a full cache (each step evicts); the largest batch
        # with bf16 cache rows and bf16 expert rows
        _decoder("decode_b1_ctx613", 1, 613, 8),
        _decoder("decode_b8_ctx8192", 8, 8192, 8),
        _decoder("decode_b16_ctx1500_bf16", 16, 1500, 8, kv_bf16=True, experts_bf16=True),
        # eight experts' gate_up matrices for dense use
        _dequant("dequant_20b_w1x8_bf16", 8, 5760, 2880, "bf16", 14),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.random()
    if kind < 0.65:
        d = f = 2880
        e, k = (32, 4) if rng.random() < 0.7 else (128, 4)
        if rng.random() < 0.25:
            d, f = 8 * _log_int(rng, 32, 360), 8 * _log_int(rng, 32, 360)
            e, k = rng.choice([(2, 2), (8, 2), (16, 4), (32, 4)])
        tokens = _log_int(rng, 1, 4096 if e <= 32 else 2048)
        c = _moe("", d, f, e, k, tokens, "bf16" if rng.random() < 0.7 else "f32", zipf=rng.random() < 0.3)
        if c["dtype"] == "f32":
            c["tokens"] = min(tokens, _log_int(rng, 1, 1024))
    elif kind < 0.9:
        c = _decoder("", _log_int(rng, 1, 16), _log_int(rng, 16, 8192), rng.randint(4, 8), rng.random() < 0.4,
                     rng.random() < 0.3)
    else:
        c = _dequant("", rng.randint(1, 8), _log_int(rng, 256, 5760), _log_int(rng, 256, 2880),
                     "bf16" if rng.random() < 0.6 else "f32", rng.choice([0, 14]))
    del c["name"]
    return c


# ---- inputs -------------------------------------------------------------------------------------


def _gen(seed, stream):
    g = torch.Generator(device=DEV)
    g.manual_seed((seed << 8) + stream)
    return g


def _bytes(g, *shape):
    return torch.randint(0, 256, shape, dtype=torch.uint8, device=DEV, generator=g)


def _scales(g, *shape):  # e8m0 bytes 127 - 8 .. 127 - 4
    return torch.randint(119, 124, shape, dtype=torch.uint8, device=DEV, generator=g)


def _normal(g, *shape, std=1.0, mean=0.0, bf16=True):
    t = torch.randn(shape, dtype=torch.float32, device=DEV, generator=g) * std + mean
    return t.bfloat16().float() if bf16 else t


def _uniform(g, bound, *shape):
    return ((torch.rand(shape, dtype=torch.float32, device=DEV, generator=g) * 2 - 1) * bound).bfloat16().float()


def _moe_weights(d, f, e, bf16, zipf, g):
    w = {
        "w1b": _bytes(g, e, 2 * f, (d + 1) // 2), "w1s": _scales(g, e, 2 * f, (d + 31) // 32),
        "w2b": _bytes(g, e, d, (f + 1) // 2), "w2s": _scales(g, e, d, (f + 31) // 32),
        "b1": _normal(g, e, 2 * f, std=0.01, bf16=bf16), "b2": _normal(g, e, d, std=0.01, bf16=bf16),
        "rw": _normal(g, e, d, std=0.02, bf16=bf16), "rb": torch.zeros(e, device=DEV),
        "gamma": _normal(g, d, std=0.1, mean=1.0, bf16=bf16),
    }
    if zipf:  # expert popularity falls about as 1 / rank^1.1 over the tokens
        rank = torch.randperm(e, device=DEV, generator=g) + 1
        w["rb"] = -1.1 * 0.7 * torch.log(rank.float())
        w["rb"] = w["rb"].bfloat16().float() if bf16 else w["rb"]
    return w


def _layer_data(w, k, dtype):
    from burnext_amd import synth
    n = {key: t.cpu().numpy() for key, t in w.items()}
    e, f2, _ = n["w1b"].shape
    return synth.MoeLayerData(n["w2b"].shape[1], f2 // 2, e, k, n["w1b"], n["w1s"], n["w2b"], n["w2s"], n["b1"], n["b2"],
                              n["rw"], n["rb"], dtype, gamma_f32=n["gamma"])


def _tokens(case, seed):
    x = _normal(_gen(seed, 1), case["tokens"], case["d"], bf16=case["dtype"] == "bf16")
    return x.bfloat16() if case["dtype"] == "bf16" else x


def _case_weights(case, seed):
    return _moe_weights(case["d"], case["f"], case["experts"], case["dtype"] == "bf16", case["zipf"], _gen(seed, 0))


def _decoder_weights(seed):
    g, d = _gen(seed, 0), 2880
    qd, kd, bd, bq = HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM, 1 / math.sqrt(2880), 1 / math.sqrt(HEADS * HEAD_DIM)
    return {
        "tok_emb": _normal(g, VOCAB, d), "norm_attn": _normal(g, LAYERS, d, std=0.1, mean=1.0),
        "wq": _uniform(g, bd, LAYERS, qd, d), "bq": _uniform(g, bd, LAYERS, qd), "wk": _uniform(g, bd, LAYERS, kd, d),
        "bk": _uniform(g, bd, LAYERS, kd), "wv": _uniform(g, bd, LAYERS, kd, d), "bv": _uniform(g, bd, LAYERS, kd),
        "wo": _uniform(g, bq, LAYERS, d, qd), "bo": _uniform(g, bq, LAYERS, d), "sinks": _normal(g, LAYERS, HEADS),
        "norm_final": _normal(g, d, std=0.1, mean=1.0), "lm_head": _uniform(g, bd, VOCAB, d),
    }


def _decoder_inputs(case, seed):
    g = _gen(seed, 1)
    rows = (LAYERS, case["batch"], case["context"], KV_HEADS, HEAD_DIM)
    # cached rows as the k / v projections of normalised rows give them (weights U(+-1/sqrt(d)): variance 1/3)
    return {"k": _normal(g, *rows, std=0.58, bf16=False), "v": _normal(g, *rows, std=0.58, bf16=False),
            "tokens": torch.randint(0, VOCAB, (case["steps"], case["batch"]), dtype=torch.int32, device=DEV, generator=g)}


def _bits(t):
    return t.bfloat16().view(torch.int16).cpu().numpy().view(np.uint16)


def prepare(case, seed):
    from burnext_amd import decoder, moe
    if case["kind"] == "moe":
        w = _case_weights(case, seed)
        layer = moe.MoeLayer(_layer_data(w, case["topk"], case["dtype"]), device=0)
        return {"kind": "moe", "layer": layer, "x": _tokens(case, seed)}
    if case["kind"] == "dequant":
        g, c = _gen(seed, 0), case
        desc = moe.QuantLinearMxFp4Desc.for_matrix(c["experts"], c["rows"], c["cols"], c["ue8"])
        return {"kind": "dequant", "desc": desc, "blocks": _bytes(g, c["experts"], c["rows"], desc.bpr),
                "scales": _scales(g, c["experts"], c["rows"], desc.gpr) + c["ue8"],
                "dtype": torch.bfloat16 if c["dtype"] == "bf16" else torch.float32}
    cfg = decoder.GptOssConfig(vocab_size=VOCAB, n_layers=LAYERS, cache_len=CACHE, max_seq_len=2 * CACHE,
                               kv_bf16=case["kv_bf16"], experts_bf16=case["experts_bf16"])
    layers = [_layer_data(_moe_weights(2880, 2880, 32, True, False, _gen(seed, 2 + l)), 4, "bf16") for l in range(LAYERS)]
    data = decoder.DecoderData(cfg=cfg, moe=layers, **{k: _bits(t) for k, t in _decoder_weights(seed).items()})
    model = decoder.GptOssDecoder(data, max_batch=case["batch"])
    return {"kind": "decoder", "model": model, "context": case["context"], **_decoder_inputs(case, seed)}


def run(state):
    if state["kind"] == "moe":
        return state["layer"].forward(state["x"])
    if state["kind"] == "dequant":
        from burnext_amd import moe
        return moe.mxfp4_dequant(state["desc"], state["blocks"], state["scales"], state["dtype"])
    model, pos, outs = state["model"], state["context"], []
    model.cache_load(state["k"], state["v"])
    for s, tok in enumerate(state["tokens"]):
        outs.append(model.decode(tok, pos + s, logits=True))
    return {"next": [o[0] for o in outs], "logits": [o[1] for o in outs]}


# ---- what a pass cannot do without ----------------------------------------------------------------


def _touched(e, k, tokens):  # expected experts with a token, uniform routing
    return e * (1 - (1 - min(k, e) / e) ** tokens)


def _expert_bytes(d, f, sb):
    return 2 * f * ((d + 1) // 2 + (d + 31) // 32) + d * ((f + 1) // 2 + (f + 31) // 32) + (2 * f + d) * sb


def work(case):
    if case["kind"] == "dequant":
        n = case["experts"] * case["rows"]
        c = case["cols"]
        return {"bytes": n * ((c + 1) // 2 + (c + 31) // 32 + c * (2 if case["dtype"] == "bf16" else 4)), "flops": n * c}
    if case["kind"] == "moe":
        d, f, e, k, t = case["d"], case["f"], case["experts"], case["topk"], case["tokens"]
        sb = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": _touched(e, k, t) * _expert_bytes(d, f, sb) + e * (d + 1) * sb + 2 * t * d * sb,
                "flops": 6 * t * k * f * d + 2 * t * e * d}
    b, d, qd, kd = case["batch"], 2880, HEADS * HEAD_DIM, KV_HEADS * HEAD_DIM
    dense = (qd + 2 * kd + qd) * d * 2
    experts = _touched(32, 4, b) * _expert_bytes(d, d, 2)
    el = 2 if case["kv_bf16"] else 4
    full, part = min(case["context"] + case["steps"] // 2, CACHE), min(case["context"] + 1, WINDOW)
    step = LAYERS * (dense + experts) + 2 * b * kd * el * (full + part) + VOCAB * d * 2 + b * VOCAB * 4
    flops = b * (LAYERS * (2 * (2 * qd + 2 * kd) * d + 6 * 4 * d * d) + 4 * qd * (full + part) + 2 * VOCAB * d)
    load = 2 * LAYERS * b * case["context"] * kd * (4 + el)  # the caller's f32 rows read, the cache's written
    return {"bytes": case["steps"] * step + load, "flops": case["steps"] * flops}


def tolerance(case):
    if case["kind"] == "dequant":
        return "exact"  # every value is a power of two times an e2m1 code
    # measured against exact(): bf16 layers 0.0034 (decode sizes) to 0.0065 (prefill sizes, activations in two short terms),
    # f32 layers 4.5e-6; f32 decoders 9e-6, with bf16 cache rows and expert rows 0.0022
    if case["kind"] == "moe":
        return {"rel": 1.5e-2} if case["dtype"] == "bf16" else {"rel": 2e-5}
    if case["kv_bf16"] or case["experts_bf16"]:
        return {"rel": 8e-3, "max": 0.05, "differ": 0.01}
    return {"rel": 4e-5, "differ": 0.01}


# ---- the same in 64 bits ----------------------------------------------------------------------------


def _dequant64(blocks, scales, cols, ue8=0):
    lut = torch.tensor(FP4, dtype=torch.float64, device=DEV)
    n = blocks.shape[0]
    codes = torch.stack((blocks & 15, blocks >> 4), dim=-1).reshape(n, -1)[:, :cols]
    exp = ((scales.int() - ue8) & 255).double() - 127
    return lut[codes.long()] * torch.exp2(exp).repeat_interleave(32, dim=1)[:, :cols]


def _rms64(x, gamma):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * gamma


def _moe64(x, w, k, round_rows=False):
    xn = _rms64(x, w["gamma"].double())
    logits = xn @ w["rw"].double().t() + w["rb"].double()
    top, idx = torch.topk(logits, k, dim=1)
    p = torch.softmax(top, dim=1)
    d, f = w["w2b"].shape[1], w["w1b"].shape[1] // 2
    rows = xn.float().bfloat16().double() if round_rows else xn
    y = x.clone()
    for e in range(w["w1b"].shape[0]):
        t, slot = torch.nonzero(idx == e, as_tuple=True)
        if t.numel() == 0:
            continue
        h = rows[t] @ _dequant64(w["w1b"][e], w["w1s"][e], d).t() + w["b1"][e].double()
        g, l = h[:, 0::2].clamp(max=LIMIT), h[:, 1::2].clamp(-LIMIT, LIMIT)
        a = g * torch.sigmoid(ALPHA * g) * (l + 1)
        a = a.float().bfloat16().double() if round_rows else a
        o = a @ _dequant64(w["w2b"][e], w["w2s"][e], f).t() + w["b2"][e].double()
        y.index_add_(0, t, o * p[t, slot, None])
    return y


def _rope64(x, pos):  # heads [b, h, d]: head h is rotated at pos + h (the reference takes the head axis as the sequence)
    d, h = x.shape[2], x.shape[1]
    i = np.arange(d // 2)
    inv = (1.0 / THETA ** (2.0 * i / d)).astype(np.float32).astype(np.float64)
    lo = d * math.log(YARN_CTX / (YARN_BETA * 2 * math.pi)) / math.log(THETA)
    hi = d * math.log(YARN_CTX / (YARN_ALPHA * 2 * math.pi)) / math.log(THETA)
    r = np.clip((2 * i - lo) / (hi - lo), 0, 1)
    inv = (inv / YARN_FACTOR * (1 - r) + inv * r).astype(np.float32)
    angle = (np.arange(pos, pos + h, dtype=np.float32)[:, None] * inv).astype(np.float64)  # the table's f32 angle
    conc = 0.1 * math.log(YARN_FACTOR) + 1
    c, s = (torch.tensor(v * conc, device=DEV) for v in (np.cos(angle), np.sin(angle)))
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack((a * c - b * s, b * c + a * s), dim=-1).flatten(2)


def _attend64(q, k, v, sinks):  # q [b, heads, d], k and v [b, n, kv heads, d]
    b, g = q.shape[0], HEADS // KV_HEADS
    out = torch.empty_like(q)
    for i in range(b):
        for h in range(KV_HEADS):
            s = q[i, h * g:(h + 1) * g] @ k[i, :, h].t()
            s = torch.cat((s, sinks[h * g:(h + 1) * g, None]), dim=1)
            out[i, h * g:(h + 1) * g] = torch.softmax(s, dim=1)[:, :-1] @ v[i, :, h]
    return out.flatten(1)


def _decoder64(case, seed):
    w = {key: t.double() for key, t in _decoder_weights(seed).items()}
    moes = [_moe_weights(2880, 2880, 32, True, False, _gen(seed, 2 + l)) for l in range(LAYERS)]
    inp, b = _decoder_inputs(case, seed), case["batch"]
    kept = (lambda t: t.float().bfloat16().double()) if case["kv_bf16"] else (lambda t: t.double())
    ks, vs = [kept(t) for t in inp["k"]], [kept(t) for t in inp["v"]]
    logits = []
    for s, tok in enumerate(inp["tokens"]):
        pos = case["context"] + s
        h = w["tok_emb"][tok.long()]
        for l in range(LAYERS):
            xn = _rms64(h, w["norm_attn"][l])
            q, k, v = (xn @ w["w" + n][l].t() + w["b" + n][l] for n in "qkv")
            q, k = _rope64(q.view(b, HEADS, HEAD_DIM), pos), _rope64(k.view(b, KV_HEADS, HEAD_DIM), pos)
            ks[l] = torch.cat((ks[l], kept(k)[:, None]), dim=1)[:, -CACHE:]
            vs[l] = torch.cat((vs[l], kept(v.view(b, 1, KV_HEADS, HEAD_DIM))), dim=1)[:, -CACHE:]
            n = ks[l].shape[1] if l % 2 == 0 else WINDOW
            o = _attend64(q, ks[l][:, -n:], vs[l][:, -n:], w["sinks"][l])
            h = _moe64(h + o @ w["wo"][l].t() + w["bo"][l], moes[l], 4, case["experts_bf16"])
        logits.append(_rms64(h, w["norm_final"]) @ w["lm_head"].t())
    return {"next": [None] * len(logits), "logits": logits}


def exact(case, seed):
    if case["kind"] == "moe":
        return _moe64(_tokens(case, seed).double(), _case_weights(case, seed), min(case["topk"], case["experts"]))
    if case["kind"] == "dequant":
        g, c = _gen(seed, 0), case
        blocks = _bytes(g, c["experts"], c["rows"], (c["cols"] + 1) // 2)
        scales = _scales(g, c["experts"], c["rows"], (c["cols"] + 31) // 32) + c["ue8"]
        return _dequant64(blocks.flatten(0, 1), scales.flatten(0, 1), c["cols"], c["ue8"])
    return _decoder64(case, seed)
