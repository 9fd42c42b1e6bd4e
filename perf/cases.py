"""Workloads of the decoder / encoder library, as a program that transcribes
audio calls it: single blocks through the op-level entry points on device
tensors, the audio encoder, prefill, and greedy decoding.

Everything is fp32 activations on bf16 weights (the only types the library
takes in earnest: checkpoints are bf16).  A case is a dict of plain values;
`kind` selects the path:

  attn_block   RMSNorm, Q|K|V projections, q/k norm, RoPE, K/V append, causal
               attention, O projection, residual (one decoder layer's first half)
  mlp_block    RMSNorm, gate|up projection, SwiGLU, down projection, residual
  attention    causal GQA attention alone
  head         the tied LM head of `vocab` entries on one row: logits and the greedy index
  encoder      mel [128][frames] -> audio rows on the device
  prefill      rows through a decoder on top of `past` cached positions, then
               one forward whose logits read every position just written
  generate     `steps` greedy tokens from `past` cached positions

`model` is 0 for the 0.6B shape and 1 for the 1.7B shape.  `layers` cuts a
decoder down to that many layers where one layer's work is the point.
"""
import importlib
import math

import numpy as np
import torch

QA = importlib.import_module("qwen-asr_amd")

HEADS, KV_HEADS, HD, VOCAB, EPS, THETA = 16, 8, 128, 151936, 1e-6, 1e6
QD, KVD = HEADS * HD, KV_HEADS * HD
HIDDEN, INTER = (1024, 2048), (3072, 6144)
ENC = ({"d": 896, "layers": 18, "heads": 14, "ffn": 3584, "out": 1024},
       {"d": 1024, "layers": 24, "heads": 16, "ffn": 4096, "out": 2048})
ENC_CH, ENC_CHUNK, ENC_TPC, ENC_WIN, ENC_EPS = 480, 100, 13, 104, 1e-5


def listed():
    return [
        # one generated token's attention half, a host program calling operator by operator: launch latency
        {"name": "attn_block_decode", "kind": "attn_block", "model": 0, "rows": 1, "past": 529},
        # one generated token's MLP half at the larger model: latency, then weight streaming
        {"name": "mlp_block_decode", "kind": "mlp_block", "model": 1, "rows": 1},
        # the attention half over a 30 s segment's prompt (390 audio rows + template)
        {"name": "attn_block_prompt", "kind": "attn_block", "model": 0, "rows": 401, "past": 0},
        # the MLP half over a two-minute segment's prompt at the larger model
        {"name": "mlp_block_prompt", "kind": "mlp_block", "model": 1, "rows": 1515},
        # attention over a long recording's prompt
        {"name": "attention_long", "kind": "attention", "rows": 4096, "past": 0},
        # the LM head of one token at the larger model, with its logits
        {"name": "head", "kind": "head", "model": 1, "vocab": VOCAB},
        # the encoder on a live stream's rolling window (a ragged last chunk)
        {"name": "encoder_window", "kind": "encoder", "model": 1, "frames": 743},
        # the encoder on a 30 s segment
        {"name": "encoder_segment", "kind": "encoder", "model": 0, "frames": 3000},
        # a live stream's next chunk: 31 new rows after the reused prefix
        {"name": "prefill_chunk", "kind": "prefill", "model": 1, "layers": 4, "rows": 31, "past": 993},
        # the whole 0.6B decoder over a 30 s segment's prompt
        {"name": "prefill_prompt", "kind": "prefill", "model": 0, "layers": 28, "rows": 401, "past": 0},
        # a long recording's prompt, a few layers of it
        {"name": "prefill_long", "kind": "prefill", "model": 0, "layers": 4, "rows": 8191, "past": 0},
        # the whole 0.6B decoder's greedy loop after a 30 s prompt
        {"name": "generate", "kind": "generate", "model": 0, "layers": 28, "past": 402, "steps": 24},
    ]


def draw(rng):
    def log_int(lo, hi):
        return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    # the paths a transcription spends its time in come up more often
    kind = rng.choice(["attn_block", "mlp_block", "attention", "head", "encoder", "encoder", "prefill", "prefill",
                       "generate"])
    model = rng.randrange(2)
    if kind == "attn_block":
        rows = 1 if rng.random() < 0.4 else log_int(2, 1515)
        return {"kind": kind, "model": model, "rows": rows, "past": rng.choice([log_int(16, 2048), 0 if rows > 1 else log_int(1, 4096)])}
    if kind == "mlp_block":
        return {"kind": kind, "model": model, "rows": 1 if rng.random() < 0.1 else log_int(2, 1515)}
    if kind == "attention":
        return {"kind": kind, "rows": log_int(2, 4096), "past": rng.choice([0, 0, log_int(16, 1024)])}
    if kind == "head":
        return {"kind": kind, "model": model, "vocab": log_int(16001, VOCAB)}
    if kind == "encoder":
        return {"kind": kind, "model": model, "frames": log_int(60, 3000)}
    if kind == "prefill":
        layers = rng.randint(2, 6)
        return {"kind": kind, "model": model, "layers": layers, "rows": log_int(8, 2048),
                "past": rng.choice([0, log_int(16, 1024)])}
    return {"kind": kind, "model": model, "layers": rng.randint(4, 10), "past": log_int(32, 2000),
            "steps": rng.randint(4, 24)}


# ---------------------------------------------------------------------------
# inputs (on the GPU, from the seed alone)
# ---------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(0x5EED + seed)
    return g


def _normal(g, *shape, std=1.0, mean=0.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).add_(mean)


def _weight(g, *shape, std=0.02):
    return _normal(g, *shape, std=std).to(torch.bfloat16)


def _rope_table(n):
    """the fp32 cos / sin rows [n][128] that a decoder of this family works with: fp32 angles p * theta^(-2i/128)"""
    e = np.arange(HD // 2, dtype=np.float64) * 2.0 / HD
    inv = (np.float32(1.0) / np.power(THETA, e).astype(np.float32)).astype(np.float32)
    a = (np.arange(n, dtype=np.float32)[:, None] * inv[None, :]).astype(np.float64)
    c, s = np.cos(a).astype(np.float32), np.sin(a).astype(np.float32)
    return torch.from_numpy(np.concatenate([c, c], 1)).cuda(), torch.from_numpy(np.concatenate([s, s], 1)).cuda()


def _attn_inputs(c, seed):
    g, D, S, past = _gen(seed), HIDDEN[c["model"]], c["rows"], c["past"]
    cos, sin = _rope_table(past + S)
    # cached rows as earlier calls leave them: normed, rotated keys and plain values
    return {"x": _normal(g, S, D), "w_in": _normal(g, D, std=0.1, mean=1.0),
            "q_norm": _normal(g, HD, std=0.1, mean=1.0), "k_norm": _normal(g, HD, std=0.1, mean=1.0),
            "wq": _weight(g, QD, D), "wk": _weight(g, KVD, D), "wv": _weight(g, KVD, D), "wo": _weight(g, D, QD),
            "k_past": _normal(g, past, KVD), "v_past": _normal(g, past, KVD),
            "cos": cos[past:].contiguous(), "sin": sin[past:].contiguous()}


def _mlp_inputs(c, seed):
    g, D, I = _gen(seed), HIDDEN[c["model"]], INTER[c["model"]]
    return {"x": _normal(g, c["rows"], D), "w_post": _normal(g, D, std=0.1, mean=1.0),
            "gate_up": _weight(g, 2 * I, D), "down": _weight(g, D, I)}


def _attention_inputs(c, seed):
    g, S, n = _gen(seed), c["rows"], c["rows"] + c["past"]
    return {"q": _normal(g, S, QD), "k": _normal(g, n, KVD), "v": _normal(g, n, KVD)}


def _head_inputs(c, seed):
    g, D = _gen(seed), HIDDEN[c["model"]]
    return {"x": _normal(g, 1, D), "emb": _weight(g, c["vocab"], D)}


LAYER_NAMES = ("wq", "wk", "wv", "wo", "gate", "up", "down", "q_norm", "k_norm", "input_norm", "post_attn_norm")


def _decoder_layer(g, model):
    D, I = HIDDEN[model], INTER[model]
    return {"wq": _weight(g, QD, D), "wk": _weight(g, KVD, D), "wv": _weight(g, KVD, D), "wo": _weight(g, D, QD),
            "gate": _weight(g, I, D), "up": _weight(g, I, D), "down": _weight(g, D, I),
            "q_norm": _normal(g, HD, std=0.1, mean=1.0), "k_norm": _normal(g, HD, std=0.1, mean=1.0),
            "input_norm": _normal(g, D, std=0.1, mean=1.0), "post_attn_norm": _normal(g, D, std=0.1, mean=1.0)}


def _decoder_inputs(c, seed):
    """embedding, final norm, the prompt's rows, then the layers (a generator: one layer at a time)"""
    g, D = _gen(seed), HIDDEN[c["model"]]
    rows = c["rows"] if c["kind"] == "prefill" else 0
    head = {"emb": _weight(g, VOCAB, D), "fnorm": _normal(g, D, std=0.1, mean=1.0),
            "past": _normal(g, c["past"], D), "rows": _normal(g, rows, D), "last": _normal(g, D),
            "first": 1000 + seed % 1000}
    return head, (_decoder_layer(g, c["model"]) for _ in range(c["layers"]))


def _encoder_inputs(c, seed):
    g, e = _gen(seed), ENC[c["model"]]
    d, f, o = e["d"], e["ffn"], e["out"]
    w = lambda *s, std=0.02: _weight(g, *s, std=std).float()
    v = lambda n, std=0.02, mean=0.0: _normal(g, n, std=std, mean=mean)
    mel = _normal(g, 128, c["frames"])
    layers = [[w(d, d), v(d), w(d, d), v(d), w(d, d), v(d), w(d, d), v(d), v(d, 0.1, 1.0), v(d),
               w(f, d), v(f), w(d, f), v(d), v(d, 0.1, 1.0), v(d)] for _ in range(e["layers"])]
    stem = [w(ENC_CH, 1, 3, 3, std=0.2), v(ENC_CH), w(ENC_CH, ENC_CH, 3, 3), v(ENC_CH), w(ENC_CH, ENC_CH, 3, 3),
            v(ENC_CH), w(d, ENC_CH * 16), v(d, 0.1, 1.0), v(d), w(d, d), v(d), w(o, d), v(o)]
    return mel, layers, stem


# ---------------------------------------------------------------------------
# what a program holds before the call
# ---------------------------------------------------------------------------
class _Rows:
    """a view of device memory that `owner` frees, for torch.as_tensor (the tensor keeps this object, it the owner)"""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<f4", "version": 2}


def _bits(t):
    return t.view(torch.int16).cpu().numpy().view(np.uint16) if t.dtype == torch.bfloat16 else t.cpu().numpy()


def _decoder(c, seed):
    D, I = HIDDEN[c["model"]], INTER[c["model"]]
    head, layers = _decoder_inputs(c, seed)
    cfg = QA.HipConfig(D, c["layers"], HEADS, KV_HEADS, HD, I, VOCAB, EPS, THETA)
    dec = QA.Decoder(cfg, 0, c["past"] + c.get("rows", 0) + c.get("steps", 0) + 8)
    for l, w in enumerate(layers):
        dec.load_layer(l, *[_bits(w[n]) for n in LAYER_NAMES])
    dec.load_embeddings(_bits(head["emb"]), _bits(head["fnorm"]))
    dec.set_keep_logits(True)
    torch.cuda.synchronize()
    if c["past"]:
        dec.prefill_device(head["past"].data_ptr(), c["past"])
    return {"dec": dec, "rows": head["rows"], "last": head["last"].cpu().numpy(), "first": head["first"]}


def prepare(case, seed):
    kind = case["kind"]
    dev = lambda *s: torch.empty(*s, device="cuda", dtype=torch.float32)
    if kind == "attn_block":
        t = _attn_inputs(case, seed)
        S, past = case["rows"], case["past"]
        # the cache holds the past rows; the call appends its own behind them
        for n in ("k", "v"):
            cache = torch.zeros(past + S, KVD, device="cuda")
            cache[:past] = t.pop(n + "_past")
            t[n] = cache
        t.update(xn=dev(S, t["x"].shape[1]), q=dev(S, QD), att=dev(S, QD), out=dev(S, t["x"].shape[1]))
    elif kind == "mlp_block":
        t = _mlp_inputs(case, seed)
        S, D, I = case["rows"], HIDDEN[case["model"]], INTER[case["model"]]
        t.update(xn=dev(S, D), gu=dev(S, 2 * I), act=dev(S, I), out=dev(S, D))
    elif kind == "attention":
        t = _attention_inputs(case, seed)
        t.update(out=dev(case["rows"], QD))
    elif kind == "head":
        t = _head_inputs(case, seed)
        t.update(logits=dev(1, case["vocab"]))
    elif kind == "encoder":
        mel, layers, stem = _encoder_inputs(case, seed)
        e = ENC[case["model"]]
        enc = QA.Encoder(QA.EncConfig(e["d"], e["layers"], e["heads"], 64, e["ffn"], e["out"], ENC_CHUNK, 800), 0)
        for l, arrs in enumerate(layers):
            enc.load_layer(l, [_bits(a) for a in arrs])
        enc.load_stem([_bits(a) for a in stem])
        t = {"enc": enc, "mel": mel}
    else:
        t = _decoder(case, seed)
    t["case"] = case
    torch.cuda.synchronize()
    return t


# ---------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    L, ok = QA.lib(), QA.check
    s = torch.cuda.current_stream().cuda_stream
    p = lambda n, off=0: state[n].data_ptr() + off
    if kind == "attn_block":
        S, past, D = case["rows"], case["past"], HIDDEN[case["model"]]
        new = past * KVD * 4                        # the appended rows' place in the cache
        ok(L.qwen_hip_rms_norm(p("xn"), p("x"), p("w_in"), S, D, EPS, s))
        if S == 1:
            ok(L.qwen_hip_linear_nobias_bf16_qkv(p("q"), p("k", new), p("v", new), p("xn"), p("wq"), p("wk"),
                                                 p("wv"), D, QD, KVD, s))
        else:
            ok(L.qwen_hip_linear_nobias_bf16(p("q"), p("xn"), p("wq"), S, D, QD, s))
            ok(L.qwen_hip_linear_nobias_bf16(p("k", new), p("xn"), p("wk"), S, D, KVD, s))
            ok(L.qwen_hip_linear_nobias_bf16(p("v", new), p("xn"), p("wv"), S, D, KVD, s))
        ok(L.qwen_hip_rms_norm_per_head(p("q"), p("q_norm"), S, HEADS, HD, EPS, s))
        ok(L.qwen_hip_rms_norm_per_head(p("k", new), p("k_norm"), S, KV_HEADS, HD, EPS, s))
        ok(L.qwen_hip_apply_rope_neox(p("q"), p("cos"), p("sin"), S, HEADS, HD, s))
        ok(L.qwen_hip_apply_rope_neox(p("k", new), p("cos"), p("sin"), S, KV_HEADS, HD, s))
        ok(L.qwen_hip_causal_attention(p("att"), p("q"), p("k"), p("v"), S, past + S, HEADS, KV_HEADS, HD,
                                       1.0 / math.sqrt(HD), past, s))
        ok(L.qwen_hip_linear_nobias_bf16(p("out"), p("att"), p("wo"), S, QD, D, s))
        ok(L.qwen_hip_add_inplace(p("out"), p("x"), S * D, s))
        return [state["out"], state["k"][past:], state["v"][past:]]
    if kind == "mlp_block":
        S, D, I = case["rows"], HIDDEN[case["model"]], INTER[case["model"]]
        act = "gu" if S == 1 else "act"             # one row: in place, as the token loop does
        ok(L.qwen_hip_rms_norm(p("xn"), p("x"), p("w_post"), S, D, EPS, s))
        ok(L.qwen_hip_linear_nobias_bf16(p("gu"), p("xn"), p("gate_up"), S, D, 2 * I, s))
        ok(L.qwen_hip_swiglu_multiply(p(act), p("gu"), S, I, s))
        ok(L.qwen_hip_linear_nobias_bf16(p("out"), p(act), p("down"), S, I, D, s))
        ok(L.qwen_hip_add_inplace(p("out"), p("x"), S * D, s))
        return state["out"]
    if kind == "attention":
        S, past = case["rows"], case["past"]
        ok(L.qwen_hip_causal_attention(p("out"), p("q"), p("k"), p("v"), S, past + S, HEADS, KV_HEADS, HD,
                                       1.0 / math.sqrt(HD), past, s))
        return state["out"]
    if kind == "head":
        D, V = HIDDEN[case["model"]], case["vocab"]
        ok(L.qwen_hip_linear_nobias_bf16(p("logits"), p("x"), p("emb"), 1, D, V, s))
        return [state["logits"], int(ok(L.qwen_hip_argmax_matvec_bf16(p("x"), p("emb"), D, V, s)))]
    if kind == "encoder":
        n, ptr = state["enc"].forward_device(state["mel"].data_ptr(), case["frames"])
        return torch.as_tensor(_Rows(ptr, (n, ENC[case["model"]]["out"]), state["enc"]), device="cuda")
    dec = state["dec"]
    dec.set_kv_len(case["past"])
    if kind == "prefill":
        dec.prefill_device(state["rows"].data_ptr(), case["rows"])
        dec.forward(state["last"])
        return dec.read_logits()
    tokens = dec.generate(state["first"], case["steps"])
    return [tokens, dec.read_logits()]


# ---------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------
def _pairs(S, past):
    return S * past + S * (S + 1) / 2.0


def work(case):
    kind = case["kind"]
    D, I = (HIDDEN[case["model"]], INTER[case["model"]]) if "model" in case else (0, 0)
    if kind == "attn_block":
        S, past = case["rows"], case["past"]
        w = (QD + 2 * KVD) * D + D * QD
        b = 2 * w + 4 * (2 * S * D + 2 * KVD * (past + 2 * S) + 2 * S * HD + D + 2 * HD)
        return {"bytes": b, "flops": 2.0 * S * w + 4.0 * HD * HEADS * _pairs(S, past)}
    if kind == "mlp_block":
        S = case["rows"]
        w = 3 * I * D
        return {"bytes": 2 * w + 4 * (2 * S * D + D), "flops": 2.0 * S * w}
    if kind == "attention":
        S, past = case["rows"], case["past"]
        return {"bytes": 4 * (2 * S * QD + 2 * KVD * (past + S)), "flops": 4.0 * HD * HEADS * _pairs(S, past)}
    if kind == "head":
        # two calls, each of which has to read the table
        V = case["vocab"]
        return {"bytes": 2 * 2 * V * D + 4 * (2 * D + V), "flops": 4.0 * V * D}
    if kind == "encoder":
        e = ENC[case["model"]]
        d, f, o, F = e["d"], e["ffn"], e["out"], case["frames"]
        full, last = F // ENC_CHUNK, F % ENC_CHUNK
        half = lambda n: (n + 1) // 2
        wid = [(full * 50 + half(last), 64), (full * 25 + half(half(last)), 32),
               (full * ENC_TPC + half(half(half(last))), 16)]
        T = wid[2][0]
        k2 = 9 * ENC_CH
        flops = 2.0 * ENC_CH * (9 * wid[0][0] * 64 + k2 * wid[1][0] * 32 + k2 * wid[2][0] * 16)
        layer = 4 * d * d + 2 * d * f
        flops += 2.0 * T * (d * ENC_CH * 16 + e["layers"] * layer + d * d + d * o)
        nw, rest = T // ENC_WIN, T % ENC_WIN
        flops += e["layers"] * 4.0 * d * (nw * ENC_WIN * ENC_WIN + rest * rest)
        w = ENC_CH * (9 + 2 * k2) + d * ENC_CH * 16 + e["layers"] * layer + d * d + d * o
        return {"bytes": 2 * w + 4 * (128 * F + T * o), "flops": flops}
    layer = (QD + 2 * KVD) * D + D * QD + 3 * I * D
    n, past = case["layers"], case["past"]
    kv = 4 * 2 * KVD * n                            # bytes of one position's K and V, all layers
    if kind == "prefill":
        S = case["rows"]
        # the prefill reads the layers once, the forward the layers and the LM head once more
        b = 2 * (2 * n * layer + VOCAB * D) + 4 * S * D + kv * (2 * past + 2 * S + 1) + 4 * VOCAB
        f = 2.0 * n * layer * (S + 1) + 2.0 * VOCAB * D + n * 4.0 * HD * HEADS * _pairs(S + 1, past)
        return {"bytes": b, "flops": f}
    k = case["steps"]
    b = k * 2 * (n * layer + VOCAB * D) + kv * (sum(past + i for i in range(k)) + k) + 4 * VOCAB
    return {"bytes": b, "flops": k * 2.0 * (n * layer + VOCAB * D) + n * 4.0 * HD * HEADS * _pairs(k, past)}


def tolerance(case):
    """About four times the distance from `exact` that these paths show.  One row runs on fp32 products (1e-7 per
    sum); several rows carry each fp32 activation as two bf16 terms on the matrix cores (2^-17 per product)."""
    kind, one = case["kind"], case.get("rows") == 1
    if kind in ("attn_block", "mlp_block"):
        return {"rel": 1e-6, "max": 5e-6} if one else {"rel": 1.1e-5, "max": 6e-5}
    if kind == "attention":
        # attention outputs shrink with the keys averaged: a first row's error is large beside the others' size
        return {"rel": 2.2e-5, "max": 1e-3}
    if kind == "head":
        return {"rel": 5e-7, "max": 2e-6}
    if kind == "encoder":
        return {"rel": 2.4e-5, "max": 1.4e-4}
    return {"rel": 1.6e-5, "max": 8e-5} if kind == "prefill" else {"rel": 5e-5, "max": 2.5e-4}


# ---------------------------------------------------------------------------
# the same in 64 bits, in plain torch
# ---------------------------------------------------------------------------
def _rms(x, w):
    return x * w.double() / torch.sqrt((x * x).mean(-1, keepdim=True) + EPS)


def _rope(x, cos, sin):
    """x [S][heads][128]; cos, sin [S][128]"""
    c, s = cos.double()[:, None, :HD // 2], sin.double()[:, None, :HD // 2]
    a, b = x[..., :HD // 2], x[..., HD // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _causal(q, k, v, past):
    """q [S][QD], k / v [past + S][KVD] -> [S][QD]"""
    S, n = q.shape[0], k.shape[0]
    out = torch.empty_like(q)
    mask = torch.arange(n, device="cuda")[None, :] > past + torch.arange(S, device="cuda")[:, None]
    for h in range(HEADS):
        g = slice(h // 2 * HD, (h // 2 + 1) * HD)
        sc = (q[:, h * HD:(h + 1) * HD] @ k[:, g].t()) / math.sqrt(HD)
        sc.masked_fill_(mask, float("-inf"))
        out[:, h * HD:(h + 1) * HD] = torch.softmax(sc, -1) @ v[:, g]
    return out


def _layer64(x, w, kc, vc, cos, sin):
    """one decoder layer on x [S][D] after the cached kc / vc; returns (x, kc, vc) with the new rows appended"""
    S, past = x.shape[0], kc.shape[0]
    xn = _rms(x, w["input_norm"])
    q = _rope(_rms((xn @ w["wq"].double().t()).view(S, HEADS, HD), w["q_norm"]), cos, sin).reshape(S, QD)
    k = _rope(_rms((xn @ w["wk"].double().t()).view(S, KV_HEADS, HD), w["k_norm"]), cos, sin).reshape(S, KVD)
    kc, vc = torch.cat([kc, k]), torch.cat([vc, xn @ w["wv"].double().t()])
    x = x + _causal(q, kc, vc, past) @ w["wo"].double().t()
    xn = _rms(x, w["post_attn_norm"])
    g, u = xn @ w["gate"].double().t(), xn @ w["up"].double().t()
    return x + (torch.nn.functional.silu(g) * u) @ w["down"].double().t(), kc, vc


def _layernorm64(x, w, b):
    m = x.mean(-1, keepdim=True)
    return (x - m) / torch.sqrt(((x - m) ** 2).mean(-1, keepdim=True) + ENC_EPS) * w.double() + b.double()


def _gelu64(x):
    return 0.5 * x * (1.0 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))


def _conv64(x, w, b):
    """3x3, stride 2, padding 1 on [n][c][h][w]"""
    n, c, h, wd = x.shape
    ho, wo = (h + 1) // 2, (wd + 1) // 2
    xp = torch.nn.functional.pad(x, (1, 2, 1, 2))
    taps = [xp[:, :, i:i + 2 * ho - 1:2, j:j + 2 * wo - 1:2] for i in range(3) for j in range(3)]
    cols = torch.stack(taps, 2).permute(0, 3, 4, 1, 2).reshape(n * ho * wo, c * 9)
    y = cols @ w.double().reshape(w.shape[0], -1).t() + b.double()
    return _gelu64(y).view(n, ho, wo, -1).permute(0, 3, 1, 2)


def _encoder64(case, seed):
    mel, layers, stem = _encoder_inputs(case, seed)
    e = ENC[case["model"]]
    d, H, F = e["d"], e["heads"], case["frames"]
    toks = []
    full = F // ENC_CHUNK * ENC_CHUNK
    images = [mel[:, :full].reshape(128, -1, ENC_CHUNK).transpose(0, 1)] if full else []
    if F > full:
        images.append(mel[None, :, full:])
    for im in images:                               # every chunk is an image of its own
        y = im[:, None].double()
        for i in range(0, 6, 2):
            y = _conv64(y, stem[i], stem[i + 1])
        n, _, _, wd = y.shape
        y = y.permute(0, 3, 1, 2).reshape(n, wd, ENC_CH * 16) @ stem[6].double().t()
        half = d // 2
        inv = np.exp(-np.arange(half) * np.float64(np.float32(math.log(10000.0)) / np.float32(half - 1)))
        a = np.arange(wd)[:, None] * inv.astype(np.float32).astype(np.float64)[None, :]
        pe = np.concatenate([np.sin(a), np.cos(a)], 1).astype(np.float32)
        toks.append((y + torch.from_numpy(pe).cuda().double()).reshape(n * wd, d))
    x = torch.cat(toks)
    T = x.shape[0]
    for w in layers:
        n = _layernorm64(x, w[8], w[9])
        q, k, v = (n @ w[2 * i].double().t() + w[2 * i + 1].double() for i in range(3))
        att = torch.empty_like(q)
        for t0 in range(0, T, ENC_WIN):
            r = slice(t0, min(T, t0 + ENC_WIN))
            qq, kk, vv = (t[r].view(-1, H, 64).transpose(0, 1) for t in (q, k, v))
            sc = torch.softmax(torch.matmul(qq, kk.transpose(1, 2).contiguous()) / 8.0, -1)
            att[r] = torch.matmul(sc, vv.contiguous()).transpose(0, 1).reshape(-1, d)
        x = x + att @ w[6].double().t() + w[7].double()
        n = _layernorm64(x, w[14], w[15])
        x = x + _gelu64(n @ w[10].double().t() + w[11].double()) @ w[12].double().t() + w[13].double()
    n = _layernorm64(x, stem[7], stem[8])
    return _gelu64(n @ stem[9].double().t() + stem[10].double()) @ stem[11].double().t() + stem[12].double()


def exact(case, seed):
    kind = case["kind"]
    if kind == "attn_block":
        t = _attn_inputs(case, seed)
        S, past = case["rows"], case["past"]
        x = t["x"].double()
        xn = _rms(x, t["w_in"])
        q = _rope(_rms((xn @ t["wq"].double().t()).view(S, HEADS, HD), t["q_norm"]), t["cos"], t["sin"])
        k = _rope(_rms((xn @ t["wk"].double().t()).view(S, KV_HEADS, HD), t["k_norm"]), t["cos"], t["sin"])
        k, v = k.reshape(S, KVD), xn @ t["wv"].double().t()
        att = _causal(q.reshape(S, QD), torch.cat([t["k_past"].double(), k]), torch.cat([t["v_past"].double(), v]),
                      past)
        return [x + att @ t["wo"].double().t(), k, v]
    if kind == "mlp_block":
        t = _mlp_inputs(case, seed)
        x = t["x"].double()
        gu = _rms(x, t["w_post"]) @ t["gate_up"].double().t()
        return x + (torch.nn.functional.silu(gu[:, 0::2]) * gu[:, 1::2]) @ t["down"].double().t()
    if kind == "attention":
        t = _attention_inputs(case, seed)
        return _causal(t["q"].double(), t["k"].double(), t["v"].double(), case["past"])
    if kind == "head":
        t = _head_inputs(case, seed)
        y = t["x"].double() @ t["emb"].double().t()
        return [y, int(y.argmax())]
    if kind == "encoder":
        return _encoder64(case, seed)
    # decoders: prompt (past, then rows) and the last row, or the greedy steps
    head, layers = _decoder_inputs(case, seed)
    layers = list(layers)
    emb, n = head["emb"].double(), case["past"] + case.get("rows", 0) + case.get("steps", 0) + 1
    cos, sin = _rope_table(n)
    kv = [[torch.empty(0, KVD, device="cuda", dtype=torch.float64)] * 2 for _ in layers]

    def rows64(x):
        at = kv[0][0].shape[0]
        r = slice(at, at + x.shape[0])
        for l, w in enumerate(layers):
            x, kv[l][0], kv[l][1] = _layer64(x, w, kv[l][0], kv[l][1], cos[r], sin[r])
        return x

    if kind == "prefill":
        x = torch.cat([head["past"], head["rows"]]).double()
        rows64(x)
        return (_rms(rows64(head["last"].double()[None]), head["fnorm"])[0] @ emb.t()).cpu().numpy()
    rows64(head["past"].double())
    tokens, tok = [], head["first"]
    for _ in range(case["steps"]):
        y = _rms(rows64(emb[tok][None]), head["fnorm"])[0] @ emb.t()
        tok = int(y.argmax())
        tokens.append(tok)
    return [np.array(tokens, np.int32), y.cpu().numpy()]
