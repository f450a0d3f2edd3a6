"""The work that performance is measured on: what a user of this library has it do.

The library computes the linear layers, attention and producers of Llama-family models from
GGUF weights, on device buffers. So the cases are the matrices and blocks of such models, each
through the entry points a device-resident engine calls: one token at a time (decode), small
batches, and whole prompts (prefill); the six types with integer kernels (Q4_0, Q5_0, Q8_0,
Q4_K, Q5_K, Q6_K) and the seven float-dot types (F32, F16, Q4_1, Q5_1, Q8_1, Q2_K, Q3_K). The
shapes are those of the repository's workloads: Llama-3-8B (4096 / 14336 / 128256, 32 query
heads over 8 KV heads of 128) and Qwen2.5-0.5B (896 / 4864 / 151936, heads of 64).

Kinds of case
  linear            y = x W^T (+ bias): matmul_quant_dev on m rows of fp32 activations
  head              RMSNorm and the output head of one row in one launch
  decode            one whole decode step: embedding, layers, final norm and head; logits
  decode_attention  RoPE and attention of one query row over the KV cache
  attention_block   the attention half of a prefill layer: norm, q/k/v, RoPE, attention, wo,
                    residual
  ffn_block         the feed-forward half of a prefill layer: norm, gate/up, SwiGLU, down,
                    residual
"""
from __future__ import annotations

import math

import torch

import cllm_inference_amd as C

TYPES = {"F32": 0, "F16": 1, "Q4_0": 2, "Q4_1": 3, "Q5_0": 6, "Q5_1": 7, "Q8_0": 8, "Q8_1": 9,
         "Q2_K": 10, "Q3_K": 11, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14}
# elements and bytes per block
BLOCK = {"F32": 1, "F16": 1, "Q4_0": 32, "Q4_1": 32, "Q5_0": 32, "Q5_1": 32, "Q8_0": 32,
         "Q8_1": 32, "Q2_K": 256, "Q3_K": 256, "Q4_K": 256, "Q5_K": 256, "Q6_K": 256}
BYTES = {"F32": 4, "F16": 2, "Q4_0": 18, "Q4_1": 20, "Q5_0": 22, "Q5_1": 24, "Q8_0": 34,
         "Q8_1": 36, "Q2_K": 84, "Q3_K": 110, "Q4_K": 144, "Q5_K": 176, "Q6_K": 210}
FLOAT_DOT = ("F32", "F16", "Q4_1", "Q5_1", "Q8_1", "Q2_K", "Q3_K")
INTEGER = ("Q4_0", "Q5_0", "Q8_0", "Q4_K", "Q5_K", "Q6_K")
EPS, THETA = 1e-5, 500000.0


def _linear(qt, n, k, m, bias=False, outliers=False, name=None):
    c = {"kind": "linear", "type": qt, "n": n, "k": k, "m": m, "bias": bias, "outliers": outliers}
    return c if name is None else {"name": name, **c}


def listed():
    return [
        # one token through the smallest model's feed-forward matrix: launch and latency bound
        _linear("Q8_0", 4864, 896, 1, name="linear_q8_0_4864x896_m1"),
        # one token through the 8B model's gate matrix, the headline decode GEMV
        _linear("Q4_K", 14336, 4096, 1, name="linear_q4_k_14336x4096_m1"),
        # the 8B model's output head after its final norm
        {"name": "head_q6_k_128256x4096", "kind": "head", "type": "Q6_K", "n": 128256, "k": 4096},
        # one whole decode step: four layers of the 8B model in the Q4_K_M mix, 1024 positions
        # in the cache, and the head
        {"name": "decode_q4_k_m_4_layers", "kind": "decode", "type": "Q4_K", "down": "Q6_K",
         "layers": 4, "n_embd": 4096, "n_head": 32, "n_kv": 8, "hd": 128, "n_ff": 14336,
         "vocab": 128256, "pos": 1024},
        # attention of one token at the end of a full 8192-position context
        {"name": "decode_attention_8192", "kind": "decode_attention", "n_head": 32, "n_kv": 8,
         "hd": 128, "pos": 8191},
        # a small batch of concurrent sequences or draft tokens, activations with outliers
        _linear("Q5_K", 14336, 4096, 16, outliers=True, name="linear_q5_k_14336x4096_m16"),
        _linear("Q8_0", 4096, 4096, 64, outliers=True, name="linear_q8_0_4096x4096_m64"),
        # a 512-token prompt through the smallest model: K = 896 is no multiple of 256
        _linear("Q8_0", 4864, 896, 512, name="linear_q8_0_4864x896_m512"),
        # the attention half of a prefill layer: the second turn of a chat, 512 new tokens
        # after 1024 cached positions
        {"name": "attention_block_512_after_1024", "kind": "attention_block", "type": "Q4_K",
         "n_embd": 4096, "n_head": 32, "n_kv": 8, "hd": 128, "rows": 512, "pos0": 1024},
        # the feed-forward half of a prefill layer, a 512-token prompt
        {"name": "ffn_block_512", "kind": "ffn_block", "type": "Q4_K", "down": "Q6_K",
         "n_embd": 4096, "n_ff": 14336, "rows": 512},
        # the small model's tied F16 output head, one token
        _linear("F16", 151936, 896, 1, name="linear_f16_151936x896_m1"),
        # a prompt of odd length through a matrix of a Q3_K file
        _linear("Q3_K", 4096, 4096, 301, name="linear_q3_k_4096x4096_m301"),
    ]


def _log(rng, lo, hi):
    """A whole number in [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


_HEADS = ((32, 8, 128), (14, 2, 64), (16, 16, 64), (32, 32, 128), (40, 8, 128), (8, 4, 256))


def draw(rng):
    kind = rng.choices(("linear", "float", "head", "decode", "decode_attention",
                        "attention_block", "ffn_block"), (42, 22, 4, 4, 10, 9, 9))[0]
    if kind == "linear":
        qt = rng.choice(INTEGER)
        step = 256 if BLOCK[qt] == 256 else rng.choice((32, 128, 256))
        k = max(1, _log(rng, 512, 14336) // step) * step
        n = _log(rng, 256, 16384)
        m = rng.choice((1, _log(rng, 2, 32), _log(rng, 16, 512), _log(rng, 16, 512)))
        return _linear(qt, n, k, m, bias=rng.random() < 0.3, outliers=rng.random() < 0.5)
    if kind == "float":
        qt = rng.choice(FLOAT_DOT)
        step = 256 if BLOCK[qt] == 256 else 32
        k = max(1, _log(rng, 256, 8192) // step) * step
        n = _log(rng, 256, 16384)
        m = rng.choice((1, _log(rng, 2, 16), _log(rng, 16, 301)))
        while n * k * m > 4096 * 4096 * 301:
            n = max(128, n // 2 + 1)
        return _linear(qt, n, k, m, bias=rng.random() < 0.3, outliers=rng.random() < 0.3)
    if kind == "head":
        return {"kind": "head", "type": rng.choice(("Q6_K", "Q8_0", "Q4_K")),
                "n": _log(rng, 32000, 128256), "k": 256 * rng.randint(4, 16)}
    if kind == "decode":
        n_head, n_kv, hd = rng.choice(((32, 8, 128), (16, 16, 64), (16, 8, 128)))
        return {"kind": "decode", "type": "Q4_K", "down": "Q6_K", "layers": rng.randint(1, 3),
                "n_embd": n_head * hd, "n_head": n_head, "n_kv": n_kv, "hd": hd,
                "n_ff": 256 * rng.randint(8, 48), "vocab": _log(rng, 8000, 64000),
                "pos": _log(rng, 1, 2048)}
    n_head, n_kv, hd = rng.choice(_HEADS)
    if kind == "decode_attention":
        return {"kind": kind, "n_head": n_head, "n_kv": n_kv, "hd": hd, "pos": _log(rng, 16, 8000)}
    if kind == "attention_block":
        n_head, n_kv, hd = rng.choice(((32, 8, 128), (16, 16, 64), (16, 8, 128), (8, 4, 256)))
        return {"kind": kind, "type": rng.choice(("Q4_K", "Q5_K")), "n_embd": n_head * hd,
                "n_head": n_head, "n_kv": n_kv, "hd": hd, "rows": _log(rng, 64, 512),
                "pos0": rng.choice((0, _log(rng, 16, 1024)))}
    down = rng.choice(("Q6_K", "Q4_K", "Q8_0"))
    return {"kind": kind, "type": rng.choice(("Q4_K", "Q5_K", "Q8_0")), "down": down,
            "n_embd": 256 * rng.randint(4, 16), "n_ff": 256 * rng.randint(8, 56),
            "rows": _log(rng, 32, 500)}


# ---- inputs -------------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _half(v):
    return v.half().view(torch.uint8).view(-1, 2)


def _weight(g, qt, n, k, gain=1.0):
    """n x k weights of type qt as the bytes of their blocks: codes, 6-bit scales and high bits
    uniform, the half-precision scales such that the weights spread around zero by about 0.02,
    as trained ones do (times gain)."""
    if qt in ("F32", "F16"):
        w = torch.randn(n * k, device="cuda", generator=g) * 0.02
        return (w if qt == "F32" else w.half()).view(torch.uint8)
    nb, ts = n * (k // BLOCK[qt]), BYTES[qt]
    raw = torch.randint(-2 ** 31, 2 ** 31 - 1, ((nb * ts + 3) // 4,), device="cuda", generator=g,
                        dtype=torch.int32)
    b = raw.view(torch.uint8)[: nb * ts].view(nb, ts)
    at, lo, hi = {"Q8_0": (0, 5e-5, 5e-4), "Q8_1": (0, 5e-5, 5e-4), "Q4_0": (0, 1e-3, 8e-3),
                  "Q4_1": (0, 1e-3, 8e-3), "Q5_0": (0, 5e-4, 4e-3), "Q5_1": (0, 5e-4, 4e-3),
                  "Q2_K": (80, 5e-4, 4e-3), "Q3_K": (108, 1e-4, 1e-3), "Q4_K": (0, 2e-5, 2e-4),
                  "Q5_K": (0, 1e-5, 1e-4), "Q6_K": (208, 1e-5, 1e-4)}[qt]
    d = torch.empty(nb, device="cuda").uniform_(lo * gain, hi * gain, generator=g)
    b[:, at:at + 2] = _half(d)
    # the minimum that centres the codes of each block or sub-block, give or take a fifth
    centre = {"Q4_1": (2, -7.5), "Q5_1": (2, -15.5), "Q2_K": (82, 1.5), "Q4_K": (2, 7.5),
              "Q5_K": (2, 15.5)}.get(qt)
    if centre:
        d *= torch.empty(nb, device="cuda").uniform_(0.8, 1.2, generator=g)
        b[:, centre[0]:centre[0] + 2] = _half(d * centre[1])
    if qt in ("Q4_K", "Q5_K"):  # sub-block minima with the codes of the scales
        b[:, 8:12] = b[:, 4:8]
        b[:, 12:16] = (b[:, 12:16] & 15) * 17
    if qt == "Q2_K":
        b[:, 0:16] = (b[:, 0:16] & 15) * 17
    if qt == "Q8_1":
        b[:, 2:4] = _half(d.half().float() * b[:, 4:36].view(torch.int8).sum(1, dtype=torch.int32))
    if qt == "Q6_K":
        sc = torch.randint(-32, 32, (nb, 16), device="cuda", generator=g, dtype=torch.int8)
        b[:, 192:208] = sc.view(torch.uint8)
    return raw.view(torch.uint8)[: nb * ts]


def _rows(g, m, k, outliers=False):
    x = torch.randn((m, k), device="cuda", generator=g)
    if outliers:
        x = torch.where(torch.rand((m, k), device="cuda", generator=g) < 0.01, x * 20.0, x)
    return x


def _norm_weight(g, k):
    return 1.0 + 0.1 * torch.randn(k, device="cuda", generator=g)


def prepare(case, seed):
    g, c = _gen(seed), case
    s = {"case": dict(c)}
    if c["kind"] == "linear":
        s["w"] = _weight(g, c["type"], c["n"], c["k"])
        s["x"] = _rows(g, c["m"], c["k"], c["outliers"])
        s["bias"] = torch.randn(c["n"], device="cuda", generator=g) if c["bias"] else None
        s["y"] = torch.empty((c["m"], c["n"]), device="cuda")
    elif c["kind"] == "head":
        s["w"] = _weight(g, c["type"], c["n"], c["k"])
        s["x"], s["norm"] = _rows(g, 1, c["k"]), _norm_weight(g, c["k"])
        s["y"] = torch.empty((1, c["n"]), device="cuda")
    elif c["kind"] == "decode":
        e, ff, q, kv = c["n_embd"], c["n_ff"], c["n_head"] * c["hd"], c["n_kv"] * c["hd"]
        # the embedding rows this program looks up: a residual stream that the layers' updates
        # are small beside, as in a trained model
        s["emb"] = _weight(g, c["type"], 512, e, gain=200.0)
        s["id"] = torch.randint(0, 512, (1,), device="cuda", generator=g, dtype=torch.int32)
        s["layers"] = []
        for _ in range(c["layers"]):
            cache = torch.randn((2, c["pos"] + 1, kv), device="cuda", generator=g)
            s["layers"].append({
                "norm1": _norm_weight(g, e), "norm2": _norm_weight(g, e),
                "wq": _weight(g, c["type"], q, e), "wk": _weight(g, c["type"], kv, e),
                "wv": _weight(g, c["type"], kv, e), "wo": _weight(g, c["type"], e, q),
                "gate": _weight(g, c["type"], ff, e), "up": _weight(g, c["type"], ff, e),
                "down": _weight(g, c["down"], e, ff), "kc": cache[0], "vc": cache[1]})
        s["norm"], s["out"] = _norm_weight(g, e), _weight(g, "Q6_K", c["vocab"], e)
        for name, n in (("x", e), ("q", q), ("a", q), ("h", ff), ("logits", c["vocab"])):
            s[name] = torch.empty((1, n), device="cuda")
    elif c["kind"] == "decode_attention":
        kv, L = c["n_kv"] * c["hd"], c["pos"] + 1
        s["q"] = _rows(g, 1, c["n_head"] * c["hd"])
        s["kc"], s["vc"] = _rows(g, L, kv), _rows(g, L, kv)
        s["k_new"] = _rows(g, 1, kv)
        s["y"] = torch.empty((1, c["n_head"] * c["hd"]), device="cuda")
    elif c["kind"] == "attention_block":
        e, m, q, kv = c["n_embd"], c["rows"], c["n_head"] * c["hd"], c["n_kv"] * c["hd"]
        s["x"], s["norm"] = _rows(g, m, e), _norm_weight(g, e)
        s["w"] = [_weight(g, c["type"], n, e) for n in (q, kv, kv)]
        s["wo"] = _weight(g, c["type"], e, q)
        s["kc"], s["vc"] = _rows(g, c["pos0"] + m, kv), _rows(g, c["pos0"] + m, kv)
        s["act"], s["act_o"] = C.mfma_act_new(e, m), C.mfma_act_new(q, m)
        s["q"], s["a"] = torch.empty((m, q), device="cuda"), torch.empty((m, q), device="cuda")
        s["o"] = torch.empty((m, e), device="cuda")
    else:
        e, m, ff = c["n_embd"], c["rows"], c["n_ff"]
        s["x"], s["norm"] = _rows(g, m, e), _norm_weight(g, e)
        s["gate"], s["up"] = _weight(g, c["type"], ff, e), _weight(g, c["type"], ff, e)
        s["down"] = _weight(g, c["down"], e, ff)
        s["act"], s["act_h"] = C.mfma_act_new(e, m), C.mfma_act_new(ff, m)
        s["gu"] = [torch.empty((m, ff), device="cuda") for _ in range(2)]
        s["o"] = torch.empty((m, e), device="cuda")
    return s


# ---- one pass -----------------------------------------------------------------------------

def run(state):
    s, c = state, state["case"]
    if c["kind"] == "linear":
        return C.matmul_quant_dev(s["x"], s["w"], TYPES[c["type"]], s["bias"], c["k"], c["n"],
                                  y=s["y"])
    if c["kind"] == "head":
        return C.rmsnorm_gemv_multi_dev(s["x"], s["norm"], EPS, [s["w"]], TYPES[c["type"]], c["k"],
                                        [c["n"]], ys=[s["y"]])
    if c["kind"] == "decode":
        e, ff, q, kv = c["n_embd"], c["n_ff"], c["n_head"] * c["hd"], c["n_kv"] * c["hd"]
        t, td, pos, x = TYPES[c["type"]], TYPES[c["down"]], c["pos"], s["x"]
        C.dequantize_rows_dev(s["emb"], t, e, s["id"], out=x)
        for l in s["layers"]:
            C.rmsnorm_gemv_multi_dev(x, l["norm1"], EPS, [l["wq"], l["wk"], l["wv"]], t, e,
                                     [q, kv, kv], ys=[s["q"], l["kc"][pos], l["vc"][pos]])
            C.attention_rope_dev(s["q"], l["kc"], l["vc"], pos, c["n_head"], c["n_kv"], c["hd"],
                                 THETA, out=s["a"])
            C.matmul_quant_residual_dev(s["a"], l["wo"], t, None, q, e, x)
            C.rmsnorm_gemv_swiglu_dev(x, l["norm2"], EPS, l["gate"], l["up"], t, e, ff, h=s["h"])
            C.matmul_quant_residual_dev(s["h"], l["down"], td, None, ff, e, x)
        C.rmsnorm_gemv_multi_dev(x, s["norm"], EPS, [s["out"]], TYPES["Q6_K"], e, [c["vocab"]],
                                 ys=[s["logits"]])
        return {"logits": s["logits"], "x": x, "k": [l["kc"][pos] for l in s["layers"]],
                "v": [l["vc"][pos] for l in s["layers"]]}
    if c["kind"] == "decode_attention":
        # the new key row arrives unrotated and is rotated in place, so each pass writes it anew
        s["kc"][c["pos"]].copy_(s["k_new"][0])
        y = C.attention_rope_dev(s["q"], s["kc"], s["vc"], c["pos"], c["n_head"], c["n_kv"],
                                 c["hd"], THETA, out=s["y"])
        return {"y": y, "k": s["kc"][c["pos"]]}
    if c["kind"] == "attention_block":
        e, m, q, kv, p = c["n_embd"], c["rows"], c["n_head"] * c["hd"], c["n_kv"] * c["hd"], c["pos0"]
        t, kn, vn = TYPES[c["type"]], s["kc"][p:], s["vc"][p:]
        C.rmsnorm_mfma_dev(s["x"], s["norm"], EPS, act=s["act"])
        C.matmul_mfma_dev(s["w"], t, e, [q, kv, kv], s["act"], m, ys=[s["q"], kn, vn])
        C.rope_neox2_dev(s["q"], c["n_head"], kn, c["n_kv"], c["hd"], p, THETA)
        C.attention_dev(s["q"], s["kc"], s["vc"], p, c["n_head"], c["n_kv"], c["hd"], out=s["a"])
        C.quantize_mfma_dev(s["a"], act=s["act_o"])
        C.matmul_mfma_dev([s["wo"]], t, q, [e], s["act_o"], m, ys=[s["o"]])
        C.add_dev(s["o"], s["x"])
        return {"o": s["o"], "a": s["a"], "k": kn, "v": vn}
    e, m, ff = c["n_embd"], c["rows"], c["n_ff"]
    C.rmsnorm_mfma_dev(s["x"], s["norm"], EPS, act=s["act"])
    C.matmul_mfma_dev([s["gate"], s["up"]], TYPES[c["type"]], e, [ff, ff], s["act"], m, ys=s["gu"])
    C.swiglu_mfma_dev(s["gu"][0], s["gu"][1], act=s["act_h"])
    C.matmul_mfma_dev([s["down"]], TYPES[c["down"]], ff, [e], s["act_h"], m, ys=[s["o"]])
    C.add_dev(s["o"], s["x"])
    return {"o": s["o"], "gate": s["gu"][0], "up": s["gu"][1]}


def _wbytes(qt, n, k):
    return n * (k // BLOCK[qt]) * BYTES[qt]


def work(case):
    c = case
    if c["kind"] == "linear":
        return {"bytes": _wbytes(c["type"], c["n"], c["k"]) + 4 * c["m"] * (c["k"] + c["n"]) +
                4 * c["n"] * c["bias"], "flops": 2.0 * c["m"] * c["n"] * c["k"]}
    if c["kind"] == "head":
        return {"bytes": _wbytes(c["type"], c["n"], c["k"]) + 8 * c["k"] + 4 * c["n"],
                "flops": 2.0 * c["n"] * c["k"]}
    if c["kind"] == "ffn_block":
        e, m, ff = c["n_embd"], c["rows"], c["n_ff"]
        return {"bytes": 2 * _wbytes(c["type"], ff, e) + _wbytes(c["down"], e, ff) +
                4 * m * (2 * e + 2 * ff), "flops": 6.0 * m * e * ff}
    q, kv = c["n_head"] * c["hd"], c["n_kv"] * c["hd"]
    if c["kind"] == "decode_attention":
        L = c["pos"] + 1
        return {"bytes": 4 * (2 * L * kv + 2 * q + kv), "flops": 4.0 * L * q}
    e = c["n_embd"]
    if c["kind"] == "decode":
        ff, L = c["n_ff"], c["pos"] + 1
        layer = (_wbytes(c["type"], 2 * q + 2 * kv + 2 * ff, e) + _wbytes(c["down"], e, ff) +
                 8 * L * kv)
        return {"bytes": c["layers"] * layer + _wbytes("Q6_K", c["vocab"], e) + 4 * c["vocab"],
                "flops": c["layers"] * (2.0 * e * (2 * q + 2 * kv + 3 * ff) + 4.0 * L * q) +
                2.0 * e * c["vocab"]}
    m, p = c["rows"], c["pos0"]
    seen = m * p + m * (m + 1) / 2.0  # (query, position) pairs of one head
    return {"bytes": _wbytes(c["type"], 2 * q + 2 * kv, e) + 4 * (2 * m * e + m * q) +
            4 * (2 * p * kv + 2 * m * kv),
            "flops": 2.0 * m * e * (2 * q + 2 * kv) + 4.0 * seen * q}


def tolerance(case):
    if case["kind"] == "linear":
        # 32-bit sums of the same products in another order
        return {"rel": 2e-6, "max": 4e-5}
    if case["kind"] == "decode_attention":
        # a last bit of the rotation's 32-bit angle, up to 8000 radians, is 5e-4 radians
        return {"rel": 2e-4, "max": 5e-3}
    # Blocks quantize intermediate rows to Q8_0: a last-bit difference before it moves now and
    # then a code to its neighbour, 1/127 of its block's largest value.
    if case["kind"] == "head":
        return {"rel": 2e-4, "max": 2e-3}
    if case["kind"] == "decode":  # such moved codes travel through every later layer
        return {"rel": 3e-2, "max": 3e-1}
    return {"rel": 1e-3, "max": 2e-2}


# ---- the same in 64 bits ------------------------------------------------------------------

def _dequantize(b, qt):
    """Blocks b (blocks x bytes) of type qt as (blocks x elements) 64-bit values."""
    if qt in ("F32", "F16"):
        return b.contiguous().view(torch.float32 if qt == "F32" else torch.float16).double()

    def f16(i):
        return b[:, i:i + 2].contiguous().view(torch.float16).double()

    def i8(i, j):
        return b[:, i:j].view(torch.int8).double()

    if qt in ("Q8_0", "Q8_1"):
        return f16(0) * (i8(2, 34) if qt == "Q8_0" else i8(4, 36))
    if qt in ("Q4_0", "Q4_1", "Q5_0", "Q5_1"):
        at = {"Q4_0": 2, "Q4_1": 4, "Q5_0": 6, "Q5_1": 8}[qt]
        qs = b[:, at:at + 16]
        q = torch.cat([qs & 15, qs >> 4], 1)
        if qt[1] == "5":
            qh = b[:, at - 4:at]
            bits = torch.stack([(qh >> i) & 1 for i in range(8)], 2).reshape(len(b), 32)
            q = q + 16 * bits
        if qt[3] == "1":
            return f16(0) * q.double() + f16(2)
        return f16(0) * (q.double() - (16 if qt[1] == "5" else 8))
    if qt in ("Q4_K", "Q5_K"):
        s = b[:, 4:16]
        sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
        mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
        at = 16 if qt == "Q4_K" else 48
        qs = b[:, at:at + 128].view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32)
        if qt == "Q5_K":
            q = q + 16 * torch.stack([(b[:, 16:48] >> j) & 1 for j in range(8)], 1)
        v = (f16(0) * sc.double())[:, :, None] * q.double() - (f16(2) * mn.double())[:, :, None]
        return v.view(-1, 256)
    if qt == "Q6_K":
        ql, qh = b[:, 0:128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 32)
        lo = torch.cat([ql & 15, ql >> 4], 2)  # half, quarter, element
        hi = torch.stack([(qh >> (2 * i)) & 3 for i in range(4)], 2)
        q = (lo.int() + 16 * hi.int() - 32).double().view(-1, 16, 16)
        return ((f16(208) * i8(192, 208))[:, :, None] * q).view(-1, 256)
    at = 16 if qt == "Q2_K" else 32
    qs = b[:, at:at + 64].view(-1, 2, 1, 32)
    q = torch.cat([(qs >> (2 * j)) & 3 for j in range(4)], 2)  # half, quarter, element
    if qt == "Q2_K":
        sc = b[:, 0:16]
        v = (f16(80) * (sc & 15).double())[:, :, None] * q.double().view(-1, 16, 16)
        return (v - (f16(82) * (sc >> 4).double())[:, :, None]).view(-1, 256)
    hm = torch.stack([(b[:, 0:32] >> i) & 1 for i in range(8)], 1).view(-1, 2, 4, 32)
    q = q.int() - 4 * (1 - hm.int())
    raw = b[:, 96:108]
    top = torch.cat([(raw[:, 8:12] >> (2 * i)) & 3 for i in range(4)], 1)
    sc = torch.cat([raw[:, 0:8] & 15, raw[:, 0:8] >> 4], 1).int() + 16 * top.int() - 32
    return ((f16(108) * sc.double())[:, :, None] * q.double().view(-1, 16, 16)).view(-1, 256)


def _quantized(x):
    """The rows x as their Q8_0 blocks hold them: d = amax / 127 and 1 / d rounded to 32 bits,
    codes rint(x / d) with the product rounded to 32 bits."""
    v = x.float().double().view(-1, 32)
    d = (v.abs().amax(1, keepdim=True) / 127.0).float().double()
    inv = torch.where(d > 0, (1.0 / d).float().double(), torch.zeros_like(d))
    q = torch.round((v * inv).float().double()).clamp(-128, 127)
    return (q * d).view(x.shape)


def _product(x, w, qt, n, k):
    """x W^T in 64 bits, x already as the type's kernels take it (Q8_0 or fp32)."""
    b = w.view(n, -1)
    y = torch.empty((x.shape[0], n), device=x.device, dtype=torch.float64)
    step = max(1, (1 << 24) // k)
    for i in range(0, n, step):
        part = b[i:i + step]
        y[:, i:i + step] = x @ _dequantize(part.reshape(-1, BYTES[qt]), qt).view(-1, k).t()
    return y


def _mm(x, w, qt, n, k):
    return _product(x.double() if qt in FLOAT_DOT else _quantized(x), w, qt, n, k)


def _norm(x, w):
    x = x.double()
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * w.double()


def _rope(x, heads, hd, pos0):
    """The angle is the 32-bit one the path computes: pos / base^(i / half)."""
    v = x.double().view(x.shape[0], heads, 2, hd // 2)
    i = torch.arange(hd // 2, device=x.device, dtype=torch.float32)
    inv = torch.pow(torch.tensor(THETA, dtype=torch.float64, device=x.device), (i / (hd // 2)).double())
    p = torch.arange(pos0, pos0 + x.shape[0], device=x.device).double()
    a = (p[:, None] / inv.float().double()).float().double()
    cs, sn = torch.cos(a)[:, None], torch.sin(a)[:, None]
    return torch.stack([v[:, :, 0] * cs - v[:, :, 1] * sn, v[:, :, 0] * sn + v[:, :, 1] * cs],
                       2).view(x.shape)


def _attention(q, kc, vc, pos0, n_head, n_kv, hd):
    m, L, rep = q.shape[0], kc.shape[0], n_head // n_kv
    q, out = q.double().view(m, n_head, hd), []
    mask = torch.arange(L, device=q.device)[None] > (pos0 + torch.arange(m, device=q.device))[:, None]
    for h in range(n_head):
        kh = kc.double().view(L, n_kv, hd)[:, h // rep]
        vh = vc.double().view(L, n_kv, hd)[:, h // rep]
        sc = (q[:, h] @ kh.t()) / math.sqrt(hd)
        out.append(torch.softmax(sc.masked_fill(mask, -math.inf), 1) @ vh)
    return torch.stack(out, 1).view(m, n_head * hd)


def _silu_mul(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def exact(case, seed):
    c, s = case, prepare(case, seed)
    if c["kind"] == "linear":
        y = _mm(s["x"], s["w"], c["type"], c["n"], c["k"])
        return y if s["bias"] is None else y + s["bias"].double()
    if c["kind"] == "head":
        return [_mm(_norm(s["x"], s["norm"]), s["w"], c["type"], c["n"], c["k"])]
    hs = (c["n_head"], c["n_kv"], c["hd"]) if "hd" in c else None
    if c["kind"] == "decode":
        e, ff, pos = c["n_embd"], c["n_ff"], c["pos"]
        q, kv = c["n_head"] * c["hd"], c["n_kv"] * c["hd"]
        t = c["type"]
        x = _dequantize(s["emb"].view(512, -1)[s["id"].long()].reshape(-1, BYTES[t]), t).view(1, e)
        ks, vs = [], []
        for l in s["layers"]:
            h = _norm(x, l["norm1"])
            qv = _rope(_mm(h, l["wq"], t, q, e), c["n_head"], c["hd"], pos)
            ks.append(_rope(_mm(h, l["wk"], t, kv, e), c["n_kv"], c["hd"], pos)[0])
            vs.append(_mm(h, l["wv"], t, kv, e)[0])
            kc = torch.cat([l["kc"][:pos].double(), ks[-1][None]])
            vc = torch.cat([l["vc"][:pos].double(), vs[-1][None]])
            x = x + _mm(_attention(qv, kc, vc, pos, *hs), l["wo"], t, e, q)
            h = _norm(x, l["norm2"])
            h = _silu_mul(_mm(h, l["gate"], t, ff, e), _mm(h, l["up"], t, ff, e))
            x = x + _mm(h, l["down"], c["down"], e, ff)
        return {"logits": _mm(_norm(x, s["norm"]), s["out"], "Q6_K", c["vocab"], e), "x": x,
                "k": ks, "v": vs}
    if c["kind"] == "decode_attention":
        qv = _rope(s["q"], c["n_head"], c["hd"], c["pos"])
        k = _rope(s["k_new"], c["n_kv"], c["hd"], c["pos"])
        kc = torch.cat([s["kc"][:-1].double(), k])
        return {"y": _attention(qv, kc, s["vc"], c["pos"], *hs), "k": k[0]}
    if c["kind"] == "attention_block":
        e, p, q, kv, t = c["n_embd"], c["pos0"], c["n_head"] * c["hd"], c["n_kv"] * c["hd"], c["type"]
        h = _norm(s["x"], s["norm"])
        qv, k, v = (_mm(h, w, t, n, e) for w, n in zip(s["w"], (q, kv, kv)))
        k = _rope(k, c["n_kv"], c["hd"], p)
        kc, vc = torch.cat([s["kc"][:p].double(), k]), torch.cat([s["vc"][:p].double(), v])
        a = _attention(_rope(qv, c["n_head"], c["hd"], p), kc, vc, p, *hs)
        return {"o": _mm(a, s["wo"], t, e, q) + s["x"].double(), "a": a, "k": k, "v": v}
    e, ff = c["n_embd"], c["n_ff"]
    h = _norm(s["x"], s["norm"])
    g, u = _mm(h, s["gate"], c["type"], ff, e), _mm(h, s["up"], c["type"], ff, e)
    return {"o": _mm(_silu_mul(g, u), s["down"], c["down"], e, ff) + s["x"].double(), "gate": g,
            "up": u}
