"""The calls whose time counts: what a program that trains or serves a GPT-style
model has this library do outside its matrix products, through the public Python
entry points (cme213_amd), over the sizes, types and directions it takes.

listed() holds fixed cases, draw(rng) gives more of the same ranges.  A case is a
dict of plain values with a "kind":

  step       the non-GEMM calls of the reference's whole training step, in its
             order: embedding, LN, residual LN, bias+ReLU, residual+bias, softmax
             cross-entropy, every backward, Adam on the flat parameter buffer
  decode     the forward calls for a few rows, as a serving loop issues them for
             one token per sequence, down to the probabilities over the vocabulary
  block      one transformer block's non-GEMM calls, forward and backward
  ln         LayerNorm forward (statistics saved) and backward
  embedding  token + position embedding, forward and backward
  ce         softmax cross-entropy with its gradient, loss left on the device
  softmax    row softmax
  ffn16      bias + activation with 16-bit activation storage
  adam       one optimizer step over a flat parameter buffer

Programs issue the same calls step after step on the same buffers, so the calls
are bound once in prepare() (cme213_amd.bind); Adam, whose step number changes,
is called directly.  Gradients accumulate (`+=`), as the entry points define.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "cme213-final-project_amd"))
import cme213_amd as M  # noqa: E402

EPS = 1e-5
LR, BETA1, BETA2, ADAM_EPS, GRAD_SCALE = 3e-4, 0.9, 0.999, 1e-8, 1.0
FIRST_STEP = 100


def listed():
    return [
        # The reference's default model (B=32, T=64, 128 wide, 65 characters): the
        # smallest step a user runs, where launches and latency count.
        {"name": "step_char_h128", "kind": "step", "B": 32, "T": 64, "C": 128, "V": 65},
        # Its widest build (512) on longer text: an ordinary training step with
        # narrow rows and few distinct ids.
        {"name": "step_char_h512", "kind": "step", "B": 32, "T": 256, "C": 512, "V": 65},
        # Serving 16 sequences of a GPT-2-XL-shaped model, one token each.
        {"name": "decode_xl_16", "kind": "decode", "rows": 16, "C": 1600, "V": 50257},
        # One GPT-2-small block at B=8, T=1024 (bias+GELU, 768 wide).
        {"name": "block_768", "kind": "block", "rows": 8192, "C": 768, "act": "gelu"},
        # One GPT-2-XL-shaped block (1600 wide).
        {"name": "block_1600", "kind": "block", "rows": 4096, "C": 1600, "act": "gelu"},
        # LayerNorm on a ragged batch and a width that is no multiple of 4.
        {"name": "ln_3001x1026", "kind": "ln", "rows": 3001, "cols": 1026},
        # The widest LayerNorm sweep of the benchmark.
        {"name": "ln_32768x4096", "kind": "ln", "rows": 32768, "cols": 4096},
        # GPT-2 embedding, B=16, T=1024, ids uniform over the vocabulary.
        {"name": "emb_gpt2_uniform", "kind": "embedding", "B": 16, "T": 1024, "C": 768,
         "V": 50257, "ids": "uniform"},
        # The same with the id frequencies that text has.
        {"name": "emb_gpt2_text", "kind": "embedding", "B": 16, "T": 1024, "C": 768,
         "V": 50257, "ids": "text"},
        # The training loss at the GPT-2 vocabulary: the largest tensors there are.
        {"name": "ce_8192x50257", "kind": "ce", "rows": 8192, "V": 50257},
        # fp16 activation storage: bias+ReLU to half, half-mask backward.
        {"name": "ffn16_relu_8192x3072", "kind": "ffn16", "rows": 8192, "cols": 3072,
         "act": "relu", "fmt": "half"},
        # Adam over GPT-2 small's parameters.
        {"name": "adam_124m", "kind": "adam", "n": 124439808},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A row width: half the time a multiple of 64, else whatever comes."""
    w = _log(rng, lo, hi)
    return max(64, w // 64 * 64) if rng.random() < 0.5 else w


def _fit(rows, cols, most):
    return max(1, min(rows, most // cols))


def draw(rng):
    kind = rng.choice(["step", "decode", "block", "ln", "ln", "embedding", "embedding", "ce",
                       "softmax", "ffn16", "adam"])
    if kind == "step":
        return {"kind": kind, "B": _log(rng, 4, 64), "T": rng.choice([32, 64, 128, 200, 256]),
                "C": rng.choice([64, 128, 192, 256, 384, 512, 768]),
                "V": rng.choice([65, 96, 256, 1000])}
    if kind == "decode":
        return {"kind": kind, "rows": _log(rng, 1, 128), "C": _log(rng, 8, 64) * 64,
                "V": rng.choice([65, 1000, 32000, 50257, _log(rng, 1000, 60000)])}
    if kind == "block":
        cols = _width(rng, 64, 4096)
        return {"kind": kind, "rows": _fit(_log(rng, 64, 16384), cols, 8 << 20), "C": cols,
                "act": rng.choice(["gelu", "relu"])}
    if kind == "ln":
        cols = _width(rng, 64, 8192)
        return {"kind": kind, "rows": _fit(_log(rng, 64, 65536), cols, 1 << 27), "cols": cols}
    if kind == "embedding":
        cols = _width(rng, 64, 2048)
        t = _log(rng, 16, 2048)
        b = _log(rng, 1, 32)
        return {"kind": kind, "B": _fit(b, t * cols, 24 << 20), "T": t, "C": cols,
                "V": rng.choice([65, 256, 32000, 50257, _log(rng, 65, 60000)]),
                "ids": rng.choice(["uniform", "text"])}
    if kind in ("ce", "softmax"):
        cols = rng.choice([_width(rng, 64, 4096), _log(rng, 1000, 60000), 32000, 50257])
        return {"kind": kind, "rows": _fit(_log(rng, 64, 32768), cols, 1 << 28),
                "V" if kind == "ce" else "cols": cols}
    if kind == "ffn16":
        cols = _width(rng, 128, 8192)
        act = rng.choice(["relu", "gelu"])
        return {"kind": kind, "rows": _fit(_log(rng, 64, 16384), cols, 32 << 20), "cols": cols,
                "act": act, "fmt": "half" if act == "relu" else rng.choice(["half", "bf16"])}
    return {"kind": "adam", "n": _log(rng, 10000, 100000000)}


# ----- inputs -------------------------------------------------------------------

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _randn(g, *shape, scale=1.0, shift=0.0):
    t = torch.randn(shape, device="cuda", generator=g)
    return t.mul_(scale).add_(shift) if (scale, shift) != (1.0, 0.0) else t


def _share(vocab):
    """Zipf-Mandelbrot frequencies of text: the r-th most frequent id's share is
    proportional to 1 / (r + 2.7)."""
    s = 1.0 / (np.arange(1, vocab + 1) + 2.7)
    return s / s.sum()


def _ids(g, n, vocab, how):
    """Token ids: uniform, or with the frequencies of text, the ranks shuffled
    over the vocabulary."""
    if how == "uniform":
        return torch.randint(0, vocab, (n,), device="cuda", generator=g, dtype=torch.int32)
    cdf = torch.from_numpy(np.cumsum(_share(vocab))).to("cuda")
    rank = torch.searchsorted(cdf, torch.rand(n, device="cuda", generator=g, dtype=torch.float64))
    where = torch.randperm(vocab, device="cuda", generator=g)
    return where[rank.clamp_(max=vocab - 1)].to(torch.int32)


def _empty(*shape):
    return torch.empty(shape, device="cuda")


def _zeros(*shape):
    return torch.zeros(shape, device="cuda")


def _step_layout(c):
    C, F = c["C"], 4 * c["C"]
    sizes = [("tok", c["V"] * C), ("pos", c["T"] * C), ("g1", C), ("be1", C), ("g2", C),
             ("be2", C), ("b1", F), ("b2", C)]
    at, out = 0, {}
    for name, n in sizes:
        out[name] = (at, n)
        at += n
    return out, at


def _views(flat, layout):
    return {k: flat[at:at + n] for k, (at, n) in layout.items()}


def _inputs(c, seed):
    """The case's inputs alone, from the seed."""
    g, k = _gen(seed), c["kind"]
    if k == "step":
        R, C, F, V = c["B"] * c["T"], c["C"], 4 * c["C"], c["V"]
        layout, n = _step_layout(c)
        param = _randn(g, n, scale=0.02)
        for name in ("g1", "g2"):
            _views(param, layout)[name].add_(1.0)
        text = _ids(g, R + 1, V, "text")  # the target of a token is the next one
        return {"param": param, "m": _randn(g, n, scale=1e-3),
                "v": _randn(g, n, scale=1e-3).square_(), "ids": text[:-1].clone(),
                "tgt": text[1:].clone(), "proj": _randn(g, R, C, scale=0.8),
                "hid": _randn(g, R, F, scale=1.5), "ffo": _randn(g, R, C, scale=0.6),
                "logits": _randn(g, R, V, scale=2.0), "gres": _randn(g, R, C, scale=0.3),
                "gact": _randn(g, R, F, scale=0.2), "gy2": _randn(g, R, C, scale=0.25),
                "gy1": _randn(g, R, C, scale=0.15)}
    if k == "decode":
        R, C, F, V = c["rows"], c["C"], 4 * c["C"], c["V"]
        d = {"wte": _randn(g, V, C, scale=0.02), "wpe": _randn(g, 1, C, scale=0.02),
             "ids": _ids(g, R, V, "text"), "a": _randn(g, R, C), "mlp": _randn(g, R, C),
             "h": _randn(g, R, F, scale=1.5), "bias": _randn(g, F, scale=0.02),
             "b2": _randn(g, C, scale=0.02), "logits": _randn(g, R, V, scale=2.0)}
        for i in (1, 2):
            d["g%d" % i] = _randn(g, C, scale=0.02, shift=1.0)
            d["be%d" % i] = _randn(g, C, scale=0.02)
        return d
    if k == "block":
        R, C, F = c["rows"], c["C"], 4 * c["C"]
        return {"r0": _randn(g, R, C), "a": _randn(g, R, C), "m": _randn(g, R, C),
                "h": _randn(g, R, F, scale=1.5), "gy1": _randn(g, R, C), "gy2": _randn(g, R, C),
                "gh": _randn(g, R, F), "gres": _randn(g, R, C),
                "g1": _randn(g, C, scale=0.02, shift=1.0), "be1": _randn(g, C, scale=0.02),
                "g2": _randn(g, C, scale=0.02, shift=1.0), "be2": _randn(g, C, scale=0.02),
                "bias": _randn(g, F, scale=0.02)}
    if k == "ln":
        R, C = c["rows"], c["cols"]
        return {"x": _randn(g, R, C), "dy": _randn(g, R, C),
                "gamma": _randn(g, C, scale=0.02, shift=1.0), "beta": _randn(g, C, scale=0.02)}
    if k == "embedding":
        return {"wte": _randn(g, c["V"], c["C"], scale=0.02),
                "wpe": _randn(g, c["T"], c["C"], scale=0.02),
                "ids": _ids(g, c["B"] * c["T"], c["V"], c["ids"]),
                "dout": _randn(g, c["B"] * c["T"], c["C"])}
    if k == "ce":
        return {"logits": _randn(g, c["rows"], c["V"], scale=2.0),
                "tgt": _ids(g, c["rows"], c["V"], "text")}
    if k == "softmax":
        return {"x": _randn(g, c["rows"], c["cols"], scale=2.0)}
    if k == "ffn16":
        R, F = c["rows"], c["cols"]
        return {"h": _randn(g, R, F, scale=1.5), "dh": _randn(g, R, F),
                "bias": _randn(g, F, scale=0.02)}
    if k == "adam":
        n = c["n"]
        return {"param": _randn(g, n, scale=0.02), "grad": _randn(g, n, scale=1e-3),
                "m": _randn(g, n, scale=1e-4), "v": _randn(g, n, scale=1e-3).square_()}
    raise ValueError(k)


# ----- one pass -----------------------------------------------------------------

def prepare(c, seed):
    d, k = _inputs(c, seed), c["kind"]
    bind = M.bind
    if k == "step":
        B, T, C, V = c["B"], c["T"], c["C"], c["V"]
        R, F = B * T, 4 * C
        layout, n = _step_layout(c)
        p = _views(d["param"], layout)
        grad = _zeros(n)
        q = _views(grad, layout)
        o = {"emb": _empty(R, C), "y1": _empty(R, C), "m1": _empty(R), "s1": _empty(R),
             "r1": _empty(R, C), "y2": _empty(R, C), "m2": _empty(R), "s2": _empty(R),
             "act": _empty(R, F), "r2": _empty(R, C), "dlogits": _empty(R, V),
             "losses": _empty(R), "loss": _empty(1), "ghid": _empty(R, F), "gres": d["gres"],
             "grad": grad, "param": d["param"], "m": d["m"], "v": d["v"],
             "norm": _empty(1), "clip": _empty(1)}
        calls = [
            bind("mi_embedding_forward", p["tok"], d["ids"], o["emb"], R, C, V),
            bind("mi_pos_embedding_forward", p["pos"], o["emb"], B, T, C),
            bind("mi_layernorm_forward_save", o["emb"], p["g1"], p["be1"], o["y1"], o["m1"],
                 o["s1"], R, C, EPS),
            bind("mi_residual_layernorm_forward_save", o["emb"], d["proj"], p["g2"], p["be2"],
                 o["r1"], o["y2"], o["m2"], o["s2"], R, C, EPS),
            bind("mi_bias_relu_forward", d["hid"], p["b1"], o["act"], R, F),
            bind("mi_residual_add_with_bias", o["r1"], d["ffo"], p["b2"], o["r2"], R, C),
            bind("mi_cross_entropy_forward_v2", d["logits"], d["tgt"], o["dlogits"],
                 o["losses"], o["loss"], R, V),
            bind("mi_bias_backward", d["gres"], q["b2"], R, C),
            bind("mi_relu_backward_with_bias_backward", o["act"], d["gact"], o["ghid"], q["b1"],
                 R, F),
            bind("mi_layernorm_backward_residual", d["gy2"], o["r1"], o["m2"], o["s2"], p["g2"],
                 d["gres"], q["g2"], q["be2"], R, C),
            bind("mi_layernorm_backward_residual", d["gy1"], o["emb"], o["m1"], o["s1"], p["g1"],
                 d["gres"], q["g1"], q["be1"], R, C),
            bind("mi_embedding_backward", d["gres"], d["ids"], q["tok"], R, C, V),
            bind("mi_pos_embedding_backward", d["gres"], q["pos"], B, T, C),
        ]
        return {"kind": k, "calls": calls, "out": o, "n": n, "step": FIRST_STEP, "grad": grad,
                "keep": d}
    if k == "decode":
        R, C, V = c["rows"], c["C"], c["V"]
        F = 4 * C
        o = {"emb": _empty(R, C), "r1": _empty(R, C), "y1": _empty(R, C), "m1": _empty(R),
             "s1": _empty(R), "act": _empty(R, F), "r2": _empty(R, C), "y2": _empty(R, C),
             "prob": _empty(R, V)}
        calls = [
            bind("mi_embedding_pos_forward", d["wte"], d["wpe"], d["ids"], o["emb"], R, 1, C, V),
            bind("mi_residual_layernorm_forward_save", o["emb"], d["a"], d["g1"], d["be1"],
                 o["r1"], o["y1"], o["m1"], o["s1"], R, C, EPS),
            bind("mi_bias_gelu_forward", d["h"], d["bias"], o["act"], R, F),
            bind("mi_residual_add_with_bias", o["r1"], d["mlp"], d["b2"], o["r2"], R, C),
            bind("mi_layernorm_forward", o["r2"], d["g2"], d["be2"], o["y2"], R, C, EPS),
            bind("mi_softmax_forward", d["logits"], o["prob"], R, V),
        ]
    elif k == "block":
        R, C = c["rows"], c["C"]
        F = 4 * C
        o = {"r1": _empty(R, C), "y1": _empty(R, C), "m1": _empty(R), "s1": _empty(R),
             "r2": _empty(R, C), "y2": _empty(R, C), "m2": _empty(R), "s2": _empty(R),
             "act": _empty(R, F), "gh": _empty(R, F), "dbias": _zeros(F), "gres": d["gres"],
             "dg1": _zeros(C), "db1": _zeros(C), "dg2": _zeros(C), "db2": _zeros(C)}
        calls = [
            bind("mi_residual_layernorm_forward_save", d["r0"], d["a"], d["g1"], d["be1"],
                 o["r1"], o["y1"], o["m1"], o["s1"], R, C, EPS),
            bind("mi_residual_layernorm_forward_save", o["r1"], d["m"], d["g2"], d["be2"],
                 o["r2"], o["y2"], o["m2"], o["s2"], R, C, EPS)]
        if c["act"] == "gelu":
            calls += [bind("mi_bias_gelu_forward", d["h"], d["bias"], o["act"], R, F),
                      bind("mi_gelu_backward_with_bias_backward", d["h"], d["bias"], d["gh"],
                           o["gh"], o["dbias"], R, F)]
        else:
            calls += [bind("mi_bias_relu_forward", d["h"], d["bias"], o["act"], R, F),
                      bind("mi_relu_backward_with_bias_backward", o["act"], d["gh"], o["gh"],
                           o["dbias"], R, F)]
        calls += [
            bind("mi_layernorm_backward_residual", d["gy2"], o["r2"], o["m2"], o["s2"], d["g2"],
                 d["gres"], o["dg2"], o["db2"], R, C),
            bind("mi_layernorm_backward_residual", d["gy1"], o["r1"], o["m1"], o["s1"], d["g1"],
                 d["gres"], o["dg1"], o["db1"], R, C)]
    elif k == "ln":
        R, C = c["rows"], c["cols"]
        o = {"y": _empty(R, C), "mean": _empty(R), "rstd": _empty(R), "dx": _empty(R, C),
             "dgamma": _zeros(C), "dbeta": _zeros(C)}
        calls = [
            bind("mi_layernorm_forward_save", d["x"], d["gamma"], d["beta"], o["y"], o["mean"],
                 o["rstd"], R, C, EPS),
            bind("mi_layernorm_backward", d["dy"], d["x"], o["mean"], o["rstd"], d["gamma"],
                 o["dx"], o["dgamma"], o["dbeta"], R, C)]
    elif k == "embedding":
        B, T, C, V = c["B"], c["T"], c["C"], c["V"]
        o = {"out": _empty(B * T, C), "dwte": _zeros(V, C), "dwpe": _zeros(T, C)}
        calls = [
            bind("mi_embedding_pos_forward", d["wte"], d["wpe"], d["ids"], o["out"], B, T, C, V),
            bind("mi_embedding_pos_backward", d["dout"], d["ids"], o["dwte"], o["dwpe"], B, T, C,
                 V)]
    elif k == "ce":
        R, V = c["rows"], c["V"]
        o = {"grad": _empty(R, V), "losses": _empty(R), "loss": _empty(1)}
        calls = [bind("mi_cross_entropy_forward_v2", d["logits"], d["tgt"], o["grad"],
                      o["losses"], o["loss"], R, V)]
    elif k == "softmax":
        o = {"p": _empty(c["rows"], c["cols"])}
        calls = [bind("mi_softmax_forward", d["x"], o["p"], c["rows"], c["cols"])]
    elif k == "ffn16":
        R, F = c["rows"], c["cols"]
        dt = torch.float16 if c["fmt"] == "half" else torch.bfloat16
        a16 = torch.empty(R, F, device="cuda", dtype=dt)
        if c["act"] == "relu":
            o = {"a16": a16, "gin": _empty(R, F), "dbias": _zeros(F)}
            calls = [bind("mi_bias_relu_forward_to_half", d["h"], d["bias"], a16, R, F),
                     bind("mi_relu_backward_with_bias_backward_half_mask", a16, d["dh"],
                          o["gin"], o["dbias"], R, F)]
        else:
            # the activation kept in 16 bits, and widened again where it is used
            o = {"a16": a16, "a32": _empty(R, F), "gin": _empty(R, F), "dbias": _zeros(F)}
            f = "half" if c["fmt"] == "half" else "bf16"
            calls = [bind("mi_bias_gelu_forward_to_" + f, d["h"], d["bias"], a16, R, F),
                     bind("mi_%s_to_float" % f, a16, o["a32"], R * F),
                     bind("mi_gelu_backward_with_bias_backward", d["h"], d["bias"], d["dh"],
                          o["gin"], o["dbias"], R, F)]
    else:
        o = {"param": d["param"], "m": d["m"], "v": d["v"], "norm": _empty(1), "clip": _empty(1)}
        return {"kind": k, "out": o, "grad": d["grad"], "n": c["n"], "step": FIRST_STEP}
    return {"kind": k, "calls": calls, "out": o, "keep": d}


def run(s):
    o = s["out"]
    if s["kind"] == "step":
        s["grad"].zero_()
    if s["kind"] != "adam":
        for call in s["calls"]:
            call()
    if s["kind"] in ("step", "adam"):
        M.adam_update(o["param"], s["grad"], o["m"], o["v"], s["n"], LR, BETA1, BETA2, ADAM_EPS,
                      s["step"], GRAD_SCALE, o["norm"], o["clip"])
        s["step"] += 1
    return o


# ----- what a pass cannot do without ----------------------------------------------

def work(c):
    """Every tensor that a call reads counts once, every tensor that it writes once;
    an activation or gradient updated in place counts twice."""
    k = c["kind"]

    def ln(R, C):
        return 2 * R * C + 2 * R + 2 * C

    def res_ln(R, C):
        return 4 * R * C + 2 * R + 2 * C

    def ln_bwd(R, C, streams):
        return streams * R * C + 2 * R + 5 * C

    def adam(n):
        return 8 * n

    if k == "step":
        B, T, C, V = c["B"], c["T"], c["C"], c["V"]
        R, F = B * T, 4 * C
        n = _step_layout(c)[1]
        tab = float((1.0 - (1.0 - _share(V)) ** R).sum()) * C
        w = n                                               # gradients cleared
        w += R + tab + R * C + 2 * R * C + T * C            # embedding, position add
        w += ln(R, C) + res_ln(R, C)
        w += 2 * R * F + F + 3 * R * C + C                  # bias+ReLU, residual+bias
        w += 2 * R * V + 3 * R                              # cross-entropy
        w += R * C + 2 * C + 3 * R * F + 2 * F              # dbias, ReLU backward
        w += 2 * ln_bwd(R, C, 4)
        w += R * C + R + 2 * tab + R * C + 2 * T * C        # embedding backward
        w += adam(n)
        elems = R * (30 * C + 10 * F + 8 * V) + 15 * n
    elif k == "decode":
        R, C, V = c["rows"], c["C"], c["V"]
        F = 4 * C
        w = R + 2 * R * C + C + res_ln(R, C) + 2 * R * F + F + 3 * R * C + C
        w += 2 * R * C + 2 * C + 2 * R * V
        elems = R * (20 * C + 12 * F + 6 * V)
    elif k == "block":
        R, C = c["rows"], c["C"]
        F = 4 * C
        w = 2 * res_ln(R, C) + 5 * R * F + 4 * F + 2 * ln_bwd(R, C, 4)
        elems = R * (50 * C + 35 * F)
    elif k == "ln":
        R, C = c["rows"], c["cols"]
        w = ln(R, C) + ln_bwd(R, C, 3)
        elems = 25 * R * C
    elif k == "embedding":
        R, C, T, V = c["B"] * c["T"], c["C"], c["T"], c["V"]
        share = _share(V) if c["ids"] == "text" else np.full(V, 1.0 / V)
        tab = float((1.0 - (1.0 - share) ** R).sum()) * C  # table rows touched, expected
        w = R + tab + R * C + T * C + R + R * C + 2 * tab + 2 * T * C
        elems = 3 * R * C
    elif k == "ce":
        w = 2 * c["rows"] * c["V"] + 2 * c["rows"]
        elems = 7 * c["rows"] * c["V"]
    elif k == "softmax":
        w = 2 * c["rows"] * c["cols"]
        elems = 5 * c["rows"] * c["cols"]
    elif k == "ffn16":
        N, F = c["rows"] * c["cols"], c["cols"]
        w = (4 * N + 3 * F) if c["act"] == "relu" else (6 * N + 4 * F)  # two halves a word
        elems = 4 * N if c["act"] == "relu" else 35 * N
    else:
        w, elems = adam(c["n"]), 15 * c["n"]
    return {"bytes": 4.0 * w, "flops": float(elems)}


def tolerance(c):
    """fp32 sums in another order: 1e-7 to 2.5e-7 off the 64-bit result as measured,
    over the vector, on every kind.  16-bit outputs carry their format's rounding
    (2.1e-4 in half) and may round the other way where a value lies between two."""
    if c["kind"] == "ffn16":
        return {"rel": 2e-4, "max": 1e-2}
    return {"rel": 1e-6, "max": 1e-4}


# ----- the same in 64 bits ---------------------------------------------------------

def _ln(x, gamma, beta):
    mean = x.mean(1)
    rstd = 1.0 / torch.sqrt(x.var(1, unbiased=False) + EPS)
    return (x - mean[:, None]) * rstd[:, None] * gamma + beta, mean, rstd


def _ln_bwd(g, x, mean, rstd, gamma):
    xh = (x - mean[:, None]) * rstd[:, None]
    dgamma, dbeta = (g * xh).sum(0), g.sum(0)
    g = g * gamma
    dx = rstd[:, None] * (g - g.mean(1, keepdim=True) - xh * (g * xh).mean(1, keepdim=True))
    return dx, dgamma, dbeta


_Z = math.sqrt(2.0 / math.pi)


def _gelu(u):
    return u / (1.0 + torch.exp(-2.0 * _Z * (u + 0.044715 * u ** 3)))


def _gelu_grad(u):
    s = 1.0 / (1.0 + torch.exp(-2.0 * _Z * (u + 0.044715 * u ** 3)))
    return s + 2.0 * u * s * (1.0 - s) * _Z * (1.0 + 3 * 0.044715 * u ** 2)


def _adam(param, grad, m, v, step):
    f = lambda x: float(np.float32(x))  # noqa: E731  the values the kernel is given
    b1, b2 = f(BETA1), f(BETA2)
    norm = grad.square().sum()
    most = 1.0 / GRAD_SCALE
    clip = torch.where(norm.sqrt() > most, most / norm.sqrt(), torch.ones_like(norm))
    g = grad * GRAD_SCALE * clip
    m = b1 * m + (1.0 - b1) * g
    v = b2 * v + (1.0 - b2) * g * g
    mh, vh = m / (1.0 - b1 ** step), v / (1.0 - b2 ** step)
    param = param - f(LR) * mh / (vh.sqrt() + f(ADAM_EPS))
    return param, m, v, norm.reshape(1), clip.reshape(1)


def _ce(logits, tgt):
    """loss = -log(p + 1e-9) per row, p = e / (sum e + 1e-9); gradient of the mean."""
    e = torch.exp(logits - logits.max(1, keepdim=True).values)
    p = e.div_(e.sum(1, keepdim=True) + 1e-9)
    t = tgt.long()[:, None]
    losses = -torch.log(p.gather(1, t)[:, 0] + 1e-9)
    p.scatter_add_(1, t, torch.full_like(p[:, :1], -1.0))
    return p.div_(logits.shape[0]), losses, losses.mean().reshape(1)


def exact(c, seed):
    d = _inputs(c, seed)
    d = {a: t if t.dtype == torch.int32 else t.double() for a, t in d.items()}
    k = c["kind"]
    if k == "step":
        B, T, C, V = c["B"], c["T"], c["C"], c["V"]
        layout, n = _step_layout(c)
        p = _views(d["param"], layout)
        grad = torch.zeros(n, device="cuda", dtype=torch.float64)
        q = _views(grad, layout)
        ids = d["ids"].long()
        o = {"emb": p["tok"].view(V, C)[ids] + p["pos"].view(T, C).repeat(B, 1)}
        o["y1"], o["m1"], o["s1"] = _ln(o["emb"], p["g1"], p["be1"])
        o["r1"] = o["emb"] + d["proj"]
        o["y2"], o["m2"], o["s2"] = _ln(o["r1"], p["g2"], p["be2"])
        o["act"] = torch.relu(d["hid"] + p["b1"])
        o["r2"] = o["r1"] + d["ffo"] + p["b2"]
        o["dlogits"], o["losses"], o["loss"] = _ce(d["logits"], d["tgt"])
        gres = d["gres"]
        q["b2"].copy_(gres.sum(0))
        o["ghid"] = torch.where(o["act"] > 0, d["gact"], torch.zeros_like(d["gact"]))
        q["b1"].copy_(o["ghid"].sum(0))
        dx, dg, db = _ln_bwd(d["gy2"], o["r1"], o["m2"], o["s2"], p["g2"])
        gres = gres + dx
        q["g2"].copy_(dg), q["be2"].copy_(db)
        dx, dg, db = _ln_bwd(d["gy1"], o["emb"], o["m1"], o["s1"], p["g1"])
        gres = gres + dx
        q["g1"].copy_(dg), q["be1"].copy_(db)
        q["tok"].view(V, C).index_add_(0, ids, gres)
        q["pos"].copy_(gres.view(B, T, C).sum(0).reshape(-1))
        o["gres"], o["grad"] = gres, grad
        o["param"], o["m"], o["v"], o["norm"], o["clip"] = _adam(d["param"], grad, d["m"], d["v"],
                                                                 FIRST_STEP)
        return o
    if k == "decode":
        o = {"emb": d["wte"][d["ids"].long()] + d["wpe"]}
        o["r1"] = o["emb"] + d["a"]
        o["y1"], o["m1"], o["s1"] = _ln(o["r1"], d["g1"], d["be1"])
        o["act"] = _gelu(d["h"] + d["bias"])
        o["r2"] = o["r1"] + d["mlp"] + d["b2"]
        o["y2"] = _ln(o["r2"], d["g2"], d["be2"])[0]
        o["prob"] = torch.softmax(d["logits"], 1)
        return o
    if k == "block":
        o = {"r1": d["r0"] + d["a"]}
        o["y1"], o["m1"], o["s1"] = _ln(o["r1"], d["g1"], d["be1"])
        o["r2"] = o["r1"] + d["m"]
        o["y2"], o["m2"], o["s2"] = _ln(o["r2"], d["g2"], d["be2"])
        u = d["h"] + d["bias"]
        if c["act"] == "gelu":
            o["act"], o["gh"] = _gelu(u), d["gh"] * _gelu_grad(u)
        else:
            o["act"] = torch.relu(u)
            o["gh"] = torch.where(u > 0, d["gh"], torch.zeros_like(u))
        o["dbias"] = o["gh"].sum(0)
        dx2, o["dg2"], o["db2"] = _ln_bwd(d["gy2"], o["r2"], o["m2"], o["s2"], d["g2"])
        dx1, o["dg1"], o["db1"] = _ln_bwd(d["gy1"], o["r1"], o["m1"], o["s1"], d["g1"])
        o["gres"] = d["gres"] + dx2 + dx1
        return o
    if k == "ln":
        o = {}
        o["y"], o["mean"], o["rstd"] = _ln(d["x"], d["gamma"], d["beta"])
        o["dx"], o["dgamma"], o["dbeta"] = _ln_bwd(d["dy"], d["x"], o["mean"], o["rstd"],
                                                   d["gamma"])
        return o
    if k == "embedding":
        ids, g = d["ids"].long(), d["dout"]
        dwte = torch.zeros_like(d["wte"]).index_add_(0, ids, g)
        return {"out": d["wte"][ids] + d["wpe"].repeat(c["B"], 1), "dwte": dwte,
                "dwpe": g.view(c["B"], c["T"], c["C"]).sum(0)}
    if k == "ce":
        grad, losses, loss = _ce(d["logits"], d["tgt"])
        return {"grad": grad, "losses": losses, "loss": loss}
    if k == "softmax":
        return {"p": torch.softmax(d["x"], 1)}
    if k == "ffn16":
        u = d["h"] + d["bias"]
        if c["act"] == "relu":
            # the stored activation is the mask: a positive u that rounds to zero in
            # half does not count
            a = torch.relu(u)
            gin = torch.where(a.to(torch.float16) > 0, d["dh"], torch.zeros_like(u))
            return {"a16": a, "gin": gin, "dbias": gin.sum(0)}
        a = _gelu(u)
        gin = d["dh"] * _gelu_grad(u)
        return {"a16": a, "a32": a, "gin": gin, "dbias": gin.sum(0)}
    param, m, v, norm, clip = _adam(d["param"], d["grad"], d["m"], d["v"], FIRST_STEP)
    return {"param": param, "m": m, "v": v, "norm": norm, "clip": clip}
