"""Workloads that the framework's performance is measured on.

Every case goes through a public entry point: the C ABI of include/cdml.h (as
cdml.native binds it, on device pointers and the caller's stream) for single
layers, and the device engines of the host module (DeviceLanguageModel,
DeviceTrainer) for whole models.  The kinds:

  lm           a small text model scores a batch of prompts and continues them greedily
  lm_train     one training step of such a model (forward, loss, backward, clipping, update)
  series       a time-series regression model's forward pass over a batch of windows
  attn         one multi-head attention layer's forward pass (prefill)
  attn_bwd     that layer's backward pass, from the forward's saved tensors
  ffn          one feed-forward block's inference pass with its residual LayerNorm
  ffn_train    that block's training pass: forward with its cache, then backward
  decode_attn  single-query attention over a cached K/V, whole batch
  decode       one decoder layer's step for a few sequences that are being generated

A case is a dict of plain values; prepare() makes its inputs on the GPU from the
seed alone, run() is one pass, exact() the same results in float64 from plain torch.
"""
from __future__ import annotations

import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "callaghandev.ml_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from cdml import host, native  # noqa: E402

DEV = "cuda"
EPS = 1e-5
ACTS = ("relu", "leakyrelu", "swish", "tanh", "sigmoid")
KINKED = ("relu", "leakyrelu")  # activations whose derivative jumps at 0


def listed():
    return [
        # the README's text model: four prompts scored, then 20 tokens generated for each
        {"name": "lm_small", "kind": "lm", "batch": 4, "len": 32, "new": 20, "vocab": 200, "dim": 64, "heads": 4,
         "layers": 2, "ff": 128, "act": "relu", "max_seq": 64},
        # the same model's training step on four sequences of 64 tokens
        {"name": "lm_train_small", "kind": "lm_train", "batch": 4, "len": 64, "vocab": 200, "dim": 64, "heads": 4,
         "layers": 2, "ff": 128, "act": "relu", "max_seq": 64},
        # a regression transformer over 256 windows of 512 steps, host arrays in and out
        {"name": "series_model", "kind": "series", "batch": 256, "len": 512, "features": 5, "dim": 256, "heads": 8,
         "layers": 6, "ff": 1024},
        # long-context prefill: one layer over four sequences of 4096 tokens
        {"name": "attn_long", "kind": "attn", "batch": 4, "len": 4096, "heads": 16, "hd": 64, "mask": "causal"},
        # an ordinary prefill
        {"name": "attn_mid", "kind": "attn", "batch": 16, "len": 1024, "heads": 8, "hd": 64, "mask": "causal"},
        # a few sequences of an odd length under an explicit sliding-window mask, head dim 40
        {"name": "attn_ragged", "kind": "attn", "batch": 3, "len": 777, "heads": 5, "hd": 40, "mask": "window"},
        # the backward passes that a long-context and a windowed training step spend their time in (a window of
        # 512 steps trains on 511 inputs)
        {"name": "attn_bwd_long", "kind": "attn_bwd", "batch": 4, "len": 4096, "heads": 16, "hd": 64},
        {"name": "attn_bwd_windows", "kind": "attn_bwd", "batch": 256, "len": 511, "heads": 8, "hd": 32},
        # the feed-forward block of the long-context layer, and the training pass of the windowed model's
        {"name": "ffn_long", "kind": "ffn", "rows": 16384, "dim": 1024, "ff": 4096, "act": "relu"},
        {"name": "ffn_train_windows", "kind": "ffn_train", "rows": 130816, "dim": 256, "ff": 1024, "act": "relu"},
        # serving: 64 sequences with 8192 cached keys each, and one layer's step for eight sequences
        {"name": "decode_attn_long", "kind": "decode_attn", "batch": 64, "keys": 8192, "heads": 16, "hd": 128,
         "full": True},
        {"name": "decode_layer", "kind": "decode", "batch": 8, "keys": 2048, "heads": 16, "hd": 64, "ff": 4096},
    ]


def _log(rng, lo, hi):
    """A whole number spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# No drawn case costs more than the largest listed one of its sort.
_MOST = {"flops": 1.1e12, "bytes": 8.6e9}


def draw(rng):
    while True:
        case = _draw(rng)
        w = work(case)
        if w["flops"] <= _MOST["flops"] and w["bytes"] <= _MOST["bytes"]:
            return case


def _draw(rng):
    kind = rng.choice(("lm", "lm_train", "series", "attn", "attn", "attn_bwd", "attn_bwd", "ffn", "ffn_train",
                       "decode_attn", "decode"))
    if kind in ("lm", "lm_train"):
        heads, hd, n = rng.choice((2, 4, 8)), rng.choice((8, 16, 24, 32)), _log(rng, 8, 128)
        case = {"kind": kind, "batch": _log(rng, 1, 16), "len": n, "vocab": _log(rng, 50, 2000), "dim": heads * hd,
                "heads": heads, "layers": rng.randint(1, 3), "ff": heads * hd * rng.choice((2, 4)),
                "act": rng.choice(ACTS), "max_seq": 192}
        if kind == "lm":
            case["new"] = _log(rng, 1, 48)
        elif case["act"] in KINKED:  # one derivative at a kink shows in all of a small model's gradients
            case["act"] = rng.choice(("swish", "tanh"))
        return case
    if kind == "series":
        heads = rng.choice((4, 8))
        dim = heads * rng.choice((16, 32, 64))
        return {"kind": kind, "batch": _log(rng, 1, 256), "len": _log(rng, 16, 1024), "features": rng.randint(1, 12),
                "dim": dim, "heads": heads, "layers": rng.randint(1, 6), "ff": dim * rng.choice((2, 4))}
    heads, hd = rng.choice((1, 2, 5, 8, 12, 16)), rng.choice((16, 32, 40, 64, 64, 96, 128))
    if kind == "attn":
        return {"kind": kind, "batch": _log(rng, 1, 64), "len": _log(rng, 16, 4096), "heads": heads, "hd": hd,
                "mask": rng.choice(("causal", "causal", "none", "window"))}
    if kind == "attn_bwd":
        return {"kind": kind, "batch": _log(rng, 1, 64), "len": _log(rng, 16, 4096), "heads": heads, "hd": hd}
    if kind in ("ffn", "ffn_train"):
        dim = rng.choice((64, 96, 200, 256, 512, 1000, 1024, 2048))
        return {"kind": kind, "rows": _log(rng, 32, 32768), "dim": dim, "ff": dim * rng.choice((2, 4)),
                "act": rng.choice(ACTS)}
    if kind == "decode_attn":
        return {"kind": kind, "batch": _log(rng, 1, 64), "keys": _log(rng, 64, 8192), "heads": heads, "hd": hd,
                "full": rng.random() < 0.5}
    return {"kind": kind, "batch": _log(rng, 1, 32), "keys": _log(rng, 64, 4096), "heads": heads, "hd": hd,
            "ff": 4 * heads * hd}


def work(case):
    """Bytes (each input read once, each output written once) and flops (matrix products, two per
    multiply-add, visible query-key pairs only) of one pass."""
    c, k = case, case["kind"]
    if k in ("lm", "lm_train", "series"):
        B, L, D, FF, NL = c["batch"], c["len"], c["dim"], c["ff"], c["layers"]
        V, F = (c["vocab"], 0) if k != "series" else (1, c["features"])
        per_row = NL * (8 * D * D + 4 * D * FF) + 2 * D * V + 2 * F * D
        params = NL * (4 * D * D + 2 * D * FF + 9 * D + FF) + V * (D + 1) + (V * D if k != "series" else D * (F + 1))
        if k == "lm_train":
            L -= 1
        core = NL * 4 * D * (L * (L + 1) // 2)
        flops, size = B * (L * per_row + core), 4 * (params + B * L * (F + 1) + B * L * V)
        if k == "lm":
            flops += sum(B * (per_row + NL * 4 * D * (L + i)) for i in range(c["new"] - 1))
            size += 4 * B * c["new"]
        if k == "lm_train":
            flops, size = 3 * flops, 4 * (3 * params + 2 * B * L)
        return {"bytes": size, "flops": flops}
    if k in ("attn", "attn_bwd"):
        B, L, D = c["batch"], c["len"], c["heads"] * c["hd"]
        rows = B * L
        if k == "attn":
            W = _window(L)
            pairs = {"causal": L * (L + 1) // 2, "none": L * L, "window": W * L - W * (W - 1) // 2}[c["mask"]]
            mask = L * L if c["mask"] == "window" else 0
            return {"bytes": 4 * (2 * rows * D + 4 * D * D + 4 * D) + mask, "flops": 8 * rows * D * D + 4 * B * D * pairs}
        return {"bytes": 4 * (7 * rows * D + B * c["heads"] * L + 8 * D * D + 4 * D),
                "flops": 16 * rows * D * D + 8 * B * D * (L * (L + 1) // 2)}
    if k in ("ffn", "ffn_train"):
        R, D, FF = c["rows"], c["dim"], c["ff"]
        if k == "ffn":
            return {"bytes": 4 * (2 * R * D + 2 * D * FF + FF + 3 * D), "flops": 4 * R * D * FF}
        return {"bytes": 4 * (4 * R * D + 2 * (2 * D * FF + FF + 3 * D)), "flops": 12 * R * D * FF}
    B, D = c["batch"], c["heads"] * c["hd"]
    keys = sum(_kv_lens(c))
    if k == "decode_attn":
        return {"bytes": 4 * (2 * keys * D + 2 * B * D), "flops": 4 * keys * D}
    FF = c["ff"]
    return {"bytes": 4 * (2 * keys * D + 4 * D * D + 2 * D * FF + 2 * B * D + 2 * B * D),
            "flops": 4 * keys * D + B * (8 * D * D + 4 * D * FF)}


def tolerance(case):
    if case["kind"] == "ffn_train" and case["act"] in KINKED:
        # a pre-activation within rounding of 0 may take either side's derivative: about one in a million does,
        # and the whole difference of the gradients below it comes from those
        return {"rel": 1.6e-3}
    return TOLERANCE[case["kind"]]


# Relative error (2-norm), and the largest error against the result's root mean square: about four times what
# was seen against float64 over the listed and some drawn cases.  The attention layers' errors are mostly the
# rotary angles' (position / base^(2p / head_dim) in 32 bits, at positions up to 4095).
TOLERANCE = {
    "lm": {"rel": 2e-6, "max": 2e-5, "differ": 0.1},
    "lm_train": {"rel": 1e-5, "max": 4e-5},
    "series": {"rel": 6e-6, "max": 4e-5},
    "attn": {"rel": 1.4e-5, "max": 1.6e-4},
    "attn_bwd": {"rel": 7e-5, "max": 7e-4},
    "ffn": {"rel": 2e-6, "max": 2e-5},
    "ffn_train": {"rel": 4e-6, "max": 4e-5},
    "decode_attn": {"rel": 2e-6, "max": 1e-5},
    "decode": {"rel": 3e-6, "max": 1.2e-3},
}


# ---- inputs ---------------------------------------------------------------

class _Rand:
    """Seeded inputs, drawn on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV)
        self.g.manual_seed(seed)

    def normal(self, *shape, std=1.0):
        t = torch.empty(shape, device=DEV, dtype=torch.float32)
        return t.normal_(0.0, std, generator=self.g)

    def xavier(self, rows, cols):
        a = math.sqrt(6.0 / (rows + cols))
        return torch.empty((rows, cols), device=DEV, dtype=torch.float32).uniform_(-a, a, generator=self.g)

    def ints(self, high, *shape):
        return torch.randint(0, high, shape, device=DEV, dtype=torch.int32, generator=self.g)


def _empty(*shape):
    return torch.empty(shape, device=DEV, dtype=torch.float32)


def _window(n):
    """Keys that a query sees under the sliding-window mask of an n-token sequence."""
    return max(1, n // 3)


def _mask(c):
    """uint8 [len, len], or None where no explicit mask is passed."""
    if c["mask"] != "window":
        return None
    i = torch.arange(c["len"], device=DEV)
    d = i[:, None] - i[None, :]
    return ((d >= 0) & (d < _window(c["len"]))).to(torch.uint8).contiguous()


def _kv_lens(c):
    """Cached keys of each sequence: all of them, or lengths spread over the cache."""
    B, T = c["batch"], c["keys"]
    if c.get("full"):
        return [T] * B
    return [max(1, T - (i * 37) % (T // 2 + 1)) for i in range(B)]


def _weights(c, seed):
    """A model's weights as the host module loads them (numpy)."""
    r = _Rand(seed)
    D, FF = c["dim"], c["ff"]

    def mat(rows, cols):
        return r.xavier(rows, cols).cpu().numpy()

    def vec(n, centre=0.0):
        return (r.normal(n, std=0.1) + centre).cpu().numpy()

    layers = [{"wq": mat(D, D), "wk": mat(D, D), "wv": mat(D, D), "wo": mat(D, D),
               "bq": vec(D), "bk": vec(D), "bv": vec(D), "bo": vec(D),
               "ln1_g": vec(D, 1.0), "ln1_b": vec(D), "ln2_g": vec(D, 1.0), "ln2_b": vec(D),
               "ffn_w1": mat(FF, D), "ffn_b1": vec(FF), "ffn_w2": mat(D, FF), "ffn_b2": vec(D)}
              for _ in range(c["layers"])]
    w = {"layers": layers}
    if c["kind"] == "series":
        w.update(input_proj=mat(D, c["features"]), input_bias=vec(D), out_proj=mat(1, D), out_bias=vec(1),
                 token_embedding=mat(2, D))
    else:
        w.update(token_embedding=mat(c["vocab"], D), out_proj=mat(c["vocab"], D), out_bias=vec(c["vocab"]))
    return w


def _config(c):
    cfg = {"dim": c["dim"], "heads": c["heads"], "layers": c["layers"], "ff": c["ff"]}
    if c["kind"] == "series":
        cfg.update(max_seq=c["len"], discrete=False, input_dim=c["features"], output_dim=1)
    else:
        cfg.update(vocab=c["vocab"], max_seq=c["max_seq"], activation=native.ACT[c["act"]])
    return cfg


def _tokens(c, seed):
    return _Rand(seed + 7).ints(c["vocab"], c["batch"], c["len"]).cpu().numpy()


def _windows(c, seed):
    """Random walks in [0, 1], one per feature: [batch * len, features]."""
    x = _Rand(seed + 7).normal(c["batch"], c["len"], c["features"], std=0.02).cumsum(1)
    lo, hi = x.amin(1, keepdim=True), x.amax(1, keepdim=True)
    return ((x - lo) / (hi - lo).clamp_min(1e-6)).reshape(-1, c["features"]).cpu().numpy()


def _layer_inputs(c, seed):
    """An attention or decoder layer's weights (out x in) and biases."""
    r = _Rand(seed)
    D = c["heads"] * c["hd"]
    t = {n: r.xavier(D, D) for n in ("wq", "wk", "wv", "wo")}
    t.update({n: r.normal(D, std=0.1) for n in ("bq", "bk", "bv", "bo")})
    if c["kind"] == "decode":
        FF = c["ff"]
        t.update(w1=r.xavier(FF, D), b1=r.normal(FF, std=0.1), w2=r.xavier(D, FF), b2=r.normal(D, std=0.1),
                 g1=1 + r.normal(D, std=0.1), h1=r.normal(D, std=0.1), g2=1 + r.normal(D, std=0.1),
                 h2=r.normal(D, std=0.1))
        t["x"] = r.normal(c["batch"], D)
        t["kc"], t["vc"] = (r.normal(c["batch"], c["keys"], D) for _ in range(2))
    else:
        t["x"] = r.normal(c["batch"] * c["len"], D)
        if c["kind"] == "attn_bwd":
            t["dy"] = r.normal(c["batch"] * c["len"], D, std=0.1)
    return t


def _ffn_inputs(c, seed):
    r = _Rand(seed)
    R, D, FF = c["rows"], c["dim"], c["ff"]
    t = {"x": r.normal(R, D), "w1": r.xavier(FF, D), "b1": r.normal(FF, std=0.1), "w2": r.xavier(D, FF),
         "b2": r.normal(D, std=0.1), "g": 1 + r.normal(D, std=0.1), "h": r.normal(D, std=0.1)}
    if c["kind"] == "ffn_train":
        t["dy"] = r.normal(R, D, std=0.1)
    return t


def _size(name, *args):
    """The answer of one of the library's workspace-size entries."""
    n = ctypes.c_size_t(0)
    native.check(getattr(native.lib(), name)(*args, ctypes.byref(n)))
    return n.value


def _workspace(nbytes):
    return torch.empty(max(256, nbytes), device=DEV, dtype=torch.uint8)


def _call(name, *args):
    """One entry of the C ABI on torch's current stream; tensors pass as pointers."""
    a = [t.data_ptr() if isinstance(t, torch.Tensor) else t for t in args]
    native.check(getattr(native.lib(), name)(*a, torch.cuda.current_stream().cuda_stream))


def prepare(case, seed):
    c, k = case, case["kind"]
    native.init(0)
    if k in ("lm", "lm_train", "series"):
        lm, _ = host.language_model(_config(c), _weights(c, seed))
        if k == "lm_train":
            trainer = host.module().DeviceTrainer(lm, host.module().TrainingConfig(), c["batch"], c["len"] - 1)
            return {"case": c, "trainer": trainer, "batch": [s for s in _tokens(c, seed)]}
        engine = host.module().DeviceLanguageModel(lm, c["batch"])
        return {"case": c, "engine": engine, "x": _windows(c, seed) if k == "series" else _tokens(c, seed)}
    s = {"case": c}
    if k in ("attn", "attn_bwd"):
        B, L, H, hd = c["batch"], c["len"], c["heads"], c["hd"]
        D, R = H * hd, B * L
        s.update(_layer_inputs(c, seed))
        s["cs"] = _empty(L, hd)
        _call("cdml_rope_table", s["cs"], L, hd, 10000.0)
        if k == "attn":
            s["mask"] = _mask(c)
            s["ws"] = _workspace(_size("cdml_mha_layer_fwd_workspace_size", B, L, D, H))
            s["y"] = _empty(R, D)
            return s
        # the forward pass of the training step, whose tensors the backward reads
        for n in ("q", "k", "v", "o", "dcat", "dq", "dk", "dv", "dx"):
            s[n] = _empty(R, D)
        s["lse"] = _empty(B * H, L)
        _call("cdml_project_qkv_rope", s["x"], s["wq"], s["bq"], s["wk"], s["bk"], s["wv"], s["bv"], s["q"], s["k"],
              s["v"], R, D, D, hd, s["cs"], L, 0, L)
        _call("cdml_sdpa_fwd_lse", s["q"], D, s["k"], D, s["v"], D, s["o"], D, s["lse"], B, L, L, D, H, _scale(hd), 1,
              None)
        s["grads"] = _empty(4 * D * D + 4 * D)
        s["ws"] = _workspace(max(_size("cdml_sdpa_bwd_saved_workspace_size", B, L, L, D, H, 1),
                                 _size("cdml_linear_backward_workspace_size", R, D, D),
                                 _size("cdml_backprop_qkv_workspace_size", R, D, D)))
        return s
    if k in ("ffn", "ffn_train"):
        R, D, FF = c["rows"], c["dim"], c["ff"]
        s.update(_ffn_inputs(c, seed))
        s["a"], s["f"], s["y"] = _empty(R, FF), _empty(R, D), _empty(R, D)
        if k == "ffn_train":
            # ReLU layers keep their output alone, the others their pre-activation too
            s["z"] = None if c["act"] in ("relu", "leakyrelu") else _empty(R, FF)
            s["res"], s["mean"], s["var"] = _empty(R, D), _empty(R), _empty(R)
            s["dr"], s["da"], s["dx"] = _empty(R, D), _empty(R, FF), _empty(R, D)
            s["grads"] = _empty(2 * D * FF + FF + 3 * D)
            s["ws"] = _workspace(max(_size("cdml_linear_backward_workspace_size", R, FF, D),
                                     _size("cdml_linear_backward_workspace_size", R, D, FF),
                                     _size("cdml_layernorm_backward_workspace_size", R, D)))
        return s
    B, T, H, hd = c["batch"], c["keys"], c["heads"], c["hd"]
    D = H * hd
    lens = torch.tensor(_kv_lens(c), dtype=torch.int32, device=DEV)
    s["lens"] = lens
    s["ws"] = _workspace(_size("cdml_decode_attn_workspace_size", B, T, D, H))
    if k == "decode_attn":
        r = _Rand(seed)
        s["q"], s["kc"], s["vc"], s["o"] = r.normal(B, D), r.normal(B, T, D), r.normal(B, T, D), _empty(B, D)
        return s
    s.update(_layer_inputs(c, seed))
    s["pos"] = (lens - 1).contiguous()  # the new token's position: its key is the last attended one
    for n in ("q", "k", "v", "o", "p", "n1", "f", "y"):
        s[n] = _empty(B, D)
    s["a"] = _empty(B, c["ff"])
    return s


def _scale(hd):
    return float(np.float32(1.0) / np.sqrt(np.float32(hd)))


# ---- one pass -------------------------------------------------------------

def run(s):
    return _RUN[s["case"]["kind"]](s)


def _run_lm(s):
    logits = s["engine"].Forward(s["x"])
    return {"logits": logits, "tokens": s["engine"].GenerateGreedy(s["x"], s["case"]["new"])}


def _run_lm_train(s):
    # learning rate 0, the first step of a warm-up: every pass sees the same weights
    loss = s["trainer"].TrainBatch(s["batch"], 0.0)
    return {"loss": loss, "gradients": s["trainer"].gradients()}


def _run_series(s):
    return s["engine"].ForwardContinuous(s["x"], s["case"]["batch"], s["case"]["len"])


def _run_attn(s):
    c = s["case"]
    D = c["heads"] * c["hd"]
    _call("cdml_mha_layer_fwd", s["x"], s["wq"], s["bq"], s["wk"], s["bk"], s["wv"], s["bv"], s["wo"], s["bo"], s["y"],
          c["batch"], c["len"], D, c["heads"], 10000.0, 1 if c["mask"] == "causal" else 0, s["mask"], s["cs"], s["ws"],
          s["ws"].numel())
    return s["y"]


def _run_attn_bwd(s):
    c = s["case"]
    B, L, H, hd = c["batch"], c["len"], c["heads"], c["hd"]
    D, R = H * hd, B * L
    g = s["grads"]
    gw = [g[i * D * D:(i + 1) * D * D] for i in range(4)]            # wq, wk, wv, wo
    gb = [g[4 * D * D + i * D:4 * D * D + (i + 1) * D] for i in range(4)]
    ws, n = s["ws"], s["ws"].numel()
    _call("cdml_zero_f32_async", g, g.numel())
    _call("cdml_linear_backward", s["o"], D, s["dy"], D, s["wo"], s["dcat"], D, gw[3], gb[3], R, D, D, 0, ws, n)
    _call("cdml_sdpa_bwd_saved_rope", s["q"], D, s["k"], D, s["v"], D, s["o"], D, s["lse"], s["dcat"], D, s["dq"], D,
          s["dk"], D, s["dv"], D, B, L, L, D, H, _scale(hd), 1, None, s["cs"], L, ws, n)
    _call("cdml_backprop_qkv", s["x"], s["dq"], s["dk"], s["dv"], s["wq"], s["wk"], s["wv"], gw[0], gb[0], gw[1], gb[1],
          gw[2], gb[2], s["dx"], R, D, D, ws, n)
    return {"dx": s["dx"], "gw": gw, "gb": gb}


def _run_ffn(s):
    c = s["case"]
    R, D, FF = c["rows"], c["dim"], c["ff"]
    _call("cdml_linear", s["x"], D, s["w1"], s["b1"], s["a"], FF, R, D, FF, native.ACT[c["act"]])
    _call("cdml_linear", s["a"], FF, s["w2"], s["b2"], s["f"], D, R, FF, D, native.ACT["none"])
    _call("cdml_residual_layernorm", s["x"], s["f"], s["g"], s["h"], s["y"], R, D, EPS)
    return s["y"]


def _run_ffn_train(s):
    c = s["case"]
    R, D, FF, act = c["rows"], c["dim"], c["ff"], native.ACT[c["act"]]
    g, n = s["grads"], D * FF
    gw1, gw2, gb1 = g[:n], g[n:2 * n], g[2 * n:2 * n + FF]
    gb2, gg, gh = (g[2 * n + FF + i * D:2 * n + FF + (i + 1) * D] for i in range(3))
    ws, nb = s["ws"], s["ws"].numel()
    _call("cdml_zero_f32_async", g, g.numel())
    _call("cdml_linear_preact", s["x"], D, s["w1"], s["b1"], s["z"], s["a"], FF, R, D, FF, act)
    _call("cdml_linear", s["a"], FF, s["w2"], s["b2"], s["f"], D, R, FF, D, native.ACT["none"])
    _call("cdml_residual_layernorm_fwd", s["x"], s["f"], s["g"], s["h"], s["y"], s["mean"], s["var"], s["res"], None,
          R, D, EPS)
    _call("cdml_layernorm_backward", s["dy"], None, None, s["g"], s["res"], s["mean"], s["var"], s["dr"], gg, gh, R, D,
          EPS, 1, ws, nb)
    dz, dact = (s["a"], act | 0x100) if s["z"] is None else (s["z"], act)
    _call("cdml_linear_backward_act", s["a"], FF, s["dr"], D, s["w2"], dz, dact, None, s["da"], FF, gw2, gb2, R, FF, D,
          ws, nb)
    _call("cdml_linear_backward_act", s["x"], D, s["da"], FF, s["w1"], None, 0, s["dr"], s["dx"], D, gw1, gb1, R, D, FF,
          ws, nb)
    return {"y": s["y"], "dx": s["dx"], "gw1": gw1, "gw2": gw2, "gb1": gb1, "gb2": gb2, "gg": gg, "gh": gh}


def _run_decode_attn(s):
    c = s["case"]
    _call("cdml_decode_attn", s["q"], s["kc"], s["vc"], s["lens"], s["o"], c["batch"], c["keys"], c["heads"] * c["hd"],
          c["heads"], _scale(c["hd"]), s["ws"], s["ws"].numel())
    return s["o"]


def _run_decode(s):
    c = s["case"]
    B, T, H, hd, FF = c["batch"], c["keys"], c["heads"], c["hd"], c["ff"]
    D = H * hd
    _call("cdml_project_qkv", s["x"], s["wq"], s["bq"], s["wk"], s["bk"], s["wv"], s["bv"], s["q"], s["k"], s["v"], B,
          D, D)
    for t in (s["q"], s["k"]):
        _call("cdml_rope", t, B, D, 0, hd, H, 10000.0, 0, 0, 0, s["pos"])
    _call("cdml_kv_cache_append", s["k"], s["v"], s["kc"], s["vc"], s["pos"], B, T, D)
    _call("cdml_decode_attn", s["q"], s["kc"], s["vc"], s["lens"], s["o"], B, T, D, H, _scale(hd), s["ws"],
          s["ws"].numel())
    _call("cdml_linear", s["o"], D, s["wo"], s["bo"], s["p"], D, B, D, D, 0)
    _call("cdml_residual_layernorm", s["x"], s["p"], s["g1"], s["h1"], s["n1"], B, D, EPS)
    _call("cdml_linear", s["n1"], D, s["w1"], s["b1"], s["a"], FF, B, D, FF, native.ACT["relu"])
    _call("cdml_linear", s["a"], FF, s["w2"], s["b2"], s["f"], D, B, FF, D, 0)
    _call("cdml_residual_layernorm", s["n1"], s["f"], s["g2"], s["h2"], s["y"], B, D, EPS)
    return {"y": s["y"], "kc": s["kc"], "vc": s["vc"]}


_RUN = {"lm": _run_lm, "lm_train": _run_lm_train, "series": _run_series, "attn": _run_attn, "attn_bwd": _run_attn_bwd,
        "ffn": _run_ffn, "ffn_train": _run_ffn_train, "decode_attn": _run_decode_attn, "decode": _run_decode}


# ---- the same in float64 --------------------------------------------------

def _d(t):
    return torch.as_tensor(t, device=DEV).double()


def _angles(pos, hd):
    """cos and sin [len(pos), hd / 2] of the rotary embedding, base 10000."""
    p = torch.arange(hd // 2, device=DEV, dtype=torch.float64)
    th = pos.double()[:, None] / (10000.0 ** (2.0 * p / hd))[None, :]
    return th.cos(), th.sin()


def _rotate(x, cos, sin):
    """Pairs (2p, 2p + 1) of x [..., rows, heads, hd] rotated by the angles of its rows."""
    a, b = x[..., 0::2], x[..., 1::2]
    cos, sin = cos[:, None, :], sin[:, None, :]
    return torch.stack((a * cos - b * sin, a * sin + b * cos), -1).flatten(-2)


def _attention(x, w, B, L, H, hide):
    """Multi-head self-attention with rotary embedding of x [B * L, D]; hide: bool [L, L], keys not seen."""
    D = x.shape[1]
    hd = D // H
    cos, sin = _angles(torch.arange(L, device=DEV), hd)
    q, k, v = ((x @ w["w" + n].T + w["b" + n]).reshape(B, L, H, hd) for n in "qkv")
    q, k = (_rotate(t, cos, sin).transpose(1, 2) for t in (q, k))
    sc = (q @ k.transpose(2, 3)) * hd ** -0.5
    if hide is not None:
        sc = sc.masked_fill(hide, -math.inf)
    o = (sc.softmax(-1) @ v.transpose(1, 2)).transpose(1, 2).reshape(B * L, D)
    return o @ w["wo"].T + w["bo"]


def _norm(x, g, b):
    return torch.nn.functional.layer_norm(x, (x.shape[1],), g, b, EPS)


def _act(z, name):
    if name == "leakyrelu":
        return torch.where(z > 0, z, 0.01 * z)
    if name == "swish":
        return z * torch.sigmoid(z)
    return {"relu": torch.relu, "tanh": torch.tanh, "sigmoid": torch.sigmoid}[name](z)


def _act_deriv(z, name):
    """The reference's derivatives: leaky ReLU takes 0.1 on its negative side."""
    if name == "relu":
        return (z >= 0).double()
    if name == "leakyrelu":
        return torch.where(z <= 0, 0.1, 1.0).double()
    s = torch.sigmoid(z)
    return {"swish": s + z * s * (1 - s), "tanh": 1 - torch.tanh(z) ** 2, "sigmoid": s * (1 - s)}[name]


def _future(L):
    return torch.ones((L, L), device=DEV, dtype=torch.bool).triu(1)


def _blocks(x, layers, B, L, H, act="relu"):
    """Post-LayerNorm decoder blocks."""
    for w in layers:
        n1 = _norm(x + _attention(x, w, B, L, H, _future(L)), w["ln1_g"], w["ln1_b"])
        f = _act(n1 @ w["ffn_w1"].T + w["ffn_b1"], act) @ w["ffn_w2"].T + w["ffn_b2"]
        x = _norm(n1 + f, w["ln2_g"], w["ln2_b"])
    return x


def _chunks(B, L, H):
    """Sequences whose scores take about 2 GB in float64."""
    return max(1, min(B, int(2.5e8 / (H * L * L))))


def exact(case, seed):
    c, k = case, case["kind"]
    if k in ("lm", "lm_train", "series"):
        w = _weights(c, seed)
        w = {n: ([{m: _d(t) for m, t in y.items()} for y in v] if n == "layers" else _d(v)) for n, v in w.items()}
        return {"lm": _exact_lm, "lm_train": _exact_lm_train, "series": _exact_series}[k](c, w, seed)
    if k == "attn":
        B, L, H = c["batch"], c["len"], c["heads"]
        t = {n: _d(v) for n, v in _layer_inputs(c, seed).items()}
        mask = _mask(c)
        hide = _future(L) if c["mask"] == "causal" else None if mask is None else mask == 0
        n = _chunks(B, L, H)
        return torch.cat([_attention(t["x"][i * L:(i + n) * L], t, min(n, B - i), L, H, hide) for i in range(0, B, n)])
    if k == "attn_bwd":
        B, L, H = c["batch"], c["len"], c["heads"]
        t = {n: _d(v) for n, v in _layer_inputs(c, seed).items()}
        names = [p + m for p in "wb" for m in "qkvo"]
        for m in names:
            t[m].requires_grad_()
        n, dx = _chunks(B, L, H), []
        for i in range(0, B, n):
            x = t["x"][i * L:(i + n) * L].clone().requires_grad_()
            (_attention(x, t, min(n, B - i), L, H, _future(L)) * t["dy"][i * L:(i + n) * L]).sum().backward()
            dx.append(x.grad)
        g = [t[m].grad for m in names]
        return {"dx": torch.cat(dx), "gw": [v.reshape(-1) for v in g[:4]], "gb": g[4:]}
    if k in ("ffn", "ffn_train"):
        return _exact_ffn(c, {n: _d(v) for n, v in _ffn_inputs(c, seed).items()})
    return _exact_decode(c, seed)


def _exact_lm(c, w, seed):
    B, L = c["batch"], c["len"]
    ids = torch.as_tensor(_tokens(c, seed), device=DEV).long()

    def logits(t):
        n = t.shape[1]
        h = _blocks(w["token_embedding"][t.reshape(-1)], w["layers"], B, n, c["heads"], c["act"])
        return h @ w["out_proj"].T + w["out_bias"]

    # the tokens are whole numbers that follow from comparisons: no value of their own in 64 bits
    return {"logits": logits(ids), "tokens": None}


def _exact_lm_train(c, w, seed):
    B, L = c["batch"], c["len"] - 1
    ids = torch.as_tensor(_tokens(c, seed), device=DEV).long()
    leaves = [(n, v) for n, v in w.items() if n != "layers"]
    leaves += [("layers.%d.%s" % (i, n), v) for i, y in enumerate(w["layers"]) for n, v in y.items()]
    for _, v in leaves:
        v.requires_grad_()
    h = _blocks(w["token_embedding"][ids[:, :L].reshape(-1)], w["layers"], B, L, c["heads"], c["act"])
    loss = torch.nn.functional.cross_entropy(h @ w["out_proj"].T + w["out_bias"], ids[:, 1:].reshape(-1))
    loss.backward()
    norm = math.sqrt(sum(float(v.grad.square().sum()) for _, v in leaves))
    return {"loss": float(loss.detach()), "gradients": {n: v.grad * min(1.0, 1.0 / norm) for n, v in leaves}}


def _exact_series(c, w, seed):
    B, L, H = c["batch"], c["len"], c["heads"]
    x = _d(_windows(c, seed)) @ w["input_proj"].T + w["input_bias"]
    n = _chunks(B, L, H)
    h = torch.cat([_blocks(x[i * L:(i + n) * L], w["layers"], min(n, B - i), L, H) for i in range(0, B, n)])
    return h @ w["out_proj"].T + w["out_bias"]


def _exact_ffn(c, t):
    z = t["x"] @ t["w1"].T + t["b1"]
    a = _act(z, c["act"])
    r = t["x"] + a @ t["w2"].T + t["b2"]
    if c["kind"] == "ffn":
        return _norm(r, t["g"], t["h"])
    mean, var = r.mean(1, keepdim=True), r.var(1, unbiased=False, keepdim=True)
    rs = (var + EPS).rsqrt()
    xn = (r - mean) * rs
    dn = t["dy"] * t["g"]
    dr = rs * (dn - dn.mean(1, keepdim=True) - xn * (dn * xn).mean(1, keepdim=True))
    da = (dr @ t["w2"]) * _act_deriv(z, c["act"])
    kinked = c["act"] in KINKED  # no value in 64 bits: see tolerance()
    return {"y": xn * t["g"] + t["h"], "dx": None if kinked else da @ t["w1"] + dr,
            "gw1": None if kinked else (da.T @ t["x"]).reshape(-1), "gb1": None if kinked else da.sum(0),
            "gw2": (dr.T @ a).reshape(-1), "gb2": dr.sum(0), "gg": (t["dy"] * xn).sum(0),
            "gh": t["dy"].sum(0)}


def _exact_decode(c, seed):
    B, T, H, hd = c["batch"], c["keys"], c["heads"], c["hd"]
    D, lens = H * hd, _kv_lens(c)

    def attend(q, kc, vc):
        out = []
        for b, n in enumerate(lens):  # one sequence at a time: the whole cache in 64 bits is large
            kk, vv = (t[b, :n].double().reshape(n, H, hd).transpose(0, 1) for t in (kc, vc))
            p = ((kk @ q[b].reshape(H, hd, 1)).squeeze(2) * hd ** -0.5).softmax(-1)
            out.append((p[:, None, :] @ vv).reshape(D))
        return torch.stack(out)

    if c["kind"] == "decode_attn":
        r = _Rand(seed)
        q, kc = r.normal(B, D), r.normal(B, T, D)
        return attend(q.double(), kc, r.normal(B, T, D))
    t = _layer_inputs(c, seed)
    kc, vc = (t.pop(n).double() for n in ("kc", "vc"))
    t = {n: _d(v) for n, v in t.items()}
    q, kn, vn = (t["x"] @ t["w" + n].T + t["b" + n] for n in "qkv")
    pos = torch.tensor(lens, device=DEV) - 1
    cos, sin = _angles(pos, hd)
    q, kn = (_rotate(y.reshape(B, H, hd), cos, sin).reshape(B, D) for y in (q, kn))
    at = torch.arange(B, device=DEV)
    kc[at, pos], vc[at, pos] = kn, vn
    n1 = _norm(t["x"] + attend(q, kc, vc) @ t["wo"].T + t["bo"], t["g1"], t["h1"])
    f = torch.relu(n1 @ t["w1"].T + t["b1"]) @ t["w2"].T + t["b2"]
    return {"y": _norm(n1 + f, t["g2"], t["h2"]), "kc": kc, "vc": vc}
