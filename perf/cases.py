"""The work whose speed is measured: the layers and the training step that a
program built on this library runs, each through the C entry points of
include/mle_hip.h as the engine's own nodes call them.

A case is a dict of plain values; `kind` names the layer and the rest are its
sizes and options:

  mlp_step     a whole training step of the two-layer classifier: forward,
               loss with its read-back, backward, AdamW
  linear       one Linear layer: forward with bias, then dX, dW and db
  ffn          Linear -> activation -> Linear, forward and backward
  attention    the fused column-softmax attention, forward and backward
  lm_head      the output projection with its cross-entropy, forward and
               backward
  norm_add     the residual Add and the LayerNorm that reads it, forward and
               backward
  group_act    GroupNorm -> activation, forward and backward
  conv         one convolution: forward with bias, dX, dW and db
  adamw        global-norm clip and AdamW over one flat arena

Everything is float32 (token ids int32), the library's only data type.
Gradients are assigned, as in a step after zero_grad.
"""
from __future__ import annotations

import ctypes
import math
import random

import torch
import torch.nn.functional as F

from ml_engine_amd import hip

DEV = "cuda"
HEAD_DIM = 64    # the fused attention's head width
EPS = 1e-5       # the normalisations' epsilon
ADAM = dict(lr=1e-3, b1=0.9, b2=0.999, eps=1e-8, wd=0.01)
MAX_FLOPS = 2.06e11  # of a drawn case: the largest listed one's
MAX_BYTES = 3.2e9

# --------------------------------------------------------------------- cases


def listed() -> list[dict]:
    return [
        # The classifier's whole step at its benchmark size: a handful of
        # launches, bound by latency.
        dict(name="mlp_step", kind="mlp_step", batch=64, inp=784, hidden=256, classes=10),
        # A Linear of a small model on a short batch, no size a multiple of a tile.
        dict(name="linear_ragged", kind="linear", rows=1000, inp=330, out=516),
        # The benchmark's Linear backward size, with its forward: the largest products.
        dict(name="linear_wide", kind="linear", rows=8192, inp=1024, out=4096),
        # The transformer block's feed-forward (32 x 256 tokens).
        dict(name="ffn_block", kind="ffn", rows=8192, d=512, ffn=2048, act="gelu"),
        # The transformer block's attention.
        dict(name="attention_block", kind="attention", batch=32, heads=8, seq=256, causal=1),
        # Longer sequences, encoder (unmasked) attention.
        dict(name="attention_long", kind="attention", batch=4, heads=8, seq=1024, causal=0),
        # The transformer block's vocabulary projection and loss.
        dict(name="lm_head", kind="lm_head", rows=8192, d=512, vocab=8000),
        # The pre-norm residual stream of the transformer block.
        dict(name="norm_add", kind="norm_add", batch=32, rows=256, cols=512),
        # GroupNorm -> SiLU of the U-Net residual block.
        dict(name="group_act", kind="group_act", batch=16, channels=128, h=64, w=64, groups=32, act="silu"),
        # The residual block's second 3 x 3 convolution.
        dict(name="conv_block", kind="conv", n=16, cin=128, cout=128, h=64, w=64, k=3, stride=1),
        # A deeper U-Net level of 28 x 28 images (14 x 14 maps, whose rows are
        # no multiple of 16 bytes).
        dict(name="conv_deep", kind="conv", n=32, cin=128, cout=192, h=14, w=14, k=3, stride=1),
        # The optimizer benchmark's parameter arena.
        dict(name="adamw", kind="adamw", n=100_000_000),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng: random.Random, lo: int, hi: int) -> int:
    """A layer width: mostly a multiple of 16, sometimes of 4, sometimes any."""
    w = _log_int(rng, lo, hi)
    m = rng.choice((16, 16, 4, 1))
    return max(m, w // m * m)


def _draw_once(rng: random.Random) -> dict:
    kind = rng.choice(("mlp_step", "linear", "linear", "ffn", "attention", "lm_head", "norm_add", "group_act", "conv",
                       "conv", "adamw"))
    if kind == "mlp_step":
        return dict(kind=kind, batch=_log_int(rng, 8, 512), inp=_width(rng, 64, 1024), hidden=_width(rng, 32, 1024),
                    classes=rng.randint(2, 64))
    if kind == "linear":
        return dict(kind=kind, rows=_log_int(rng, 64, 16384), inp=_width(rng, 48, 4096), out=_width(rng, 48, 4096))
    if kind == "ffn":
        d = _width(rng, 64, 1024)
        return dict(kind=kind, rows=_log_int(rng, 64, 16384), d=d, ffn=rng.choice((2, 3, 4)) * d,
                    act=rng.choice(("gelu", "silu")))
    if kind == "attention":
        return dict(kind=kind, batch=_log_int(rng, 1, 32), heads=rng.randint(1, 16), seq=64 * _log_int(rng, 1, 16),
                    causal=rng.randint(0, 1))
    if kind == "lm_head":
        return dict(kind=kind, rows=_log_int(rng, 128, 8192), d=_width(rng, 64, 1024), vocab=_width(rng, 256, 16000))
    if kind == "norm_add":
        return dict(kind=kind, batch=_log_int(rng, 1, 64), rows=_log_int(rng, 16, 512), cols=_width(rng, 64, 1024))
    if kind == "group_act":
        groups = rng.choice((4, 8, 16, 32))
        return dict(kind=kind, batch=_log_int(rng, 1, 32), channels=groups * _log_int(rng, 1, 8),
                    h=_log_int(rng, 7, 64), w=_log_int(rng, 7, 64), groups=groups,
                    act=rng.choice(("silu", "relu", "gelu")))
    if kind == "conv":
        side = rng.choice((7, 8, 14, 16, 28, 32, 56, 64))
        return dict(kind=kind, n=_log_int(rng, 1, 32), cin=_width(rng, 3, 256), cout=_width(rng, 16, 256), h=side,
                    w=side, k=rng.choice((3, 3, 3, 1)), stride=rng.choice((1, 1, 1, 2)))
    return dict(kind="adamw", n=_log_int(rng, 10_000, 100_000_000))


def draw(rng: random.Random) -> dict:
    while True:
        case = _draw_once(rng)
        w = work(case)
        if w["flops"] <= MAX_FLOPS and w["bytes"] <= MAX_BYTES:
            return case


# ------------------------------------------------------------------ plumbing


def _gen(seed: int) -> torch.Generator:
    hip.init(0)
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _normal(g, *shape, scale=1.0):
    return torch.randn(*shape, generator=g, device=DEV).mul_(scale)


def _uniform(g, *shape, bound=1.0):
    return torch.rand(*shape, generator=g, device=DEV).mul_(2 * bound).sub_(bound)


def _ids(g, n, hi):
    return torch.randint(0, hi, (n,), generator=g, device=DEV, dtype=torch.int64).to(torch.int32)


def _new(*shape):
    return torch.empty(*shape, device=DEV)


class _Ws:
    """A workspace of a queried size: None where none is needed."""

    def __init__(self, nbytes: int):
        self.nbytes = int(nbytes)
        self.buf = torch.empty(max(self.nbytes, 1), dtype=torch.uint8, device=DEV) if self.nbytes else None
        self.ptr = self.buf.data_ptr() if self.nbytes else None


def _p(t):
    return t.data_ptr()


def _linear_w(g, inp, out):
    """Weights and bias at the scale a trained layer has: outputs of order one."""
    return _uniform(g, inp, out, bound=math.sqrt(3.0 / inp)), _uniform(g, out, bound=0.1)


def _conv_out(c):
    pad = c["k"] // 2
    return pad, (c["h"] + 2 * pad - c["k"]) // c["stride"] + 1, (c["w"] + 2 * pad - c["k"]) // c["stride"] + 1


# ------------------------------------------------------------------- prepare


def prepare(case: dict, seed: int) -> dict:
    g = _gen(seed)
    s = _PREPARE[case["kind"]](case, g)
    s["case"] = case
    return s


def _prep_mlp(c, g):
    L = hip.lib()
    n, i, h, k = c["batch"], c["inp"], c["hidden"], c["classes"]
    # pixels in [0, 1), a model in the middle of its training: the moments are
    # those of gradients seen before
    w1, b1 = _linear_w(g, i, h)
    w2, b2 = _linear_w(g, h, k)
    sizes = [i * h, h, h * k, k]
    flat = torch.cat([t.reshape(-1) for t in (w1, b1, w2, b2)])
    m = _normal(g, flat.numel(), scale=1e-3)
    v = m.square() + 1e-7
    grad = torch.zeros_like(flat)
    off = [0]
    for z in sizes:
        off.append(off[-1] + z)
    part = lambda t: [t[a:b] for a, b in zip(off, off[1:])]  # noqa: E731
    return dict(x=torch.rand(n, i, generator=g, device=DEV), keys=_ids(g, n, k), p=flat, g=grad, m=m, v=v,
                pp=part(flat), gp=part(grad), t=1000, h=_new(n, h), a=_new(n, h), logits=_new(n, k),
                stats=_new(n, 2), loss=_new(1), dlogits=_new(n, k), da=_new(n, h), dh=_new(n, h), dx=_new(n, i),
                ws1=_Ws(L.mle_gemm_ws_bytes(n, h, i, 1)), ws2=_Ws(L.mle_linear_bwd_ws_bytes(n, h, k, 1)),
                ws3=_Ws(L.mle_linear_bwd_ws_bytes(n, i, h, 1)))


def _prep_linear(c, g):
    L = hip.lib()
    r, i, o = c["rows"], c["inp"], c["out"]
    w, b = _linear_w(g, i, o)
    return dict(x=_normal(g, r, i), w=w, b=b, dy=_normal(g, r, o, scale=1e-3), y=_new(r, o), dx=_new(r, i),
                dw=_new(i, o), db=_new(o), wsf=_Ws(L.mle_gemm_ws_bytes(r, o, i, 1)),
                wsb=_Ws(L.mle_linear_bwd_ws_bytes(r, i, o, 1)))


def _prep_ffn(c, g):
    L = hip.lib()
    r, d, f = c["rows"], c["d"], c["ffn"]
    w1, b1 = _linear_w(g, d, f)
    w2, b2 = _linear_w(g, f, d)
    return dict(x=_normal(g, r, d), w1=w1, b1=b1, w2=w2, b2=b2, dy=_normal(g, r, d, scale=1e-3), h=_new(r, f),
                a=_new(r, f), y=_new(r, d), da=_new(r, f), dh=_new(r, f), dx=_new(r, d), dw1=_new(d, f), db1=_new(f),
                dw2=_new(f, d), db2=_new(d), ws1=_Ws(L.mle_gemm_ws_bytes(r, f, d, 1)),
                ws2=_Ws(L.mle_gemm_ws_bytes(r, d, f, 1)), wsb2=_Ws(L.mle_linear_bwd_ws_bytes(r, f, d, 1)),
                wsb1=_Ws(L.mle_linear_bwd_ws_bytes(r, d, f, 1)))


def _prep_attention(c, g):
    shape = (c["batch"], c["seq"], c["heads"] * HEAD_DIM)
    s = {k: _normal(g, *shape) for k in ("q", "k", "v")}
    s["do"] = _normal(g, *shape, scale=1e-3)
    s.update({k: _new(*shape) for k in ("out", "dq", "dk", "dv")})
    s["ws"] = _Ws(hip.lib().mle_attention_ws_bytes(c["batch"], c["heads"], c["seq"]))
    return s


def _prep_lm_head(c, g):
    L = hip.lib()
    r, d, v = c["rows"], c["d"], c["vocab"]
    w, b = _linear_w(g, d, v)
    ldp = 2 * ((v + 63) // 64)
    return dict(x=_normal(g, r, d), w=w, b=b, keys=_ids(g, r, v), logits=_new(r, v), part=_new(r, ldp),
                stats=_new(r, 2), loss=_new(1), dlogits=_new(r, v), dx=_new(r, d), dw=_new(d, v), db=_new(v),
                wsf=_Ws(L.mle_gemm_ws_bytes(r, v, d, 1)), wsl=_Ws(L.mle_loss_ws_bytes(r * v)),
                wsb=_Ws(L.mle_linear_bwd_ws_bytes(r, d, v, 1)))


def _prep_norm_add(c, g):
    shape = (c["batch"], c["rows"], c["cols"])
    s = dict(a=_normal(g, *shape), b=_normal(g, *shape, scale=0.5), dy=_normal(g, *shape, scale=1e-3),
             dres=_normal(g, *shape, scale=1e-3))
    s.update({k: _new(*shape) for k in ("r", "y", "dr", "da", "db")})
    s["stats"] = _new(c["batch"], 2)
    s["ws"] = _Ws(hip.lib().mle_norm_ws_bytes(c["batch"], 1, c["rows"] * c["cols"], 1))
    return s


def _prep_group_act(c, g):
    shape = (c["batch"], c["channels"], c["h"], c["w"])
    s = dict(x=_normal(g, *shape), da=_normal(g, *shape, scale=1e-3))
    s.update({k: _new(*shape) for k in ("y", "a", "dy", "dx")})
    s["stats"] = _new(c["batch"] * c["groups"], 2)
    s["ws"] = _Ws(hip.lib().mle_norm_ws_bytes(c["batch"], c["channels"], c["h"] * c["w"], c["groups"]))
    return s


def _prep_conv(c, g):
    n, ci, co, k = c["n"], c["cin"], c["cout"], c["k"]
    pad, oh, ow = _conv_out(c)
    return dict(x=_normal(g, n, ci, c["h"], c["w"]), w=_uniform(g, co, ci, k, k, bound=math.sqrt(3.0 / (ci * k * k))),
                b=_uniform(g, co, bound=0.1), dy=_normal(g, n, co, oh, ow, scale=1e-3), y=_new(n, co, oh, ow),
                dx=_new(n, ci, c["h"], c["w"]), dw=_new(co, ci, k, k), db=_new(co),
                ws=_Ws(hip.lib().mle_conv2d_wgrad_ws_bytes(n, ci, c["h"], c["w"], co, k, k, pad, c["stride"])))


def _prep_adamw(c, g):
    n = c["n"]
    m = _normal(g, n, scale=1e-4)
    return dict(p=_normal(g, n, scale=0.02), g=_normal(g, n, scale=1e-3), m=m, v=m.square() + 1e-8, t=1000,
                norm=torch.zeros(1, dtype=torch.float64, device=DEV), ws=_Ws(hip.lib().mle_adamw_clip_ws_bytes(n)))


_PREPARE = dict(mlp_step=_prep_mlp, linear=_prep_linear, ffn=_prep_ffn, attention=_prep_attention,
                lm_head=_prep_lm_head, norm_add=_prep_norm_add, group_act=_prep_group_act, conv=_prep_conv,
                adamw=_prep_adamw)

# ----------------------------------------------------------------------- run


def run(state: dict):
    return _RUN[state["case"]["kind"]](state, state["case"])


def _run_mlp(s, c):
    call = hip.call
    n, i, h, k = c["batch"], c["inp"], c["hidden"], c["classes"]
    w1, b1, w2, b2 = s["pp"]
    dw1, db1, dw2, db2 = s["gp"]
    relu = hip.ACT["relu"]
    loss = ctypes.c_float()
    call("mle_gemm_act_fwd", None, 0, 0, n, h, i, 1.0, _p(s["x"]), i, _p(w1), h, 0.0, _p(s["h"]), _p(b1), relu,
         _p(s["a"]), s["ws1"].ptr, s["ws1"].nbytes)
    call("mle_linear_xent_keys_small_read", None, n, h, k, _p(s["a"]), _p(w2), _p(b2), _p(s["logits"]), _p(s["keys"]),
         n, n, _p(s["stats"]), n, _p(s["loss"]), _p(s["dlogits"]), ctypes.addressof(loss))
    call("mle_linear_bwd_act", None, n, h, k, _p(s["a"]), _p(s["dlogits"]), _p(w2), _p(s["da"]), 0, _p(dw2), _p(db2), 0,
         relu, _p(s["h"]), _p(s["dh"]), 0, s["ws2"].ptr, s["ws2"].nbytes)
    call("mle_linear_bwd_ex", None, n, i, h, 1, _p(s["x"]), _p(s["dh"]), 0, _p(w1), 0, _p(s["dx"]), 0, _p(dw1), _p(db1),
         0, 0, s["ws3"].ptr, s["ws3"].nbytes)
    call("mle_adam_update", None, _p(s["p"]), _p(s["g"]), _p(s["m"]), _p(s["v"]), s["p"].numel(), s["t"], ADAM["lr"],
         ADAM["b1"], ADAM["b2"], ADAM["eps"], ADAM["wd"], 1, None)
    s["t"] += 1
    return dict(loss=float(loss.value), logits=s["logits"], grads=s["g"], p=s["p"], m=s["m"], v=s["v"])


def _run_linear(s, c):
    r, i, o = c["rows"], c["inp"], c["out"]
    hip.call("mle_gemm_ex", None, 0, 0, r, o, i, 1.0, _p(s["x"]), i, 0, _p(s["w"]), o, 0, 0.0, _p(s["y"]), o, 0, 1,
             None, _p(s["b"]), s["wsf"].ptr, s["wsf"].nbytes)
    hip.call("mle_linear_bwd_ex", None, r, i, o, 1, _p(s["x"]), _p(s["dy"]), 0, _p(s["w"]), 0, _p(s["dx"]), 0,
             _p(s["dw"]), _p(s["db"]), 0, 0, s["wsb"].ptr, s["wsb"].nbytes)
    return {k: s[k] for k in ("y", "dx", "dw", "db")}


def _run_ffn(s, c):
    call = hip.call
    r, d, f = c["rows"], c["d"], c["ffn"]
    act = hip.ACT[c["act"]]
    call("mle_gemm_ex", None, 0, 0, r, f, d, 1.0, _p(s["x"]), d, 0, _p(s["w1"]), f, 0, 0.0, _p(s["h"]), f, 0, 1, None,
         _p(s["b1"]), s["ws1"].ptr, s["ws1"].nbytes)
    call("mle_act_fwd", None, act, _p(s["h"]), _p(s["a"]), r * f)
    call("mle_gemm_ex", None, 0, 0, r, d, f, 1.0, _p(s["a"]), f, 0, _p(s["w2"]), d, 0, 0.0, _p(s["y"]), d, 0, 1, None,
         _p(s["b2"]), s["ws2"].ptr, s["ws2"].nbytes)
    call("mle_linear_bwd_act", None, r, f, d, _p(s["a"]), _p(s["dy"]), _p(s["w2"]), _p(s["da"]), 0, _p(s["dw2"]),
         _p(s["db2"]), 0, act, _p(s["h"]), _p(s["dh"]), 0, s["wsb2"].ptr, s["wsb2"].nbytes)
    call("mle_linear_bwd_ex", None, r, d, f, 1, _p(s["x"]), _p(s["dh"]), 0, _p(s["w1"]), 0, _p(s["dx"]), 0,
         _p(s["dw1"]), _p(s["db1"]), 0, 0, s["wsb1"].ptr, s["wsb1"].nbytes)
    return {k: s[k] for k in ("y", "dx", "dw1", "db1", "dw2", "db2")}


def _run_attention(s, c):
    b, h, n = c["batch"], c["heads"], c["seq"]
    scale, ws = 1.0 / math.sqrt(HEAD_DIM), s["ws"]
    hip.call("mle_attention_fwd", None, _p(s["q"]), _p(s["k"]), _p(s["v"]), _p(s["out"]), b, h, n, HEAD_DIM,
             h * HEAD_DIM, scale, c["causal"], ws.ptr, ws.nbytes)
    hip.call("mle_attention_bwd", None, _p(s["q"]), _p(s["k"]), _p(s["v"]), _p(s["do"]), _p(s["dq"]), _p(s["dk"]),
             _p(s["dv"]), b, h, n, HEAD_DIM, h * HEAD_DIM, scale, c["causal"], 0, 0, 0, 1, ws.ptr, ws.nbytes)
    return {k: s[k] for k in ("out", "dq", "dk", "dv")}


def _run_lm_head(s, c):
    call = hip.call
    r, d, v = c["rows"], c["d"], c["vocab"]
    ldp = s["part"].shape[1]
    call("mle_gemm_rowstats", None, 0, 0, r, v, d, 1.0, _p(s["x"]), d, _p(s["w"]), v, 0.0, _p(s["logits"]), v,
         _p(s["b"]), _p(s["part"]), ldp, s["wsf"].ptr, s["wsf"].nbytes)
    call("mle_softmax_xent_keys_fwd_rowstats", None, _p(s["logits"]), _p(s["part"]), ldp, _p(s["keys"]), r, r,
         _p(s["stats"]), r, v, _p(s["loss"]), s["wsl"].ptr, s["wsl"].nbytes)
    call("mle_softmax_xent_keys_bwd", None, _p(s["logits"]), _p(s["stats"]), _p(s["keys"]), r, r, None,
         _p(s["dlogits"]), r, v, r)
    call("mle_linear_bwd_ex", None, r, d, v, 1, _p(s["x"]), _p(s["dlogits"]), 0, _p(s["w"]), 0, _p(s["dx"]), 0,
         _p(s["dw"]), _p(s["db"]), 0, 0, s["wsb"].ptr, s["wsb"].nbytes)
    return {k: s[k] for k in ("logits", "loss", "dlogits", "dx", "dw", "db")}


def _run_norm_add(s, c):
    b, n, ws = c["batch"], c["rows"] * c["cols"], s["ws"]
    hip.call("mle_add_norm_partials", None, _p(s["a"]), _p(s["b"]), b * n, _p(s["r"]), b, 1, n, 1, ws.ptr, ws.nbytes)
    hip.call("mle_norm_fwd_ex", None, _p(s["r"]), _p(s["y"]), _p(s["stats"]), b, 1, n, 1, EPS, ws.ptr, ws.nbytes, 1)
    hip.call("mle_norm_bwd_partials", None, _p(s["y"]), _p(s["dy"]), None, -1, 0, b, 1, n, 1, 0, ws.ptr, ws.nbytes)
    hip.call("mle_norm_bwd_apply_add", None, _p(s["y"]), _p(s["dy"]), _p(s["dr"]), 1, _p(s["dres"]), _p(s["da"]), 0,
             _p(s["db"]), 0, _p(s["stats"]), b, 1, n, 1, EPS, 0, ws.ptr, ws.nbytes)
    return {k: s[k] for k in ("r", "y", "dr", "da", "db")}


def _run_group_act(s, c):
    b, ch, hw, gr, ws = c["batch"], c["channels"], c["h"] * c["w"], c["groups"], s["ws"]
    act = hip.ACT[c["act"]]
    hip.call("mle_norm_fwd_act", None, _p(s["x"]), _p(s["y"]), _p(s["a"]), act, _p(s["stats"]), b, ch, hw, gr, EPS,
             ws.ptr, ws.nbytes, 0)
    hip.call("mle_norm_bwd_act", None, _p(s["y"]), _p(s["da"]), act, _p(s["dy"]), 0, _p(s["dx"]), _p(s["stats"]), b, ch,
             hw, gr, EPS, 0, ws.ptr, ws.nbytes, 0)
    return {k: s[k] for k in ("y", "a", "dy", "dx")}


def _run_conv(s, c):
    pad, _, _ = _conv_out(c)
    dims = (c["n"], c["cin"], c["h"], c["w"], c["cout"], c["k"], c["k"], pad, c["stride"])
    ws = s["ws"]
    hip.call("mle_conv2d_fwd", None, _p(s["x"]), _p(s["w"]), _p(s["b"]), _p(s["y"]), *dims)
    hip.call("mle_conv2d_dgrad", None, _p(s["dy"]), _p(s["w"]), _p(s["dx"]), *dims, 0)
    hip.call("mle_conv2d_wgrad_bias", None, _p(s["x"]), _p(s["dy"]), _p(s["dw"]), _p(s["db"]), 0, *dims, ws.ptr,
             ws.nbytes)
    return {k: s[k] for k in ("y", "dx", "dw", "db")}


def _run_adamw(s, c):
    ws = s["ws"]
    hip.call("mle_adamw_clip_fused", None, _p(s["p"]), _p(s["g"]), _p(s["m"]), _p(s["v"]), c["n"], s["t"], ADAM["lr"],
             ADAM["b1"], ADAM["b2"], ADAM["eps"], ADAM["wd"], 1, 1.0, _p(s["norm"]), ws.ptr, ws.nbytes)
    s["t"] += 1
    return {k: s[k] for k in ("p", "m", "v", "norm")}


_RUN = dict(mlp_step=_run_mlp, linear=_run_linear, ffn=_run_ffn, attention=_run_attention, lm_head=_run_lm_head,
            norm_add=_run_norm_add, group_act=_run_group_act, conv=_run_conv, adamw=_run_adamw)

# ---------------------------------------------------------------- work, tolerance


def work(case: dict) -> dict:
    c, k = case, case["kind"]
    if k == "mlp_step":
        n, i, h, o = c["batch"], c["inp"], c["hidden"], c["classes"]
        par = i * h + h + h * o + o
        # inputs and parameters read, moments and parameters read and written,
        # gradients, logits and the input's gradient written
        return dict(flops=6.0 * n * (i * h + h * o), bytes=4.0 * (2 * n * i + n * o + n + 7 * par))
    if k == "linear":
        r, i, o = c["rows"], c["inp"], c["out"]
        return dict(flops=6.0 * r * i * o, bytes=4.0 * (2 * r * i + 2 * r * o + 2 * i * o + 2 * o))
    if k == "ffn":
        r, d, f = c["rows"], c["d"], c["ffn"]
        return dict(flops=12.0 * r * d * f, bytes=4.0 * (4 * r * d + 4 * d * f + 2 * (d + f)))
    if k == "attention":
        b, h, n = c["batch"], c["heads"], c["seq"]
        # two products forward, four backward (and the scores and dP once
        # each), over the unmasked half when causal
        half = (n + 1) / (2.0 * n) if c["causal"] else 1.0
        return dict(flops=6 * 2.0 * b * h * n * n * HEAD_DIM * half, bytes=4.0 * 8 * b * n * h * HEAD_DIM)
    if k == "lm_head":
        r, d, v = c["rows"], c["d"], c["vocab"]
        return dict(flops=6.0 * r * d * v, bytes=4.0 * (2 * r * d + 2 * d * v + 2 * r * v + r + 2 * v))
    if k == "norm_add":
        # a, b, dy, dres read; r, y, dr, da, db written
        return dict(flops=0.0, bytes=4.0 * 9 * c["batch"] * c["rows"] * c["cols"])
    if k == "group_act":
        # x, da read; y, a, dy, dx written
        return dict(flops=0.0, bytes=4.0 * 6 * c["batch"] * c["channels"] * c["h"] * c["w"])
    if k == "conv":
        _, oh, ow = _conv_out(c)
        n, ci, co, kk = c["n"], c["cin"], c["cout"], c["k"] * c["k"]
        return dict(flops=6.0 * n * co * oh * ow * ci * kk,
                    bytes=4.0 * (2 * n * ci * c["h"] * c["w"] + 2 * n * co * oh * ow + 2 * co * ci * kk + 2 * co))
    return dict(flops=0.0, bytes=28.0 * c["n"])  # p, g, m, v read; p, m, v written


# About four times the relative error against 64 bits that the float32 path
# shows over the declared ranges.
_TOLERANCE = dict(mlp_step=1e-5, linear=8e-6, ffn=8e-6, attention=4e-6, lm_head=8e-6, norm_add=1e-6, group_act=1e-6,
                  conv=5e-6, adamw=1e-6)


def tolerance(case: dict):
    rel = _TOLERANCE[case["kind"]]
    if case["kind"] == "mlp_step" and case["batch"] * case["hidden"] > 50_000:
        # With this many hidden values one may lie so near 0 that its rounding
        # decides the ReLU: that moves dW1 by about one part in the square
        # root of the active values, and single elements of it by their size.
        return dict(rel=4 * math.sqrt(2.0 / (case["batch"] * case["hidden"])), max=0.5)
    return dict(rel=rel, max=40 * rel)


# --------------------------------------------------------------------- exact


def exact(case: dict, seed: int):
    """What run() returns for prepare(case, seed), in 64 bits with torch alone."""
    s = prepare(case, seed)
    return _EXACT[case["kind"]](s, case)


def _act(kind, x):
    """The library's activations (its GELU is the tanh form)."""
    if kind == "relu":
        return x.clamp(min=0)
    if kind == "silu":
        return x * torch.sigmoid(x)
    return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))


def _act_grad(kind, x):
    x = x.detach().requires_grad_(True)
    if kind == "relu":
        return (x > 0).to(x.dtype)
    return torch.autograd.grad(_act(kind, x).sum(), x)[0].detach()


def _d(s, *names):
    return [s[n].double() for n in names]


def _adam_exact(p, g, m, v, t):
    m = ADAM["b1"] * m + (1 - ADAM["b1"]) * g
    v = ADAM["b2"] * v + (1 - ADAM["b2"]) * g * g
    mh, vh = m / (1 - ADAM["b1"] ** t), v / (1 - ADAM["b2"] ** t)
    return p - ADAM["lr"] * (mh / (vh.sqrt() + ADAM["eps"]) + ADAM["wd"] * p), m, v


def _exact_mlp(s, c):
    n, i, h, k = c["batch"], c["inp"], c["hidden"], c["classes"]
    x, p, m, v = _d(s, "x", "p", "m", "v")
    w1, b1, w2, b2 = torch.split(p, [i * h, h, h * k, k])
    w1, w2 = w1.view(i, h), w2.view(h, k)
    hid = x @ w1 + b1
    a = hid.clamp(min=0)
    logits = a @ w2 + b2
    keys = s["keys"].long()
    prob = torch.softmax(logits, 1)
    onehot = F.one_hot(keys, k).double()
    loss = -(onehot * torch.log(prob + 1e-27)).sum() / (n * k)
    dl = (prob - onehot) / n
    dh = (dl @ w2.T) * (hid > 0)
    g = torch.cat([(x.T @ dh).reshape(-1), dh.sum(0), (a.T @ dl).reshape(-1), dl.sum(0)])
    p, m, v = _adam_exact(p, g, m, v, s["t"])
    return dict(loss=float(loss), logits=logits, grads=g, p=p, m=m, v=v)


def _exact_linear(s, c):
    x, w, b, dy = _d(s, "x", "w", "b", "dy")
    return dict(y=x @ w + b, dx=dy @ w.T, dw=x.T @ dy, db=dy.sum(0))


def _exact_ffn(s, c):
    x, w1, b1, w2, b2, dy = _d(s, "x", "w1", "b1", "w2", "b2", "dy")
    h = x @ w1 + b1
    a = _act(c["act"], h)
    dh = (dy @ w2.T) * _act_grad(c["act"], h)
    return dict(y=a @ w2 + b2, dx=dh @ w1.T, dw1=x.T @ dh, db1=dh.sum(0), dw2=a.T @ dy, db2=dy.sum(0))


def _exact_attention(s, c):
    b, h, n, hd = c["batch"], c["heads"], c["seq"], HEAD_DIM
    scale = 1.0 / math.sqrt(hd)
    outs = {k: torch.empty(b, n, h * hd, dtype=torch.float64, device=DEV) for k in ("out", "dq", "dk", "dv")}
    keep = torch.ones(n, n, dtype=torch.bool, device=DEV).tril() if c["causal"] else None
    for i in range(b):
        q, k, v, do = (t[i].double().view(n, h, hd).transpose(0, 1).contiguous()
                       for t in (s["q"], s["k"], s["v"], s["do"]))
        kt, vt = k.transpose(1, 2).contiguous(), v.transpose(1, 2).contiguous()
        sc = (q @ kt) * scale
        e = (sc - sc.amax(1, keepdim=True)).exp()  # each key's maximum over every query
        if keep is not None:
            e = e * keep
        p = e / e.sum(1, keepdim=True)
        dp = do @ vt
        ds = p * (dp - (p * dp).sum(1, keepdim=True))
        flat = lambda t: t.transpose(0, 1).reshape(n, h * hd)  # noqa: E731
        outs["out"][i] = flat(p @ v)
        outs["dv"][i] = flat(p.transpose(1, 2).contiguous() @ do)
        outs["dq"][i] = flat(scale * (ds @ k))
        # the reference's K gradient: (dS q)^T, its rows written one after
        # another into the head's [n, 64] block
        dk = scale * (ds @ q)
        outs["dk"][i] = flat(dk.transpose(1, 2).reshape(h, n, hd))
    return outs


def _exact_lm_head(s, c):
    r, v = c["rows"], c["vocab"]
    x, w, b = _d(s, "x", "w", "b")
    logits = x @ w + b
    rows, keys = torch.arange(r, device=DEV), s["keys"].long()
    dl = torch.softmax(logits, 1)
    loss = -torch.log(dl[rows, keys] + 1e-27).sum() / (r * v)
    dl[rows, keys] -= 1
    dl /= r
    return dict(logits=logits, loss=loss.view(1), dlogits=dl, dx=dl @ w.T, dw=x.T @ dl, db=dl.sum(0))


def _norm(x, dims):
    mean = x.mean(dims, keepdim=True)
    var = (x - mean).square().mean(dims, keepdim=True)
    rstd = (var + EPS).rsqrt()
    return (x - mean) * rstd, rstd


def _norm_grad(y, dy, rstd, dims):
    return rstd * (dy - dy.mean(dims, keepdim=True) - y * (dy * y).mean(dims, keepdim=True))


def _exact_norm_add(s, c):
    a, b, dy, dres = _d(s, "a", "b", "dy", "dres")
    r = a + b
    y, rstd = _norm(r, (1, 2))
    dr = dres + _norm_grad(y, dy, rstd, (1, 2))
    return dict(r=r, y=y, dr=dr, da=dr, db=dr)


def _exact_group_act(s, c):
    shape = (c["batch"], c["groups"], -1)
    x, da = (t.view(shape) for t in _d(s, "x", "da"))
    y, rstd = _norm(x, (2,))
    dy = da * _act_grad(c["act"], y)
    full = lambda t: t.reshape(s["x"].shape)  # noqa: E731
    return dict(y=full(y), a=full(_act(c["act"], y)), dy=full(dy), dx=full(_norm_grad(y, dy, rstd, (2,))))


def _exact_conv(s, c):
    n, ci, co, k, st = c["n"], c["cin"], c["cout"], c["k"], c["stride"]
    pad, oh, ow = _conv_out(c)
    w = s["w"].double().view(co, -1)
    out = dict(y=torch.empty(n, co, oh, ow, dtype=torch.float64, device=DEV),
               dx=torch.empty(n, ci, c["h"], c["w"], dtype=torch.float64, device=DEV))
    dw = torch.zeros_like(w)
    for i in range(n):
        cols = F.unfold(s["x"][i:i + 1].double(), k, padding=pad, stride=st)[0]
        dy = s["dy"][i].double().view(co, -1)
        out["y"][i] = (w @ cols + s["b"].double()[:, None]).view(co, oh, ow)
        out["dx"][i] = F.fold((w.T @ dy)[None], (c["h"], c["w"]), k, padding=pad, stride=st)[0]
        dw += dy @ cols.T
    return dict(out, dw=dw.view(co, ci, k, k), db=s["dy"].double().sum((0, 2, 3)))


def _exact_adamw(s, c):
    p, g, m, v = _d(s, "p", "g", "m", "v")
    norm = g.square().sum().sqrt().clamp(min=1.0)
    p, m, v = _adam_exact(p, g / norm, m, v, s["t"])
    return dict(p=p, m=m, v=v, norm=norm.view(1))


_EXACT = dict(mlp_step=_exact_mlp, linear=_exact_linear, ffn=_exact_ffn, attention=_exact_attention,
              lm_head=_exact_lm_head, norm_add=_exact_norm_add, group_act=_exact_group_act, conv=_exact_conv,
              adamw=_exact_adamw)
