"""The work that users of this library have it do, as measurable cases.

Each listed case is a call (or a short chain of calls) through the public
entry points on device-resident buffers, as a program that keeps its data on
the GPU makes them; ``draw`` gives further cases of the same families over the
whole range of sizes, types, layouts and options.  The families:

===============  ==========================================================
gn               GroupNorm (+ SiLU): the executor's fp32 NCHW op and the
                 channels-last fp16 form; the smallest calls, where latency
                 and launches count
conv32           the executor's Conv: NCHW fp32, with the fused bias / SiLU /
                 residual epilogue of the conv bench
conv16           channels-last fp16 conv (3x3, 1x1, stride 2, 2x upsample)
resnet           ResNet block with timestep embedding
transformer      Transformer block (self-attention, cross-attention, GEGLU)
attn             flash self-attention, from bench size to the 96x96 latent
cross            cross-attention over text tokens
ffn              feed-forward block: fp32 tanh-GELU and fp16 GEGLU
exec_attn        attention the executor's way, one op per call on fp32:
                 transposes, MatMul, scale, Softmax, MatMul, transpose
unet             one whole denoise step (SD2.1 architecture, graph replay)
vae              one whole image decode (graph replay)
===============  ==========================================================

Every output is the whole device buffer; it is read back only when somebody
looks at it (``Outputs``), because a program that chains calls on the device
does not copy between them.
"""
from __future__ import annotations

import math
import os
import sys
import zlib

import numpy as np
import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.getcwd(), "draw-instant_amd"))

from drawinstant import F16, F32, NCHW, NHWC, Device, call  # noqa: E402
from drawinstant import blocks as di_blocks  # noqa: E402
from drawinstant.executor import create_dispatchers, row_major_strides  # noqa: E402
from drawinstant.unet import UNet  # noqa: E402
from drawinstant.vae import VAE  # noqa: E402

CONV_UPSAMPLE2X, CONV_SILU = 2, 4
ACT_GELU, ACT_GEGLU, ACT_GELU_TANH = 1, 2, 4
CONTEXT_TOKENS, CONTEXT_DIM, TIME_DIM, GROUPS = 77, 1024, 1280, 32
VAE_SCALE = 1.0 / 0.18215

# What a drawn case may cost, in operations and in bytes moved by its calls:
# below the largest listed case of every family.
MAX_FLOPS = {"conv32": 3.0e10, "conv16": 1.2e11, "resnet": 1.5e11, "transformer": 1.2e11,
             "attn": 2.2e11, "cross": 2.0e10, "ffn": 1.1e11}
MAX_BYTES = 2.0e8


def listed():
    return [
        # the executor's GroupNorm + SiLU at the first level of a 512 x 512 image
        {"name": "gn_silu_f32_320x64x64", "kind": "gn", "N": 1, "C": 320, "H": 64, "W": 64,
         "silu": True, "f16": False},
        # the conv bench: bias, SiLU and residual in one exact fp32 call
        {"name": "conv3x3_f32_1280x16x16", "kind": "conv32", "N": 1, "Cin": 1280, "Cout": 1280,
         "H": 16, "W": 16, "K": 3, "S": 1, "silu": True, "res": True},
        # the most frequent conv of a denoise step
        {"name": "conv3x3_f16_320x64x64", "kind": "conv16", "N": 1, "Cin": 320, "Cout": 320,
         "H": 64, "W": 64, "K": 3, "S": 1, "up": 1},
        # a level change of the U-Net, one image
        {"name": "resnet_320_640_32x32", "kind": "resnet", "B": 1, "Cin": 320, "Cout": 640,
         "H": 32, "W": 32},
        # the largest transformer block of a 512 x 512 step
        {"name": "transformer_320_64x64", "kind": "transformer", "B": 1, "C": 320, "H": 64, "W": 64,
         "S": 77},
        # self-attention of a 768 x 768 image, a guided pair of samples
        {"name": "attn_f16_b2_h5_s9216", "kind": "attn", "B": 2, "H": 5, "S": 9216, "f16": True,
         "bhsd": False},
        # the cross-attention bench: a guided pair over 77 text tokens
        {"name": "cross_f32_b2_h20_s256x77", "kind": "cross", "B": 2, "H": 20, "Sq": 256,
         "Skv": 77, "f16": False, "bhsd": True},
        # the feed-forward bench, fp32 as the executor holds it
        {"name": "ffn_f32_2048x1280x5120", "kind": "ffn", "rows": 2048, "D": 1280, "F": 5120,
         "act": ACT_GELU_TANH, "f16": False},
        # GEGLU feed-forward of a batch of four 640 x 512 images' second level (40 x 32 pixels)
        {"name": "ffn_geglu_f16_5120x640x2560", "kind": "ffn", "rows": 5120, "D": 640, "F": 2560,
         "act": ACT_GEGLU, "f16": True},
        # a self-attention of the exported graph, run one op per node
        {"name": "exec_attn_f32_h5_s2304", "kind": "exec_attn", "B": 1, "H": 5, "S": 2304},
        # the headline: one denoise step of a 512 x 512 image
        {"name": "unet_step_b1_64x64", "kind": "unet", "B": 1, "H": 64, "W": 64},
        # decode of the architecture's native 768 x 768 image
        {"name": "vae_decode_96x96", "kind": "vae", "B": 1, "H": 96, "W": 96},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_kind(rng, kind):
    if kind == "gn":
        return {"kind": kind, "N": rng.choice([1, 1, 2, 3, 4]), "C": 32 * rng.randint(2, 60),
                "H": _log(rng, 8, 128), "W": _log(rng, 8, 128), "silu": rng.random() < 0.7,
                "f16": rng.random() < 0.4}
    if kind == "conv32":
        c = {"kind": kind, "N": rng.choice([1, 1, 2]),
             "Cin": rng.choice([4, 64, 128, 320, 512, 640, 960, 1280, 1920, rng.randint(3, 700)]),
             "Cout": rng.choice([4, 64, 128, 320, 512, 640, 1280, rng.randint(3, 700)]),
             "H": _log(rng, 8, 72), "W": _log(rng, 8, 72), "K": rng.choice([1, 3, 3]),
             "S": rng.choice([1, 1, 1, 2]), "silu": rng.random() < 0.3}
        c["res"] = rng.random() < 0.4
        return c
    if kind == "conv16":
        up = rng.choice([1, 1, 1, 2])
        return {"kind": kind, "N": rng.choice([1, 1, 2, 4]),
                "Cin": rng.choice([64, 128, 256, 320, 512, 640, 960, 1280, 1920,
                                   8 * rng.randint(2, 160)]),
                "Cout": rng.choice([64, 128, 256, 320, 512, 640, 1280, 8 * rng.randint(2, 160)]),
                "H": _log(rng, 8, 128), "W": _log(rng, 8, 128),
                "K": rng.choice([1, 3, 3, 3]), "S": 1 if up == 2 else rng.choice([1, 1, 1, 2]),
                "up": up}
    if kind == "resnet":
        return {"kind": kind, "B": rng.choice([1, 1, 2, 3, 4]),
                "Cin": rng.choice([64, 320, 640, 960, 1280, 32 * rng.randint(2, 60)]),
                "Cout": rng.choice([64, 320, 640, 1280, 32 * rng.randint(2, 40)]),
                "H": _log(rng, 8, 96), "W": _log(rng, 8, 96)}
    if kind == "transformer":
        return {"kind": kind, "B": rng.choice([1, 1, 2, 3, 4]),
                "C": rng.choice([320, 640, 1280, 64 * rng.randint(1, 20)]),
                "H": _log(rng, 8, 96), "W": _log(rng, 8, 96), "S": rng.choice([77, 77, 77, 154, 20])}
    if kind == "attn":
        return {"kind": kind, "B": rng.choice([1, 2, 2, 4]), "H": rng.choice([5, 10, 20, rng.randint(1, 20)]),
                "S": _log(rng, 64, 16384), "f16": rng.random() < 0.6, "bhsd": rng.random() < 0.5}
    if kind == "cross":
        return {"kind": kind, "B": rng.choice([1, 2, 2, 4]), "H": rng.choice([5, 10, 20, rng.randint(1, 20)]),
                "Sq": _log(rng, 64, 16384), "Skv": rng.choice([77, 77, 154, rng.randint(1, 300)]),
                "f16": rng.random() < 0.6, "bhsd": rng.random() < 0.5}
    if kind == "ffn":
        d = rng.choice([320, 640, 1280, 64 * rng.randint(1, 20)])
        f16 = rng.random() < 0.5
        return {"kind": kind, "rows": _log(rng, 64, 16384), "D": d, "F": 4 * d,
                "act": rng.choice([ACT_GEGLU, ACT_GELU, ACT_GELU_TANH]), "f16": f16}
    if kind == "exec_attn":
        return {"kind": kind, "B": rng.choice([1, 1, 2]), "H": rng.choice([5, 10, 20, rng.randint(1, 20)]),
                "S": _log(rng, 64, 4096)}
    if kind == "unet":
        return {"kind": kind, "B": rng.choice([1, 1, 2, 4]), "H": 8 * rng.randint(2, 12),
                "W": 8 * rng.randint(2, 12)}
    return {"kind": "vae", "B": rng.choice([1, 1, 2]), "H": rng.randint(8, 80),
            "W": rng.randint(8, 80)}


def draw(rng):
    kind = rng.choice(["gn", "conv32", "conv16", "resnet", "transformer", "attn", "cross", "ffn",
                       "exec_attn", "unet", "vae"])
    while True:
        c = _draw_kind(rng, kind)
        w = work(c)
        if kind == "unet":
            if c["B"] * c["H"] * c["W"] <= 2 * 64 * 64:
                return c
        elif kind == "vae":
            if c["B"] * c["H"] * c["W"] <= 64 * 64:
                return c
        elif kind == "exec_attn":
            if c["B"] * c["H"] * c["S"] ** 2 <= 5 * 2304 ** 2:
                return c
        elif w["flops"] <= MAX_FLOPS.get(kind, 1e12) and w["bytes"] <= MAX_BYTES:
            return c


# ------------------------------------------------------------------ device --
_kept = {}


def _dev() -> Device:
    if "dev" not in _kept:
        _kept["dev"] = Device(0)
    return _kept["dev"]


class _Owned:
    """Device buffers that go back to the pool with their last user."""

    def __init__(self):
        self.items = []

    def storage(self, a):
        self.items.append(_dev().storage(a))
        return self.items[-1]

    def create(self, nbytes):
        self.items.append(_dev().create_buffer(nbytes))
        return self.items[-1]

    def keep(self, x):
        self.items.append(x)
        return x

    def __del__(self):
        try:
            for x in self.items:
                x.destroy()
        except Exception:
            pass


class Outputs(dict):
    """Named device buffers, read back when an entry is looked up."""

    def __init__(self, owner, **specs):
        super().__init__(specs)  # name -> (buffer, numpy dtype, shape)
        self._owner = owner

    def __getitem__(self, name):
        buf, dt, shape = dict.__getitem__(self, name)
        return torch.from_numpy(_dev().download(buf, dt, shape))


def _rng(case, seed):
    return np.random.default_rng([int(seed) & 0x7FFFFFFF, zlib.crc32(case["kind"].encode())])


def _normal(rng, shape, std=1.0, mean=0.0):
    a = rng.standard_normal(shape, dtype=np.float32)
    if std != 1.0:
        a *= np.float32(std)
    if mean:
        a += np.float32(mean)
    return a


def _affine(rng, sd, p, c):
    sd[p + ".weight"] = _normal(rng, (c,), 0.02, 1.0)
    sd[p + ".bias"] = _normal(rng, (c,), 0.02)


def _linear(rng, sd, p, o, i, bias=True):
    sd[p + ".weight"] = _normal(rng, (o, i), 1.0 / math.sqrt(i))
    if bias:
        sd[p + ".bias"] = _normal(rng, (o,), 0.02)


def _conv(rng, sd, p, o, i, k):
    sd[p + ".weight"] = _normal(rng, (o, i, k, k), math.sqrt(2.0 / (i * k * k)))
    sd[p + ".bias"] = _normal(rng, (o,), 0.01)


# ------------------------------------------------------------ host inputs --
# The arrays of a case, from its seed alone; ``prepare`` uploads them and
# ``exact`` computes on them.
def _conv_out(c):
    hi, wi = c["H"] * c.get("up", 1), c["W"] * c.get("up", 1)
    p = c["K"] // 2
    return (hi + 2 * p - c["K"]) // c["S"] + 1, (wi + 2 * p - c["K"]) // c["S"] + 1


def _inputs(c, seed):
    r, k = _rng(c, seed), c["kind"]
    if k == "gn":
        return {"x": _normal(r, (c["N"], c["C"], c["H"], c["W"])),
                "g": _normal(r, (c["C"],), 0.02, 1.0), "b": _normal(r, (c["C"],), 0.02)}
    if k in ("conv32", "conv16"):
        d = {"x": _normal(r, (c["N"], c["Cin"], c["H"], c["W"]))}
        _conv(r, d, "c", c["Cout"], c["Cin"], c["K"])
        if c.get("res"):
            d["r"] = _normal(r, (c["N"], c["Cout"]) + _conv_out(c))
        return d
    if k == "resnet":
        d = {"x": _normal(r, (c["B"], c["Cin"], c["H"], c["W"])),
             "temb": _normal(r, (c["B"], TIME_DIM))}
        _affine(r, d, "p.norm1", c["Cin"])
        _conv(r, d, "p.conv1", c["Cout"], c["Cin"], 3)
        _linear(r, d, "p.time_emb_proj", c["Cout"], TIME_DIM)
        _affine(r, d, "p.norm2", c["Cout"])
        _conv(r, d, "p.conv2", c["Cout"], c["Cout"], 3)
        if c["Cin"] != c["Cout"]:
            _conv(r, d, "p.conv_shortcut", c["Cout"], c["Cin"], 1)
        return d
    if k == "transformer":
        C, t = c["C"], "p.transformer_blocks.0"
        d = {"x": _normal(r, (c["B"], C, c["H"], c["W"])),
             "ctx": _normal(r, (c["B"], c["S"], CONTEXT_DIM))}
        _affine(r, d, "p.norm", C)
        _linear(r, d, "p.proj_in", C, C)
        for i in (1, 2, 3):
            _affine(r, d, f"{t}.norm{i}", C)
        for a, kv in (("attn1", C), ("attn2", CONTEXT_DIM)):
            _linear(r, d, f"{t}.{a}.to_q", C, C, False)
            _linear(r, d, f"{t}.{a}.to_k", C, kv, False)
            _linear(r, d, f"{t}.{a}.to_v", C, kv, False)
            _linear(r, d, f"{t}.{a}.to_out.0", C, C)
        _linear(r, d, f"{t}.ff.net.0.proj", 8 * C, C)
        _linear(r, d, f"{t}.ff.net.2", C, 4 * C)
        _linear(r, d, "p.proj_out", C, C)
        return d
    if k in ("attn", "cross", "exec_attn"):
        sq = c.get("Sq", c.get("S"))
        skv = c.get("Skv", c.get("S"))
        sh = (lambda s: (c["B"], c["H"], s, 64)) if c.get("bhsd") else (lambda s: (c["B"], s, c["H"], 64))
        return {"q": _normal(r, sh(sq)), "k": _normal(r, sh(skv)), "v": _normal(r, sh(skv))}
    if k == "ffn":
        n1 = c["F"] * (2 if c["act"] == ACT_GEGLU else 1)
        return {"x": _normal(r, (c["rows"], c["D"])),
                "w1": _normal(r, (n1, c["D"]), 1.0 / math.sqrt(c["D"])),
                "b1": _normal(r, (n1,), 0.02),
                "w2": _normal(r, (c["D"], c["F"]), 1.0 / math.sqrt(c["F"])),
                "b2": _normal(r, (c["D"],), 0.02)}
    if k == "unet":
        return {"x": _normal(r, (c["B"], 4, c["H"], c["W"])),
                "t": r.integers(1, 1000, c["B"]).astype(np.float32),
                "ctx": _normal(r, (c["B"], CONTEXT_TOKENS, CONTEXT_DIM))}
    return {"x": _normal(r, (c["B"], 4, c["H"], c["W"]), 0.18215 * 5.0)}


def _tokens(a):
    """NCHW -> channels-last fp16."""
    return np.ascontiguousarray(a.transpose(0, 2, 3, 1)).astype(np.float16)


def _typed(c, a):
    return a.astype(np.float16) if c["f16"] else a


# ----------------------------------------------------------- whole models --
def _unet() -> UNet:
    if "unet" not in _kept:
        _kept["unet"] = UNet(_dev(), seed=11)
    return _kept["unet"]


def _vae() -> VAE:
    if "vae" not in _kept:
        _kept["vae"] = VAE(_dev(), seed=11)
    return _kept["vae"]


def _session(c):
    """The fixed buffers a program captures its graph on, one set per shape:
    new inputs are copied into them."""
    key = (c["kind"], c["B"], c["H"], c["W"])
    if _kept.get("session_key") != key:
        for b in _kept.get("session", ()):
            b.destroy()
        B, n = c["B"], c["B"] * 4 * c["H"] * c["W"] * 4
        mk = _dev().create_buffer
        _kept["session"] = (mk(n), mk(4 * B), mk(B * CONTEXT_TOKENS * CONTEXT_DIM * 4), mk(n)) \
            if c["kind"] == "unet" else (mk(n), mk(n * 48))
        _kept["session_key"] = key
    return _kept["session"]


# ---------------------------------------------------------------- prepare --
def prepare(case, seed):
    c, k = case, case["kind"]
    dev, own = _dev(), _Owned()
    d = _inputs(c, seed)
    ctx = dev.ctx

    if k == "gn":
        x = own.storage(_tokens(d["x"]) if c["f16"] else d["x"])
        g, b = own.storage(d["g"]), own.storage(d["b"])
        dt, lay, npdt = (F16, NHWC, np.float16) if c["f16"] else (F32, NCHW, np.float32)
        y = own.create(d["x"].size * np.dtype(npdt).itemsize)
        shape = (c["N"], c["H"], c["W"], c["C"]) if c["f16"] else d["x"].shape
        out = Outputs(own, y=(y, npdt, shape))
        args = (ctx, x.handle, g.handle, b.handle, y.handle, c["N"], GROUPS, c["C"] // GROUPS,
                c["H"] * c["W"], 1e-5, 1 if c["silu"] else 0, dt, lay)
        return {"go": lambda: call("di_group_norm", *args), "out": out}

    if k in ("conv32", "conv16"):
        ho, wo = _conv_out(c)
        f16 = k == "conv16"
        x = own.storage(_tokens(d["x"]) if f16 else d["x"])
        w = own.storage(di_blocks.conv_ohwi(d["c.weight"]) if f16 else d["c.weight"])
        b = own.storage(d["c.bias"])
        r = own.storage(d["r"]) if "r" in d else None
        npdt = np.float16 if f16 else np.float32
        y = own.create(c["N"] * c["Cout"] * ho * wo * np.dtype(npdt).itemsize)
        shape = (c["N"], ho, wo, c["Cout"]) if f16 else (c["N"], c["Cout"], ho, wo)
        flags = (CONV_SILU if c.get("silu") else 0) | (CONV_UPSAMPLE2X if c.get("up") == 2 else 0)
        args = (ctx, x.handle, w.handle, b.handle, r.handle if r else 0, y.handle, c["N"],
                c["Cin"], c["Cout"], c["H"], c["W"], c["K"], c["S"], c["K"] // 2, flags,
                F16 if f16 else F32, NHWC if f16 else NCHW)
        return {"go": lambda: call("di_conv2d", *args), "out": Outputs(own, y=(y, npdt, shape))}

    if k == "resnet":
        w = own.keep(di_blocks.upload_resnet(dev, d, "p"))
        x, temb = own.storage(_tokens(d["x"])), own.storage(d["temb"])
        shape = (c["B"], c["H"], c["W"], c["Cout"])
        y = own.create(int(np.prod(shape)) * 2)
        return {"go": lambda: di_blocks.resnet_block(dev, w, x, temb, y, c["B"], c["Cin"],
                                                     c["Cout"], c["H"], c["W"]),
                "out": Outputs(own, y=(y, np.float16, shape))}

    if k == "transformer":
        w = own.keep(di_blocks.upload_transformer(dev, d, "p"))
        x, cx = own.storage(_tokens(d["x"])), own.storage(d["ctx"].astype(np.float16))
        shape = (c["B"], c["H"], c["W"], c["C"])
        y = own.create(int(np.prod(shape)) * 2)
        return {"go": lambda: di_blocks.transformer_block(dev, w, x, cx, y, c["B"], c["C"],
                                                          c["H"], c["W"], c["S"], CONTEXT_DIM),
                "out": Outputs(own, y=(y, np.float16, shape))}

    if k in ("attn", "cross"):
        q, kk, v = (own.storage(_typed(c, d[n])) for n in "qkv")
        npdt = np.float16 if c["f16"] else np.float32
        y = own.create(d["q"].size * np.dtype(npdt).itemsize)
        tail = (64, 1 if c["bhsd"] else 0, 0.0, F16 if c["f16"] else F32)
        head = (ctx, q.handle, kk.handle, v.handle, y.handle, c["B"], c["H"])
        out = Outputs(own, y=(y, npdt, d["q"].shape))
        if k == "attn":
            return {"go": lambda: call("di_attn_self", *head, c["S"], *tail), "out": out}
        return {"go": lambda: call("di_attn_cross", *head, c["Sq"], c["Skv"], *tail), "out": out}

    if k == "ffn":
        if c["act"] == ACT_GEGLU:  # rows in groups of [16 hidden | 16 gate]
            d["w1"], d["b1"] = _geglu_rows(d["w1"]), _geglu_rows(d["b1"])
        x, w1, w2 = (own.storage(_typed(c, d[n])) for n in ("x", "w1", "w2"))
        b1, b2 = own.storage(d["b1"]), own.storage(d["b2"])
        npdt = np.float16 if c["f16"] else np.float32
        y = own.create(d["x"].size * np.dtype(npdt).itemsize)
        args = (ctx, x.handle, w1.handle, b1.handle, w2.handle, b2.handle, y.handle, c["rows"],
                c["D"], c["F"], c["act"], F16 if c["f16"] else F32)
        return {"go": lambda: call("di_ffn", *args),
                "out": Outputs(own, y=(y, npdt, d["x"].shape))}

    if k == "exec_attn":
        return _prepare_exec_attn(c, d, own)

    if k == "unet":
        u = _unet()
        xs, ts, cx = own.storage(d["x"]), own.storage(d["t"]), own.storage(d["ctx"])
        y = own.create(d["x"].nbytes)
        state = {"out": Outputs(own, y=(y, np.float32, d["x"].shape))}

        def step():
            sx, st, sc, so = _session(c)
            dev.copy(sx, xs, d["x"].nbytes)
            dev.copy(st, ts, d["t"].nbytes)
            dev.copy(sc, cx, d["ctx"].nbytes)
            u.forward(sx, st, sc, so, c["B"], c["H"], c["W"], CONTEXT_TOKENS, graph=True)
            dev.copy(y, so, d["x"].nbytes)
        state["go"] = step
        return state

    v = _vae()
    z = own.storage(d["x"])
    shape = (c["B"], 3, 8 * c["H"], 8 * c["W"])
    nb = int(np.prod(shape)) * 4
    y = own.create(nb)

    def decode():
        sz, si = _session(c)
        dev.copy(sz, z, d["x"].nbytes)
        v.decode(sz, si, c["B"], c["H"], c["W"], VAE_SCALE, graph=True)
        dev.copy(y, si, nb)
    return {"go": decode, "out": Outputs(own, y=(y, np.float32, shape))}


def _geglu_rows(a):
    hid, gate = np.split(a, 2, axis=0)
    n = hid.shape[0] // 16
    return np.ascontiguousarray(np.concatenate([hid.reshape((n, 1, 16) + a.shape[1:]),
                                                gate.reshape((n, 1, 16) + a.shape[1:])],
                                               1)).reshape(a.shape)


def _prepare_exec_attn(c, d, own):
    dev = _dev()
    dp = create_dispatchers(dev)
    B, H, S = c["B"], c["H"], c["S"]
    bh, n = B * H, B * H * S * 64
    q, k, v = (own.storage(d[x]) for x in "qkv")
    qh, kh, vh, kt, ob, y = (own.create(n * 4) for _ in range(6))
    sc, pr = own.create(bh * S * S * 4), own.create(bh * S * S * 4)
    one = own.storage(np.array([1.0 / math.sqrt(64.0)], np.float32))

    def transpose(src, dst, dims, perm):
        new = [dims[i] for i in perm]
        pad = [1] * (4 - len(dims))
        dp.transpose(src, dst, len(dims), new + pad, row_major_strides(dims) + [0] * len(pad),
                     list(perm) + [0] * len(pad), n)

    def go():
        transpose(q, qh, [B, S, H, 64], [0, 2, 1, 3])
        transpose(k, kh, [B, S, H, 64], [0, 2, 1, 3])
        transpose(v, vh, [B, S, H, 64], [0, 2, 1, 3])
        transpose(kh, kt, [bh, S, 64], [0, 2, 1])
        dp.matmul(qh, kt, sc, S, S, 64, bh, 1)
        dp.binary_bcast["Mul"](sc, one, pr, 3, [bh, S, S], [S * S, S, 1], [0, 0, 0], bh * S * S)
        dp.softmax(pr, sc, S, bh * S)
        dp.matmul(sc, vh, ob, S, 64, S, bh, 1)
        transpose(ob, y, [B, H, S, 64], [0, 2, 1, 3])
    return {"go": go, "out": Outputs(own, y=(y, np.float32, (B, S, H, 64)))}


def run(state):
    state["go"]()
    return state["out"]


# ------------------------------------------------------------------- work --
def _resnet_flops(cin, cout, hw):
    f = 18.0 * hw * cout * (cin + cout)
    return f + (2.0 * hw * cin * cout if cin != cout else 0.0)


def _transformer_flops(c, hw, s):
    return 40.0 * hw * c * c + 4.0 * hw * hw * c + 4.0 * hw * s * c + 4.0 * s * CONTEXT_DIM * c


def _unet_flops(H, W):
    ch = (320, 640, 1280, 1280)
    hw = [H * W // 4 ** i for i in range(4)]
    tf = lambda i: _transformer_flops(ch[i], hw[i], CONTEXT_TOKENS) if i < 3 else 0.0  # noqa: E731
    f = 18.0 * hw[0] * 4 * 320 * 2
    skips, prev = [320], 320
    for i in range(4):
        for _ in range(2):
            f += _resnet_flops(prev, ch[i], hw[i]) + tf(i)
            prev = ch[i]
            skips.append(prev)
        if i < 3:
            f += 18.0 * hw[i + 1] * prev * prev
            skips.append(prev)
    f += 2 * _resnet_flops(1280, 1280, hw[3]) + _transformer_flops(1280, hw[3], CONTEXT_TOKENS)
    for i in (3, 2, 1, 0):
        for _ in range(3):
            f += _resnet_flops(prev + skips.pop(), ch[i], hw[i]) + tf(i)
            prev = ch[i]
        if i:
            f += 18.0 * hw[i - 1] * prev * prev
    return f


def _vae_flops(H, W):
    hw = H * W
    f = 18.0 * hw * 4 * 512 + 2 * _resnet_flops(512, 512, hw) + 8.0 * hw * 512 * 512 + 4.0 * hw * hw * 512
    prev = 512
    for i, c in enumerate((512, 512, 256, 128)):
        for _ in range(3):
            f += _resnet_flops(prev, c, hw)
            prev = c
        if i < 3:
            hw *= 4
            f += 18.0 * hw * c * c
    return f + 18.0 * hw * 128 * 3


def work(case):
    """Operations, and bytes with each input and weight read once and each
    output written once (of every call, where the case is a chain of calls)."""
    c, k = case, case["kind"]
    if k == "gn":
        n = c["N"] * c["C"] * c["H"] * c["W"]
        return {"bytes": 2.0 * n * (2 if c["f16"] else 4) + 8 * c["C"], "flops": 10.0 * n}
    if k in ("conv32", "conv16"):
        ho, wo = _conv_out(c)
        es = 2 if k == "conv16" else 4
        nin, nout = c["N"] * c["Cin"] * c["H"] * c["W"], c["N"] * c["Cout"] * ho * wo
        kk = c["Cin"] * c["K"] * c["K"]
        return {"bytes": float(es * (nin + nout * (2 if c.get("res") else 1) + c["Cout"] * kk)),
                "flops": 2.0 * nout * kk}
    if k == "resnet":
        hw, ci, co = c["H"] * c["W"], c["Cin"], c["Cout"]
        wts = 9 * co * (ci + co) + co * TIME_DIM + (ci * co if ci != co else 0)
        return {"bytes": 2.0 * (c["B"] * hw * (ci + co) + wts),
                "flops": c["B"] * _resnet_flops(ci, co, hw) + 2.0 * c["B"] * co * TIME_DIM}
    if k == "transformer":
        hw, C = c["H"] * c["W"], c["C"]
        wts = 20 * C * C + 2 * C * CONTEXT_DIM
        return {"bytes": 2.0 * (2 * c["B"] * hw * C + wts + c["B"] * c["S"] * CONTEXT_DIM),
                "flops": c["B"] * _transformer_flops(C, hw, c["S"])}
    if k in ("attn", "cross"):
        sq, skv = c.get("Sq", c.get("S")), c.get("Skv", c.get("S"))
        es = 2 if c["f16"] else 4
        return {"bytes": 128.0 * es * c["B"] * c["H"] * (sq + skv),
                "flops": 256.0 * c["B"] * c["H"] * sq * skv}
    if k == "ffn":
        es, m = (2 if c["f16"] else 4), (3 if c["act"] == ACT_GEGLU else 2)
        return {"bytes": float(es * (2 * c["rows"] * c["D"] + m * c["D"] * c["F"])),
                "flops": 2.0 * m * c["rows"] * c["D"] * c["F"]}
    if k == "exec_attn":
        n, s = c["B"] * c["H"] * c["S"] * 64, c["B"] * c["H"] * c["S"] ** 2
        return {"bytes": 4.0 * (14 * n + 6 * s), "flops": 256.0 * s}
    if k == "unet":
        io = c["B"] * (8 * c["H"] * c["W"] + CONTEXT_TOKENS * CONTEXT_DIM)
        return {"bytes": 1.732e9 + 4.0 * io, "flops": c["B"] * _unet_flops(c["H"], c["W"])}
    px = c["B"] * c["H"] * c["W"]
    return {"bytes": 9.9e7 + 4.0 * px * (4 + 192), "flops": c["B"] * _vae_flops(c["H"], c["W"])}


def tolerance(case):
    """About four times what the library measures against ``exact`` over these
    ranges: fp32 sums 8e-7 (up to 1.9e-6 over the longest convolutions),
    GroupNorm 1e-7, one fp16 rounding of a result 2.1e-4, a block of fp16
    layers 3.3e-4 to 4.8e-4, attention 3.7e-4 to 5e-4, the decoder 1.2e-3, a
    denoise step 1.7e-3; the largest single differences 3.8e-7 (GroupNorm),
    1.5e-5 (fp32 sums) and 5e-4 to 8e-3 (fp16)."""
    k = case["kind"]
    if k == "conv32":
        return {"rel": 8e-6, "max": 8e-5}
    if k == "gn":
        return {"rel": 8e-4, "max": 2e-3} if case["f16"] else {"rel": 4e-7, "max": 2e-6}
    if k == "ffn":
        return {"rel": 1e-3, "max": 5e-3} if case["f16"] else {"rel": 4e-6, "max": 5e-5}
    if k == "exec_attn":
        return {"rel": 4e-6, "max": 4e-5}
    if k == "conv16":
        return {"rel": 8e-4, "max": 2e-3}
    if k in ("attn", "cross"):
        return {"rel": 2e-3, "max": 2e-2}
    if k == "unet":
        return {"rel": 7e-3, "max": 3e-2}
    if k == "vae":
        return {"rel": 5e-3, "max": 4e-2}
    return {"rel": 2e-3, "max": 1.2e-2}


# ------------------------------------------------------------------ exact --
def _t(a, half=False):
    """float64 on the device; ``half``: of the fp16 rounding, as stored."""
    a = np.asarray(a)
    if half:
        a = a.astype(np.float16)
    return torch.from_numpy(np.ascontiguousarray(a)).to("cuda").double()


def _silu(x):
    return x * torch.sigmoid(x)


def _gn(x, g, b, eps):
    return F.group_norm(x, GROUPS, g, b, eps)


def _conv64(x, w, b, stride=1):
    """3x3 / 1x1 convolution as a matrix product of the unfolded input."""
    o, i, k, _ = w.shape
    ho = (x.shape[2] + 2 * (k // 2) - k) // stride + 1
    wo = (x.shape[3] + 2 * (k // 2) - k) // stride + 1
    wm = w.reshape(o, i * k * k)
    y = torch.empty((x.shape[0], o, ho, wo), dtype=torch.float64, device=x.device)
    for n in range(x.shape[0]):
        cols = F.unfold(x[n:n + 1], k, padding=k // 2, stride=stride)[0]
        y[n] = (wm @ cols + b[:, None]).reshape(o, ho, wo)
    return y


def _attn64(q, k, v):
    """softmax(q k^T / sqrt(d)) v over [..., S, d], head by head."""
    lead, d = q.shape[:-2], q.shape[-1]
    q, k, v = (t.reshape((-1,) + t.shape[-2:]) for t in (q, k, v))
    o = torch.empty_like(q)
    for h in range(q.shape[0]):
        kt = (k[h].t() / math.sqrt(d)).contiguous()
        for i in range(0, q.shape[1], 4096):
            o[h, i:i + 4096] = torch.softmax(q[h, i:i + 4096] @ kt, -1) @ v[h]
    return o.reshape(lead + o.shape[-2:])


class _Weights:
    """Weights of a diffusers-named dict as float64 on the device."""

    def __init__(self, sd, half=True):
        self.sd, self.half = sd, half

    def __call__(self, name):
        a = self.sd[name]
        return _t(a, self.half and a.ndim > 1)

    def has(self, name):
        return name in self.sd

    def lin(self, p, x):
        y = x @ self(p + ".weight").t().contiguous()
        return y + self(p + ".bias") if self.has(p + ".bias") else y

    def conv(self, p, x, stride=1):
        return _conv64(x, self(p + ".weight"), self(p + ".bias"), stride)

    def gn(self, p, x, eps):
        return _gn(x, self(p + ".weight"), self(p + ".bias"), eps)


def _resnet64(w, p, x, temb, eps):
    h = w.conv(p + ".conv1", _silu(w.gn(p + ".norm1", x, eps)))
    if temb is not None:
        h = h + w.lin(p + ".time_emb_proj", _silu(temb))[:, :, None, None]
    h = w.conv(p + ".conv2", _silu(w.gn(p + ".norm2", h, eps)))
    if w.has(p + ".conv_shortcut.weight"):
        x = w.conv(p + ".conv_shortcut", x)
    return x + h


def _heads(t, n):
    return t.reshape(t.shape[0], t.shape[1], n, -1).transpose(1, 2)


def _transformer64(w, p, x, ctx):
    B, C, H, W = x.shape
    t = p + ".transformer_blocks.0"
    h = w.lin(p + ".proj_in", w.gn(p + ".norm", x, 1e-6).permute(0, 2, 3, 1).reshape(B, H * W, C))
    for i, kv in ((1, None), (2, ctx)):
        n = F.layer_norm(h, (C,), w(f"{t}.norm{i}.weight"), w(f"{t}.norm{i}.bias"), 1e-5)
        src, a = (n if kv is None else kv), f"{t}.attn{i}"
        o = _attn64(_heads(w.lin(a + ".to_q", n), C // 64), _heads(w.lin(a + ".to_k", src), C // 64),
                    _heads(w.lin(a + ".to_v", src), C // 64))
        h = h + w.lin(a + ".to_out.0", o.transpose(1, 2).reshape(B, H * W, C))
    n = F.layer_norm(h, (C,), w(f"{t}.norm3.weight"), w(f"{t}.norm3.bias"), 1e-5)
    hid, gate = w.lin(f"{t}.ff.net.0.proj", n).chunk(2, -1)
    h = h + w.lin(f"{t}.ff.net.2", hid * F.gelu(gate))
    h = w.lin(p + ".proj_out", h)
    return x + h.reshape(B, H, W, C).permute(0, 3, 1, 2)


def _up2(x):
    return F.interpolate(x, scale_factor=2.0, mode="nearest")


def _unet64(w, x, t, ctx):
    f = torch.exp(torch.arange(160, dtype=torch.float64, device="cuda") * (-math.log(1e4) / 160))
    a = t[:, None] * f[None]
    temb = w.lin("time_embedding.linear_2", _silu(w.lin(
        "time_embedding.linear_1", torch.cat([torch.cos(a), torch.sin(a)], 1))))
    h = w.conv("conv_in", x)
    skips = [h]
    for i in range(4):
        b = f"down_blocks.{i}"
        for j in range(2):
            h = _resnet64(w, f"{b}.resnets.{j}", h, temb, 1e-5)
            if i < 3:
                h = _transformer64(w, f"{b}.attentions.{j}", h, ctx)
            skips.append(h)
        if i < 3:
            h = w.conv(f"{b}.downsamplers.0.conv", h, 2)
            skips.append(h)
    h = _resnet64(w, "mid_block.resnets.0", h, temb, 1e-5)
    h = _transformer64(w, "mid_block.attentions.0", h, ctx)
    h = _resnet64(w, "mid_block.resnets.1", h, temb, 1e-5)
    for i in range(4):
        b = f"up_blocks.{i}"
        for j in range(3):
            h = _resnet64(w, f"{b}.resnets.{j}", torch.cat([h, skips.pop()], 1), temb, 1e-5)
            if i > 0:
                h = _transformer64(w, f"{b}.attentions.{j}", h, ctx)
        if i < 3:
            h = w.conv(f"{b}.upsamplers.0.conv", _up2(h))
    return w.conv("conv_out", _silu(w.gn("conv_norm_out", h, 1e-5)))


def _vae64(w, z):
    h = w.conv("decoder.conv_in", _conv64(z, w("post_quant_conv.weight"), w("post_quant_conv.bias")))
    m = "decoder.mid_block"
    h = _resnet64(w, m + ".resnets.0", h, None, 1e-6)
    B, C, H, W = h.shape
    a = m + ".attentions.0"
    t = w.gn(a + ".group_norm", h, 1e-6).permute(0, 2, 3, 1).reshape(B, H * W, C)
    o = w.lin(a + ".to_out.0", _attn64(w.lin(a + ".to_q", t), w.lin(a + ".to_k", t),
                                       w.lin(a + ".to_v", t)))
    h = h + o.reshape(B, H, W, C).permute(0, 3, 1, 2)
    h = _resnet64(w, m + ".resnets.1", h, None, 1e-6)
    for i in range(4):
        for j in range(3):
            h = _resnet64(w, f"decoder.up_blocks.{i}.resnets.{j}", h, None, 1e-6)
        if i < 3:
            h = w.conv(f"decoder.up_blocks.{i}.upsamplers.0.conv", _up2(h))
    return w.conv("decoder.conv_out", _silu(w.gn("decoder.conv_norm_out", h, 1e-6)))


def exact(case, seed):
    c, k = case, case["kind"]
    d = _inputs(c, seed)
    last = lambda t: t.permute(0, 2, 3, 1).contiguous()  # noqa: E731
    if k == "gn":
        y = _gn(_t(d["x"], c["f16"]), _t(d["g"]), _t(d["b"]), 1e-5)
        y = _silu(y) if c["silu"] else y
        return {"y": last(y) if c["f16"] else y}
    if k in ("conv32", "conv16"):
        f16 = k == "conv16"
        x = _t(d["x"], f16)
        y = _conv64(_up2(x) if c.get("up") == 2 else x, _t(d["c.weight"], f16), _t(d["c.bias"]),
                    c["S"])
        y = _silu(y) if c.get("silu") else y
        y = y + _t(d["r"]) if "r" in d else y
        return {"y": last(y) if f16 else y}
    if k == "resnet":
        return {"y": last(_resnet64(_Weights(d), "p", _t(d["x"], True), _t(d["temb"]), 1e-5))}
    if k == "transformer":
        return {"y": last(_transformer64(_Weights(d), "p", _t(d["x"], True), _t(d["ctx"], True)))}
    if k in ("attn", "cross", "exec_attn"):
        q, kk, v = (_t(d[n], c.get("f16", False)) for n in "qkv")
        if c.get("bhsd"):
            return {"y": _attn64(q, kk, v)}
        return {"y": _attn64(*(t.transpose(1, 2) for t in (q, kk, v))).transpose(1, 2).contiguous()}
    if k == "ffn":
        x, w1, w2 = (_t(d[n], c["f16"]) for n in ("x", "w1", "w2"))
        h = x @ w1.t().contiguous() + _t(d["b1"])
        if c["act"] == ACT_GEGLU:
            hid, gate = h.chunk(2, -1)
            h = hid * F.gelu(gate)
        else:
            h = F.gelu(h, approximate="tanh" if c["act"] == ACT_GELU_TANH else "none")
        return {"y": h @ w2.t().contiguous() + _t(d["b2"]) + x}
    if k == "unet":
        w = _Weights(_unet().state_dict(np.float16), half=False)
        for p in _unet().params:  # fp32 parameters whole
            if p["dtype"] == np.float32 and p["layout"] == 0:
                w.sd[p["name"]] = _unet().download_param(p)
        return {"y": _unet64(w, _t(d["x"]), _t(d["t"]), _t(d["ctx"]))}
    w = _Weights(_vae().state_dict(), half=False)
    return {"y": _vae64(w, _t(d["x"]) * VAE_SCALE)}
