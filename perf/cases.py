"""The work that programs on this framework have it do: single ops, the blocks of the
networks (3-D UNet, VQ decoder) and one whole sampling run, each through the public entry
point a program calls, over the range of sizes and types that it is used at.

``listed()`` names twelve of them; ``draw`` gives others of the same ranges. Tensors are
channels-last NDHWC unless said otherwise, activations ~N(0, 1), conv and dense weights
~N(0, 1 / fan_in), norm weights near 1: what normalised networks meet.
"""

from __future__ import annotations

import importlib
import math

import numpy as np
import torch

_PKG = "lesiondiffusion-mlx_amd"
_DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}
_BYTES = {"fp16": 2, "bf16": 2, "fp32": 4}

# The largest listed case's FLOPs; a drawn case stays below it.
_MOST_FLOPS = 3.2e12


def _pkg():
    return importlib.import_module(_PKG)


def listed() -> list[dict]:
    return [
        # A UNet level's tokens against 77 projected text tokens: the smallest call of a
        # denoise step, where the launch and the host path count.
        {"name": "cross_attention", "kind": "attention", "dtype": "fp16", "b": 1, "heads": 8, "d": 64, "lq": 1600,
         "lk": 77},
        # The spatial transformer of the 256-channel level (8 x 10 x 10) of the conditioned
        # UNet: norms, thirteen small dense layers, self and cross attention.
        {"name": "transformer", "kind": "transformer", "b": 1, "c": 256, "head": 32, "grid": "8x10x10", "text": 77},
        # One 64 -> 64 conv of a 32 x 40 x 40 latent, no norm: the op-level conv call.
        {"name": "conv_64", "kind": "conv", "dtype": "fp16", "b": 1, "grid": "32x40x40", "c": 64, "o": 64,
         "stride": 1, "up": False},
        # A decoder's nearest-2x upsampling conv on an odd grid, in bf16.
        {"name": "upsample_bf16", "kind": "conv", "dtype": "bf16", "b": 1, "grid": "19x21x37", "c": 128, "o": 128,
         "stride": 1, "up": True},
        # The decoder ResBlock of the finest UNet level: concatenated skip, time shift, 1x1
        # skip projection.
        {"name": "unet_resblock", "kind": "resblock", "dtype": "fp16", "b": 1, "grid": "32x40x40", "c": 128,
         "c1": 64, "o": 64},
        # The finest level of the FP32 mask network (model width 16, 76 x 128 x 152, which
        # is 23,104 tokens two levels down).
        {"name": "resblock_fp32", "kind": "resblock", "dtype": "fp32", "b": 1, "grid": "76x128x152", "c": 16,
         "c1": 0, "o": 16},
        # That network's self attention: two 32-wide heads over 23,104 tokens, FP32.
        {"name": "attention_fp32", "kind": "attention", "dtype": "fp32", "b": 1, "heads": 2, "d": 32, "lq": 23104,
         "lk": 23104},
        # Self attention of the inpainting network's attention level (512 channels as
        # 32-wide heads, 20 x 20 x 16 tokens).
        {"name": "self_attention", "kind": "attention", "dtype": "fp16", "b": 1, "heads": 16, "d": 32, "lq": 6400,
         "lk": 6400},
        # The VQ decoder's 96-channel ResBlock at full resolution (128 x 160 x 160): the
        # largest tensors of the path.
        {"name": "vq_resblock", "kind": "vq_resblock", "dtype": "fp16", "b": 1, "grid": "128x160x160", "c": 96,
         "o": 96},
        # Nearest-codebook search of a whole 64 x 80 x 80 latent before the decode.
        {"name": "quantize", "kind": "quantize", "dtype": "fp32", "positions": 409600, "entries": 8192},
        # GroupNorm, SiLU and conv in the source-order arithmetic (NCDHW fp16), bit for bit.
        {"name": "source_conv", "kind": "source", "b": 1, "grid": "32x40x40", "c": 64, "o": 64, "k": 3, "stride": 1},
        # Masked DDIM sampling with the conditioned UNet, one captured graph per step: what
        # a sampling program repeats 200 times.
        {"name": "ddim", "kind": "ddim", "width": 64, "grid": "32x40x40", "steps": 2},
    ]


# ------------------------------------------------------------------ drawn cases

def _log(rng, lo: float, hi: float) -> int:
    return max(int(lo), min(int(hi), round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _grid(rng, voxels: float) -> str:
    """A box of about ``voxels`` voxels with unequal, often odd sides."""
    side = voxels ** (1.0 / 3.0)
    a, b = side * rng.uniform(0.6, 1.5), side * rng.uniform(0.6, 1.5)
    return "x".join(str(max(2, round(n))) for n in (a, b, voxels / (a * b)))


def _sides(case: dict) -> list[int]:
    return [int(n) for n in case["grid"].split("x")]


def _drawn(rng) -> dict:
    kind = rng.choice(["self", "self", "cross", "attention_fp32", "transformer", "conv", "conv", "resblock", "resblock",
                       "resblock_fp32", "resblock_fp32", "vq_resblock", "quantize", "source", "ddim"])
    if kind == "self":
        d = rng.choice([32, 32, 64, 64, 128, 256])
        n = _log(rng, 100, 51200)
        return {"kind": "attention", "dtype": rng.choice(["fp16", "fp16", "bf16"]), "b": rng.choice([1, 1, 2]),
                "heads": 1 if d == 256 else rng.choice([2, 4, 8, 16]), "d": d, "lq": n, "lk": n}
    if kind == "cross":
        return {"kind": "attention", "dtype": "fp16", "b": rng.choice([1, 1, 2]), "heads": rng.choice([4, 8, 16]),
                "d": rng.choice([32, 64]), "lq": _log(rng, 100, 6400), "lk": rng.choice([5, 33, 77, 77, 128])}
    if kind == "attention_fp32":
        n = _log(rng, 300, 24000)
        return {"kind": "attention", "dtype": "fp32", "b": 1, "heads": rng.choice([1, 2, 4]), "d": rng.choice([32, 32, 64]),
                "lq": n, "lk": n}
    if kind == "transformer":
        return {"kind": "transformer", "b": 1, "c": rng.choice([64, 128, 256, 512]), "head": 32,
                "grid": _grid(rng, _log(rng, 100, 6400)), "text": rng.choice([0, 77, 77])}
    if kind == "conv":
        c = rng.choice([32, 64, 96, 128, 256])
        return {"kind": "conv", "dtype": rng.choice(["fp16", "fp16", "bf16"]), "b": rng.choice([1, 1, 2]),
                "grid": _grid(rng, _log(rng, 200, 200000)), "c": c, "o": rng.choice([c, c, 32, 64, 128]),
                **rng.choice([{"stride": 1, "up": False}, {"stride": 2, "up": False}, {"stride": 1, "up": True}])}
    if kind == "resblock":
        c = rng.choice([64, 128, 256, 512])
        skip = rng.choice([0, c // 2, c])
        return {"kind": "resblock", "dtype": "fp16", "b": rng.choice([1, 1, 2]),
                "grid": _grid(rng, _log(rng, 100, 400000 * 64 / c)), "c": c, "c1": skip,
                "o": c if skip == 0 else rng.choice([c, c // 2])}
    if kind == "resblock_fp32":
        c, most = rng.choice([(16, 1500000), (32, 190000), (64, 24000), (64, 24000)])
        skip = rng.choice([0, c])
        return {"kind": "resblock", "dtype": "fp32", "b": 1, "grid": _grid(rng, _log(rng, most / 30, most)), "c": c,
                "c1": skip, "o": c}
    if kind == "vq_resblock":
        c = rng.choice([32, 64, 96, 128, 192])
        return {"kind": "vq_resblock", "dtype": rng.choice(["fp16", "fp16", "fp32"]), "b": 1,
                "grid": _grid(rng, _log(rng, 30000, 1000000)), "c": c, "o": rng.choice([c, c, c // 2])}
    if kind == "quantize":
        return {"kind": "quantize", "dtype": rng.choice(["fp32", "fp16"]), "positions": _log(rng, 500, 409600),
                "entries": _log(rng, 256, 8192)}
    if kind == "source":
        c = rng.choice([32, 64, 96, 128])
        return {"kind": "source", "b": 1, "grid": _grid(rng, _log(rng, 1000, 60000)), "c": c, "o": rng.choice([c, 32, 64]),
                "k": rng.choice([1, 3, 3]), "stride": rng.choice([1, 1, 2])}
    return {"kind": "ddim", "width": rng.choice([32, 64]), "grid": "x".join(str(8 * rng.choice([2, 3, 4, 5])) for _ in range(3)),
            "steps": rng.choice([1, 2, 2])}


def draw(rng) -> dict:
    while True:
        case = _drawn(rng)
        f = work(case)["flops"]
        # fp32 products cost three on the matrix units, the source order runs on the VALU and
        # the search costs some twenty operations per code: each kind stays below its listed
        # case's size, all below the largest case.
        if f * (4 if case.get("dtype") == "fp32" and case["kind"] != "quantize" else 1) <= _MOST_FLOPS:
            return case


# ------------------------------------------------------------------ inputs

class _Make:
    """Seeded device tensors."""

    def __init__(self, seed: int):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)

    def n(self, *shape, dtype=torch.float32, scale=1.0) -> torch.Tensor:
        return (torch.randn(shape, generator=self.g, device="cuda") * scale).to(dtype)

    def conv(self, w: dict, key: str, ci: int, co: int, k: int, dtype) -> None:
        w[key + ".weight"] = self.n(co, ci, k, k, k, dtype=dtype, scale=(ci * k ** 3) ** -0.5)
        w[key + ".bias"] = self.n(co, dtype=dtype, scale=0.01)

    def lin(self, w: dict, key: str, ci: int, co: int, dtype, bias=True) -> None:
        w[key + ".weight"] = self.n(co, ci, dtype=dtype, scale=ci ** -0.5)
        if bias:
            w[key + ".bias"] = self.n(co, dtype=dtype, scale=0.01)

    def norm(self, w: dict, key: str, c: int, dtype) -> None:
        w[key + ".weight"] = (1 + self.n(c, scale=0.1)).to(dtype)
        w[key + ".bias"] = self.n(c, dtype=dtype, scale=0.1)


def _resblock_weights(m: _Make, key: str, ci: int, co: int, dtype, temb: int | None) -> dict:
    w: dict = {}
    m.norm(w, key + ".in_layers.0", ci, dtype)
    m.conv(w, key + ".in_layers.2", ci, co, 3, dtype)
    if temb:
        m.lin(w, key + ".emb_layers.1", temb, co, dtype)
    m.norm(w, key + ".out_layers.0", co, dtype)
    m.conv(w, key + ".out_layers.3", co, co, 3, dtype)
    if ci != co:
        m.conv(w, key + ".skip_connection", ci, co, 1, dtype)
    return w


def _transformer_weights(m: _Make, key: str, c: int, context: int | None, dtype) -> dict:
    w: dict = {}
    m.norm(w, key + ".norm", c, dtype)
    m.conv(w, key + ".proj_in", c, c, 1, dtype)
    m.conv(w, key + ".proj_out", c, c, 1, dtype)
    blk = key + ".transformer_blocks.0"
    for n in ("norm1", "norm2", "norm3"):
        m.norm(w, f"{blk}.{n}", c, dtype)
    for a in ("attn1", "attn2"):
        kd = c if (a == "attn1" or context is None) else context
        for n, ci in (("to_q", c), ("to_k", kd), ("to_v", kd)):
            m.lin(w, f"{blk}.{a}.{n}", ci, c, dtype, bias=False)
        m.lin(w, f"{blk}.{a}.to_out.0", c, c, dtype)
    m.lin(w, blk + ".ff.net.0.0", c, 4 * c, dtype)
    m.lin(w, blk + ".ff.net.2", 4 * c, c, dtype)
    return w


def _alphas() -> np.ndarray:
    """The linear latent-diffusion schedule, stored in half precision as checkpoints do."""
    betas = np.linspace(0.0015 ** 0.5, 0.0195 ** 0.5, 1000, dtype=np.float64) ** 2
    return np.cumprod(1.0 - betas).astype(np.float16)


def _inputs(case: dict, seed: int) -> dict:
    """Seeded inputs and weights, before anything of the framework is made of them."""
    m, kind = _Make(seed), case["kind"]
    dt = _DTYPES[case.get("dtype", "fp16")]
    if kind == "attention":
        f = case["heads"] * case["d"]
        if case["lq"] == case["lk"]:   # one projection's columns, as a fused q/k/v layer leaves them
            qkv = m.n(case["b"], case["lq"], 3 * f, dtype=dt)
            return {"q": qkv[..., :f], "k": qkv[..., f:2 * f], "v": qkv[..., 2 * f:]}
        kv = m.n(case["b"], case["lk"], 2 * f, dtype=dt)
        return {"q": m.n(case["b"], case["lq"], f, dtype=dt), "k": kv[..., :f], "v": kv[..., f:]}
    if kind == "transformer":
        return {"x": m.n(case["b"], *_sides(case), case["c"], dtype=dt),
                "text": m.n(case["b"], case["text"], 768, dtype=dt) if case["text"] else None,
                "w": {**_transformer_weights(m, "t", case["c"], 768 if case["text"] else None, dt),
                      **({"context_linear_projection.weight": m.n(768, 768, dtype=dt, scale=768 ** -0.5)}
                         if case["text"] else {})}}
    if kind == "conv":
        w: dict = {}
        m.conv(w, "c", case["c"], case["o"], 3, dt)
        return {"x": m.n(case["b"], *_sides(case), case["c"], dtype=dt), "w": w["c.weight"], "bias": w["c.bias"].float()}
    if kind == "resblock":
        x1 = m.n(case["b"], *_sides(case), case["c1"], dtype=dt) if case["c1"] else None
        return {"x": m.n(case["b"], *_sides(case), case["c"], dtype=dt), "x1": x1,
                "shift": m.n(case["b"], case["o"], dtype=dt, scale=0.3),
                "w": _resblock_weights(m, "r", case["c"] + case["c1"], case["o"], dt, 64)}
    if kind == "vq_resblock":
        w = {}
        m.norm(w, "r.norm1", case["c"], dt)
        m.conv(w, "r.conv1", case["c"], case["o"], 3, dt)
        m.norm(w, "r.norm2", case["o"], dt)
        m.conv(w, "r.conv2", case["o"], case["o"], 3, dt)
        if case["c"] != case["o"]:
            m.conv(w, "r.nin_shortcut", case["c"], case["o"], 1, dt)
        return {"x": m.n(case["b"], *_sides(case), case["c"], dtype=dt), "w": w}
    if kind == "quantize":
        cb = m.n(case["entries"], 4, dtype=dt)
        return {"z": m.n(case["positions"], 4, dtype=dt), "codebook": cb}
    if kind == "source":
        w = {}
        m.conv(w, "c", case["c"], case["o"], case["k"], dt)
        m.norm(w, "n", case["c"], dt)
        return {"x": m.n(case["b"], case["c"], *_sides(case), dtype=dt), "w": w}
    # ddim
    wd, mult, temb = case["width"], (1, 2, 4, 4), 4 * case["width"]
    w = {}
    m.lin(w, "time_embed.0", wd, temb, dt)
    m.lin(w, "time_embed.2", temb, temb, dt)
    w["context_linear_projection.weight"] = m.n(768, 768, dtype=dt, scale=768 ** -0.5)
    m.conv(w, "input_blocks.0.0", 9, wd, 3, dt)
    chans, ch, block, res = [wd], wd, 1, 1
    for level, k in enumerate(mult):
        for _ in range(2):
            w.update(_resblock_weights(m, f"input_blocks.{block}.0", ch, k * wd, dt, temb))
            ch = k * wd
            if res in (4, 8):
                w.update(_transformer_weights(m, f"input_blocks.{block}.1", ch, 768, dt))
            chans.append(ch)
            block += 1
        if level < 3:
            m.conv(w, f"input_blocks.{block}.0.op", ch, ch, 3, dt)
            chans.append(ch)
            block, res = block + 1, res * 2
    w.update(_resblock_weights(m, "middle_block.0", ch, ch, dt, temb))
    w.update(_transformer_weights(m, "middle_block.1", ch, 768, dt))
    w.update(_resblock_weights(m, "middle_block.2", ch, ch, dt, temb))
    block = 0
    for level in (3, 2, 1, 0):
        for i in range(3):
            w.update(_resblock_weights(m, f"output_blocks.{block}.0", ch + chans.pop(), mult[level] * wd, dt, temb))
            ch = mult[level] * wd
            if res in (4, 8):
                w.update(_transformer_weights(m, f"output_blocks.{block}.1", ch, 768, dt))
            if level and i == 2:
                m.conv(w, f"output_blocks.{block}.{2 if res in (4, 8) else 1}.conv", ch, ch, 3, dt)
                res //= 2
            block += 1
    m.norm(w, "out.0", ch, dt)
    m.conv(w, "out.2", ch, 4, 3, dt)
    d, h, wv = _sides(case)
    mask = torch.zeros((1, d, h, wv), device="cuda")
    mask[:, d // 4:d - d // 4, h // 4:h - h // 4, wv // 4:wv - wv // 4] = 1.0
    return {"w": w, "text": m.n(1, 77, 768, dtype=dt), "mask": mask, "cond": m.n(1, d, h, wv, 4),
            "init": m.n(1, d, h, wv, 4), "noise": m.n(case["steps"], 1, d, h, wv, 4)}


# ------------------------------------------------------------------ one pass

def prepare(case: dict, seed: int) -> dict:
    pkg, kind, i = _pkg(), case["kind"], _inputs(case, seed)
    dt = _DTYPES[case.get("dtype", "fp16")]
    if kind == "attention":
        return {**i, "kind": kind, "heads": case["heads"], "scale": case["d"] ** -0.5, "ops": pkg.ops}
    if kind == "transformer":
        cfg = pkg.unet.UnetConfig(case["c"], 1, (1,), (1,), case["head"], skip_context=not case["text"])
        net = pkg.unet.LdmUnet(i["w"], cfg)
        return {"kind": kind, "net": net, "x": i["x"], "kv": net.project_context(i["text"])}
    if kind == "conv":
        pack = pkg.ops.pack_upsample_weight if case["up"] else pkg.ops.pack_weight
        return {"kind": kind, "ops": pkg.ops, "x": i["x"], "packed": pack(i["w"]), "bias": i["bias"],
                "stride": case["stride"], "up": case["up"]}
    if kind == "resblock":
        net = pkg.unet.LdmUnet(i["w"], pkg.unet.UnetConfig(case["o"], 1, ()), dtype=dt)
        return {"kind": kind, "net": net, "x": i["x"], "x1": i["x1"], "shift": i["shift"]}
    if kind == "vq_resblock":
        return {"kind": kind, "net": pkg.vq.VqDecoder(i["w"], dtype=dt), "x": i["x"]}
    if kind == "quantize":
        return {"kind": kind, "ops": pkg.ops, "z": i["z"], "codebook": i["codebook"],
                "norms": pkg.ops.squared_norms4(i["codebook"])}
    if kind == "source":
        return {"kind": kind, "ops": pkg.ops, "x": i["x"], "w": i["w"], "groups": pkg.layers.groups_for(case["c"]),
                "stride": case["stride"], "padding": case["k"] // 2}
    net = pkg.unet.LdmUnet(i["w"], pkg.unet.UnetConfig(case["width"], 2, (4, 8), (1, 2, 4, 4)))
    denoise = net.prepare_denoiser(i["text"])
    out: dict = {}

    def denoiser(x, t):
        out["eps"] = denoise(x, t)
        return out["eps"]

    sampler = pkg.sampling.DdimSampler(_alphas(), case["steps"])
    sample = sampler.prepare(denoiser, i["cond"], i["mask"], masked_conditioning=True)
    sample.set_noise(i["init"], i["noise"])
    sample.capture()
    return {"kind": kind, "sample": sample, "out": out, "init": i["init"], "noise": i["noise"]}


def run(s: dict):
    kind = s["kind"]
    if kind == "attention":
        return s["ops"].flash_attention(s["q"], s["k"], s["v"], heads=s["heads"], scale=s["scale"])
    if kind == "transformer":
        return s["net"].transformer(s["x"], s["kv"], "t")
    if kind == "conv":
        return s["ops"].nax_conv3d(s["x"], s["packed"], s["bias"], stride=s["stride"], upsample=s["up"])
    if kind == "resblock":
        return s["net"].residual(s["x"], s["shift"], "r", x1=s["x1"])
    if kind == "vq_resblock":
        return s["net"].residual(s["x"], "r")
    if kind == "quantize":
        out = torch.empty_like(s["z"])
        return s["ops"].nearest_codebook4(s["z"], s["codebook"], s["norms"], quantized=out), out
    if kind == "source":
        o, w = s["ops"], s["w"]
        y = o.group_norm_half(s["x"], w["n.weight"], w["n.bias"], groups=s["groups"], eps=1e-5)
        return y, o.conv3d_half(o.silu(y), w["c.weight"], w["c.bias"], padding=s["padding"], stride=s["stride"])
    s["sample"].set_noise(s["init"], s["noise"])
    return s["sample"].run(), s["out"]["eps"]


# ------------------------------------------------------------------ work and tolerance

def _conv_work(b, grid, c, o, k, es, stride=1, up=False) -> tuple[float, float]:
    vin = b * math.prod(grid)
    vout = b * math.prod(2 * n if up else (n - 1) // stride + 1 for n in grid)
    taps = 8 if up else k ** 3      # a folded upsampling conv needs 8 taps
    return float(es * (vin * c + vout * o + c * o * k ** 3)), 2.0 * vout * c * o * taps


def _resblock_work(b, grid, ci, o, es) -> tuple[float, float]:
    v = b * math.prod(grid)
    f = 2.0 * v * 27 * (ci * o + o * o) + (2.0 * v * ci * o if ci != o else 0.0)
    return float(es * (v * (ci + o) + 27 * (ci * o + o * o))), f


def _transformer_work(b, n, c, text) -> tuple[float, float]:
    f = 2.0 * b * n * c * c * (2 + 4 + 2 + 8 + (0 if text else 2)) + 4.0 * b * n * n * c + 4.0 * b * n * (text or n) * c
    return float(2 * (2 * b * n * c + c * c * (16 + (0 if text else 2)) + 2 * b * text * c)), f


def work(case: dict) -> dict:
    kind, es = case["kind"], _BYTES[case.get("dtype", "fp16")]
    if kind == "attention":
        f = case["heads"] * case["d"]
        by = float(es * case["b"] * f * (2 * case["lq"] + 2 * case["lk"]))
        return {"bytes": by, "flops": 4.0 * case["b"] * f * case["lq"] * case["lk"]}
    if kind == "transformer":
        by, fl = _transformer_work(case["b"], math.prod(_sides(case)), case["c"], case["text"])
    elif kind == "conv":
        by, fl = _conv_work(case["b"], _sides(case), case["c"], case["o"], 3, es, case["stride"], case["up"])
    elif kind == "resblock":
        by, fl = _resblock_work(case["b"], _sides(case), case["c"] + case["c1"], case["o"], es)
    elif kind == "vq_resblock":
        by, fl = _resblock_work(case["b"], _sides(case), case["c"], case["o"], es)
    elif kind == "quantize":
        p, e = case["positions"], case["entries"]
        by, fl = float(p * (8 * es + 4) + e * 5 * es), 11.0 * p * e
    elif kind == "source":
        by, fl = _conv_work(case["b"], _sides(case), case["c"], case["o"], case["k"], 2, case["stride"])
        by += 2.0 * case["b"] * case["c"] * math.prod(_sides(case))
    else:
        wd, mult = case["width"], (1, 2, 4, 4)
        by = fl = 0.0
        chans, ch, block, n = [wd], wd, 1, _sides(case)
        fl += 2.0 * math.prod(n) * 27 * 9 * wd
        for level, k in enumerate(mult):
            for _ in range(2):
                r, f = _resblock_work(1, n, ch, k * wd, 2)
                ch, fl = k * wd, fl + f
                if level >= 2:
                    fl += _transformer_work(1, math.prod(n), ch, 77)[1]
                chans.append(ch)
            if level < 3:
                fl += _conv_work(1, n, ch, ch, 3, 2, 2)[1]
                n = [v // 2 for v in n]
                chans.append(ch)
        fl += 2 * _resblock_work(1, n, ch, ch, 2)[1] + _transformer_work(1, math.prod(n), ch, 77)[1]
        for level in (3, 2, 1, 0):
            for i in range(3):
                fl += _resblock_work(1, n, ch + chans.pop(), mult[level] * wd, 2)[1]
                ch = mult[level] * wd
                if level >= 2:
                    fl += _transformer_work(1, math.prod(n), ch, 77)[1]
            if level:
                fl += _conv_work(1, n, ch, ch, 3, 2, 1, True)[1]
                n = [2 * v for v in n]
        fl += 2.0 * math.prod(n) * 27 * 4 * ch
        v = math.prod(_sides(case))
        # The weights (about 4,900 width^2 values, the text projections among them) and the
        # latent, conditioning, mask and noise, once per step.
        by = 2.0 * 4900 * wd * wd + v * 4.0 * (4 + 4 + 1 + 4 + 4)
        return {"bytes": by * case["steps"], "flops": fl * case["steps"]}
    return {"bytes": by, "flops": fl}


def tolerance(case: dict):
    """About four times the error against 64 bits that the path was measured at (fp16 ops
    2.1e-4 to 2.9e-4, blocks up to 4.6e-4, bf16 2.4e-3, FP32 1.6e-7 and 1.0e-6 with
    attention, two sampling steps 1.2e-3)."""
    kind = case["kind"]
    if kind in ("quantize", "source"):
        return "exact"      # the entry points promise the reference's values bit for bit
    if kind == "ddim":
        return {"rel": 5e-3}
    if kind == "transformer":
        return {"rel": 2e-3}
    if kind in ("attention", "conv"):
        return {"rel": {"fp16": 1e-3, "bf16": 1e-2, "fp32": 4e-6}[case["dtype"]]}
    return {"rel": {"fp16": 1.5e-3, "fp32": 2e-6}[case["dtype"]]}


# ------------------------------------------------------------------ the same in 64 bits

def _conv64(x, w, bias=None, stride=1):
    """Zero-padded conv of NDHWC ``x`` as one matrix product per tap."""
    o, c, k = w.shape[0], w.shape[1], w.shape[2]
    w = w.double()
    b, d, h, wd, _ = x.shape
    p = k // 2
    xp = torch.nn.functional.pad(x.double(), (0, 0, p, p, p, p, p, p))
    ext = [(n - 1) // stride + 1 for n in (d, h, wd)]
    y = torch.zeros((b * math.prod(ext), o), dtype=torch.float64, device=x.device)
    for kd in range(k):
        for kh in range(k):
            for kw in range(k):
                tap = xp[:, kd:kd + stride * (ext[0] - 1) + 1:stride, kh:kh + stride * (ext[1] - 1) + 1:stride,
                         kw:kw + stride * (ext[2] - 1) + 1:stride]
                y.addmm_(tap.reshape(-1, c), w[:, :, kd, kh, kw].t().contiguous())
    if bias is not None:
        y += bias.double()
    return y.view(b, *ext, o)


def _gn64(x, gamma, beta, groups, eps):
    x = x.double()
    b, c = x.shape[0], x.shape[-1]
    g = x.reshape(b, -1, groups, c // groups)
    mean = g.mean((1, 3), keepdim=True)
    var = (g - mean).square().mean((1, 3), keepdim=True)
    return (((g - mean) * (var + eps).rsqrt()).reshape(b, -1, c) * gamma.double() + beta.double()).view(x.shape)


def _ln64(x, gamma, beta):
    return torch.nn.functional.layer_norm(x.double(), (x.shape[-1],), gamma.double(), beta.double(), 1e-5)


def _silu64(x):
    return x * torch.sigmoid(x)


def _attention64(q, k, v, heads):
    """(B, L, heads * d) attention, a head and a run of query rows at a time."""
    b, lq, f = q.shape
    d = f // heads
    out = torch.empty((b, lq, f), dtype=torch.float64, device=q.device)
    rows = max(1, int(2e8) // k.shape[1])
    for i in range(b):
        for h in range(heads):
            s = slice(h * d, (h + 1) * d)
            kt, vv = k[i, :, s].double().t().contiguous(), v[i, :, s].double().contiguous()
            for r in range(0, lq, rows):
                a = torch.softmax(q[i, r:r + rows, s].double() @ kt * d ** -0.5, -1)
                out[i, r:r + rows, s] = a @ vv
    return out


def _groups(c):
    return 32 if c % 32 == 0 else c


def _resblock64(w, key, x, shift, x1=None):
    xx = x.double() if x1 is None else torch.cat([x.double(), x1.double()], -1)
    norm = lambda t, n: _silu64(_gn64(t, w[f"{key}.{n}.weight"], w[f"{key}.{n}.bias"], _groups(t.shape[-1]), 1e-5))  # noqa: E731
    conv = lambda t, n: _conv64(t, w[f"{key}.{n}.weight"], w[f"{key}.{n}.bias"])  # noqa: E731
    h = conv(norm(xx, "in_layers.0"), "in_layers.2") + shift.double()[:, None, None, None, :]
    h = conv(norm(h, "out_layers.0"), "out_layers.3")
    return h + (conv(xx, "skip_connection") if f"{key}.skip_connection.weight" in w else xx)


def _transformer64(w, key, x, ctx, head):
    """``ctx``: the projected text tokens, or None for attention to the block's own tokens."""
    b, c = x.shape[0], x.shape[-1]
    lin = lambda t, n: t.double() @ w[n + ".weight"].double().t() + w[n + ".bias"].double()  # noqa: E731
    g = _gn64(x, w[key + ".norm.weight"], w[key + ".norm.bias"], 32, 1e-6)
    t = _conv64(g, w[key + ".proj_in.weight"], w[key + ".proj_in.bias"]).view(b, -1, c)
    blk = key + ".transformer_blocks.0"
    for a, n in (("attn1", "norm1"), ("attn2", "norm2")):
        s = _ln64(t, w[f"{blk}.{n}.weight"], w[f"{blk}.{n}.bias"])
        src = s if a == "attn1" or ctx is None else ctx
        q, k, v = (y @ w[f"{blk}.{a}.{p}.weight"].double().t() for y, p in ((s, "to_q"), (src, "to_k"), (src, "to_v")))
        t = t + lin(_attention64(q, k, v, c // head), f"{blk}.{a}.to_out.0")
    s = _ln64(t, w[blk + ".norm3.weight"], w[blk + ".norm3.bias"])
    t = t + lin(torch.nn.functional.gelu(lin(s, blk + ".ff.net.0.0")), blk + ".ff.net.2")
    return x.double() + _conv64(t.view(x.shape), w[key + ".proj_out.weight"], w[key + ".proj_out.bias"])


def _up64(x):
    for axis in (1, 2, 3):
        x = x.repeat_interleave(2, axis)
    return x


def _unet64(w, wd, x, t, ctx):
    lin = lambda y, n: y @ w[n + ".weight"].double().t() + w[n + ".bias"].double()  # noqa: E731
    conv = lambda y, n, s=1: _conv64(y, w[n + ".weight"], w[n + ".bias"], s)  # noqa: E731
    f = torch.exp(-math.log(1e4) * torch.arange(wd // 2, device="cuda", dtype=torch.float64) / (wd // 2)) * t
    emb = _silu64(lin(_silu64(lin(torch.cat([f.cos(), f.sin()])[None], "time_embed.0")), "time_embed.2"))
    shift = lambda key: lin(emb, key + ".emb_layers.1")  # noqa: E731
    x = conv(x, "input_blocks.0.0")
    skips, block, res = [x], 1, 1
    for level in range(4):
        for _ in range(2):
            key = f"input_blocks.{block}"
            x = _resblock64(w, key + ".0", x, shift(key + ".0"))
            if res in (4, 8):
                x = _transformer64(w, key + ".1", x, ctx, 32)
            skips.append(x)
            block += 1
        if level < 3:
            x = conv(x, f"input_blocks.{block}.0.op", 2)
            skips.append(x)
            block, res = block + 1, res * 2
    x = _resblock64(w, "middle_block.0", x, shift("middle_block.0"))
    x = _transformer64(w, "middle_block.1", x, ctx, 32)
    x = _resblock64(w, "middle_block.2", x, shift("middle_block.2"))
    block = 0
    for level in (3, 2, 1, 0):
        for i in range(3):
            key = f"output_blocks.{block}"
            x = _resblock64(w, key + ".0", x, shift(key + ".0"), skips.pop())
            if res in (4, 8):
                x = _transformer64(w, key + ".1", x, ctx, 32)
            if level and i == 2:
                x = conv(_up64(x), f"{key}.{2 if res in (4, 8) else 1}.conv")
                res //= 2
            block += 1
    return conv(_silu64(_gn64(x, w["out.0.weight"], w["out.0.bias"], 32, 1e-5)), "out.2")


def exact(case: dict, seed: int):
    i, kind = _inputs(case, seed), case["kind"]
    if kind == "attention":
        return _attention64(i["q"], i["k"], i["v"], case["heads"])
    if kind == "transformer":
        ctx = None
        if case["text"]:
            ctx = i["text"].double() @ i["w"]["context_linear_projection.weight"].double().t()
        return _transformer64(i["w"], "t", i["x"], ctx, case["head"])
    if kind == "conv":
        return _conv64(_up64(i["x"]) if case["up"] else i["x"], i["w"], i["bias"], case["stride"])
    if kind == "resblock":
        return _resblock64(i["w"], "r", i["x"], i["shift"], i["x1"])
    if kind == "vq_resblock":
        w, x = i["w"], i["x"]
        h = _conv64(_silu64(_gn64(x, w["r.norm1.weight"], w["r.norm1.bias"], 16, 1e-6)), w["r.conv1.weight"], w["r.conv1.bias"])
        h = _conv64(_silu64(_gn64(h, w["r.norm2.weight"], w["r.norm2.bias"], 16, 1e-6)), w["r.conv2.weight"], w["r.conv2.bias"])
        return h + (_conv64(x, w["r.nin_shortcut.weight"], w["r.nin_shortcut.bias"]) if case["c"] != case["o"] else x.double())
    if kind == "quantize":
        return None         # indices, and codebook rows chosen by distances of stated roundings
    if kind == "source":
        w, x = i["w"], i["x"].permute(0, 2, 3, 4, 1)
        y = _gn64(x, w["n.weight"], w["n.bias"], _groups(case["c"]), 1e-5)
        z = _conv64(_silu64(y), w["c.weight"], w["c.bias"], case["stride"])
        return tuple(t.permute(0, 4, 1, 2, 3) for t in (y, z))
    ac = _alphas()
    ts = [v + 1 for v in range(0, 1000, 1000 // case["steps"])]
    sel = ac[ts]
    prev = np.concatenate([ac[:1], sel[:-1]])
    one = np.float16(1)
    s1m, inv = np.sqrt(one - sel).astype(np.float64), (one / (one - sel)).astype(np.float64)
    a, prev = sel.astype(np.float64), prev.astype(np.float64)
    sig = np.sqrt((1 - prev) * inv * (1 - a / prev))
    m, cond = i["mask"].double()[..., None], i["cond"].double()
    ctx = i["text"].double() @ i["w"]["context_linear_projection.weight"].double().t()
    x, eps = i["init"].double(), None
    for n, j in enumerate(reversed(range(case["steps"]))):
        x = x * m + (1 - m) * cond
        eps = _unet64(i["w"], case["width"], torch.cat([x, cond * (1 - m), m], -1), float(ts[j]), ctx)
        x = (math.sqrt(prev[j]) * (x - s1m[j] * eps) / math.sqrt(a[j]) + math.sqrt(1 - prev[j] - sig[j] ** 2) * eps
             + sig[j] * i["noise"][n].double())
    return x * m + (1 - m) * cond, eps
