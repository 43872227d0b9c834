"""The calls that programs make of this library, as measurable cases.

listed() names one case of each kind of work at a size that its model has;
draw() gives more of the same kinds over their whole range of sizes. prepare()
puts a case's inputs into the library's device memory, run() makes one pass
through the public entry points (sdhip.Backend, sdhip.ZImage), work() and
tolerance() say what a pass needs and how far two correct results may lie
apart, and exact() computes the same outputs in 64 bits with plain torch.

The kinds, and where a program makes the calls:

  timestep_mlp    the timestep embedding's two fp32 linears with SiLU between
                  (Z-Image: 256 -> 1024 -> 256, one row; SD 1.5's UNet:
                  320 -> 1280 -> 1280, two rows under guidance). The smallest
                  calls: latency and launches.
  text_attention  one causal self-attention of a text encoder over a prompt:
                  Qwen3's grouped heads (QK-norm and rotate-half RoPE first) or
                  CLIP's plain ones.
  rows            the elementwise / normalisation / rotary passes over token
                  rows in a DiT block; a drawn case is any one of them.
  dit_ffn         the DiT's feed-forward: SwiGLU of two bf16-weight
                  projections, then the projection back.
  dit_attention   QK-norm, interleaved RoPE and full self-attention of a
                  Z-Image layer over the joint image + text sequence.
  unet_ff         a UNet transformer block's GEGLU feed-forward front: an fp32
                  linear with bias, then GEGLU.
  unet_attention  SD 1.5's attention: self over the latent's pixels or cross
                  to 77 text tokens; head sizes 40, 80 and 160.
  unet_resnet     a UNet residual block under guidance (two samples):
                  GroupNorm+SiLU, 3x3 convolution, time bias, GroupNorm+SiLU,
                  3x3 convolution, residual (through a 1x1 convolution where
                  the channels change); some are followed by the stride-2
                  convolution of a down block.
  vae_norm        GroupNorm+SiLU alone at the VAE decoder's sizes.
  vae_resnet      a VAE decoder residual block; some are followed by the
                  nearest 2x upsampling and its convolution. The largest work.
  vae_attention   the VAE mid block's one-head attention over 512 channels:
                  GroupNorm, layout change, fp32 projections, attention,
                  projection back, layout change, residual.
  zimage_forward  a whole Z-Image forward (fewer layers than the checkpoint's
                  30) from a latent, a timestep and text features in host
                  memory to the predicted noise in host memory.
"""
import math
import os
import sys

import numpy as np
import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "stablediffusion-cpp_amd"))

import sdhip  # noqa: E402

_BACKEND = None


def _be():
    global _BACKEND
    if _BACKEND is None:
        _BACKEND = sdhip.Backend()
    return _BACKEND


# ------------------------------------------------------------------- the cases
def listed():
    return [
        {"name": "timestep_mlp", "kind": "timestep_mlp", "rows": 1, "cin": 256, "hidden": 1024, "cout": 256},
        {"name": "text_attention", "kind": "text_attention", "S": 203, "heads": 32, "kv_heads": 8, "d": 128,
         "qknorm": True},
        {"name": "dit_rows", "kind": "rows", "op": "rms_norm_gated_add_modulate_bf16", "rows": 4224, "C": 3840},
        {"name": "dit_ffn", "kind": "dit_ffn", "rows": 4224, "dim": 3840, "hidden": 10240},
        {"name": "dit_attention", "kind": "dit_attention", "S": 4224, "heads": 30},
        {"name": "unet_ff", "kind": "unet_ff", "rows": 8192, "dim": 320},
        {"name": "unet_attention", "kind": "unet_attention", "N": 2, "Sq": 4096, "Skv": 4096, "heads": 8, "d": 40},
        {"name": "unet_resnet", "kind": "unet_resnet", "N": 2, "cin": 960, "cout": 640, "H": 32, "W": 32,
         "down": False},
        {"name": "vae_norm", "kind": "vae_norm", "C": 512, "H": 128, "W": 128},
        {"name": "vae_resnet", "kind": "vae_resnet", "cin": 256, "cout": 256, "H": 256, "W": 256, "up": True},
        {"name": "vae_attention", "kind": "vae_attention", "H": 64, "W": 64},
        {"name": "zimage_forward", "kind": "zimage_forward", "layers": 2, "H": 64, "W": 64, "L": 77},
    ]


def _log(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


_ROW_OPS = ("rms_norm_gated_add_modulate_bf16", "rms_norm_modulate_bf16", "add_rms_norm", "ln_modulate_gate",
            "layer_norm", "swiglu", "rope_qk", "softmax_rows")


def draw(rng):
    kind = rng.choice([c["kind"] for c in listed()])
    if kind == "timestep_mlp":
        return {"kind": kind, "rows": rng.choice((1, 2, 4, 8)), "cin": _log(rng, 64, 1280),
                "hidden": _log(rng, 256, 2048), "cout": _log(rng, 64, 1280)}
    if kind == "text_attention":
        if rng.random() < 0.5:
            return {"kind": kind, "S": _log(rng, 5, 512), "heads": 32, "kv_heads": 8, "d": 128, "qknorm": True}
        return {"kind": kind, "S": _log(rng, 5, 256), "heads": rng.choice((12, 16)), "kv_heads": 0, "d": 64,
                "qknorm": False}
    if kind == "rows":
        op = rng.choice(_ROW_OPS)
        C = rng.choice((320, 768, 1000, 1280, 2560, 3840, 3840, 5120))
        if op in ("swiglu", "softmax_rows"):
            C = rng.choice((77, 1000, 1280, 4096, 4224, 10240))
        if op == "rope_qk":
            C = 128 * rng.choice((2, 8, 16, 30, 32))
        return {"kind": kind, "op": op, "rows": _log(rng, 1, 8192), "C": C}
    if kind == "dit_ffn":
        dim, hidden = rng.choice(((3840, 10240), (3840, 10240), (2560, 9728), (256, 512)))
        return {"kind": kind, "rows": _log(rng, 32, 4608), "dim": dim, "hidden": hidden}
    if kind == "dit_attention":
        return {"kind": kind, "S": _log(rng, 64, 4608), "heads": rng.choice((2, 30, 30))}
    if kind == "unet_ff":
        dim = rng.choice((320, 640, 1280))
        return {"kind": kind, "rows": _log(rng, 64, 8192 * 320 // dim), "dim": dim}
    if kind == "unet_attention":
        d = rng.choice((40, 80, 160))
        Sq = _log(rng, 64, {40: 4608, 80: 1152, 160: 512}[d])
        return {"kind": kind, "N": rng.choice((1, 2)), "Sq": Sq, "Skv": rng.choice((Sq, 77)), "heads": 8, "d": d}
    if kind == "unet_resnet":
        level = rng.randrange(4)  # channels and the side of a 512 x 512 image's latent at that level
        cout = (320, 640, 1280, 1280)[level]
        side = 64 >> level
        cin = rng.choice(((320, 640, 960), (320, 640, 960, 1280, 1920), (640, 1280, 1920, 2560), (1280, 2560))[level])
        return {"kind": kind, "N": rng.choice((1, 2)), "cin": cin, "cout": cout, "H": side + rng.randrange(0, side // 2),
                "W": side - rng.randrange(0, side // 4 + 1), "down": level < 3 and rng.random() < 0.3}
    if kind == "vae_norm":
        C = rng.choice((128, 256, 512))
        H = _log(rng, 24, {128: 1024, 256: 640, 512: 384}[C])
        return {"kind": kind, "C": C, "H": H, "W": max(16, H - rng.randrange(0, H // 3))}
    if kind == "vae_resnet":
        cin, cout = rng.choice(((512, 512), (512, 256), (256, 256), (256, 128), (128, 128)))
        H = _log(rng, 24, {512: 128, 256: 256, 128: 448}[cin])
        return {"kind": kind, "cin": cin, "cout": cout, "H": H, "W": max(16, H - rng.randrange(0, H // 3)),
                "up": cout >= 256 and rng.random() < 0.4}
    if kind == "vae_attention":
        H = _log(rng, 16, 80)
        return {"kind": kind, "H": H, "W": max(12, H - rng.randrange(0, H // 3))}
    return {"kind": "zimage_forward", "layers": rng.choice((1, 2)), "H": 2 * rng.randrange(8, 41),
            "W": 2 * rng.randrange(8, 41), "L": _log(rng, 5, 256)}


# ---------------------------------------------------------------------- inputs
class _Span:
    """A DArray seen by torch (torch.as_tensor keeps it, and so the memory, alive)."""

    def __init__(self, arr):
        self.arr = arr
        self.__cuda_array_interface__ = {"shape": arr.shape, "data": (arr.ptr, False), "version": 2,
                                         "typestr": "<f4" if arr.dtype == np.float32 else "<i2"}


def _view(arr):
    t = torch.as_tensor(_Span(arr), device="cuda")
    return t if arr.dtype == np.float32 else t.view(torch.bfloat16)


class _Make:
    """Seeded inputs on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def randn(self, *shape, mean=0.0, std=1.0):
        return torch.randn(shape, generator=self.g, device="cuda", dtype=torch.float32) * std + mean

    def linear(self, out, inn):
        return self.randn(out, inn, std=1.0 / math.sqrt(inn))

    def stream(self, rows, C):
        """Hidden rows: channels of unequal size, as a residual stream has them."""
        return self.randn(rows, C) * torch.exp(0.5 * self.randn(C))


def _rope_tables(S, dim, interleaved):
    """cos and sin [S, dim] of positions 0 .. S-1: angles stored twice, side by side (interleaved) or half by half."""
    theta = 256.0 if interleaved else 1e6
    f = theta ** (-torch.arange(0, dim, 2, device="cuda", dtype=torch.float64) / dim)
    a = (torch.arange(S, device="cuda", dtype=torch.float64)[:, None] * f).float()
    a = a.repeat_interleave(2, dim=1) if interleaved else torch.cat((a, a), dim=1)
    return a.cos(), a.sin()


def _resnet_inputs(m, N, cin, cout, H, W, time, extra):
    d = {"x": m.randn(N, cin, H, W), "g1": m.randn(cin, mean=1.0, std=0.1), "b1": m.randn(cin, std=0.1),
         "w1": m.linear(cout, cin * 9), "c1": m.randn(cout, std=0.02),
         "g2": m.randn(cout, mean=1.0, std=0.1), "b2": m.randn(cout, std=0.1),
         "w2": m.linear(cout, cout * 9), "c2": m.randn(cout, std=0.02)}
    if cin != cout:
        d.update(ws=m.linear(cout, cin), cs=m.randn(cout, std=0.02))
    if time:
        d["temb"] = m.randn(N, cout, std=0.5)
    if extra:
        d.update(we=m.linear(cout, cout * 9), ce=m.randn(cout, std=0.02))
    return d


def _inputs(c, seed):
    """The case's inputs, from the seed alone."""
    m, kind = _Make(seed), c["kind"]
    if kind == "timestep_mlp":
        return {"x": m.randn(c["rows"], c["cin"], std=0.7), "w1": m.linear(c["hidden"], c["cin"]),
                "b1": m.randn(c["hidden"], std=0.02), "w2": m.linear(c["cout"], c["hidden"]),
                "b2": m.randn(c["cout"], std=0.02)}
    if kind == "text_attention":
        S, d = c["S"], c["d"]
        kv = c["kv_heads"] or c["heads"]
        t = {"q": m.randn(1, S, c["heads"] * d), "k": m.randn(1, S, kv * d), "v": m.randn(1, S, kv * d)}
        if c["qknorm"]:
            t.update(gq=m.randn(d, mean=1.0, std=0.1), gk=m.randn(d, mean=1.0, std=0.1))
            t["cos"], t["sin"] = _rope_tables(S, d, False)
        return t
    if kind == "rows":
        R, C, op = c["rows"], c["C"], c["op"]
        if op == "swiglu":
            return {"x": m.randn(R, C, std=1.5), "a": m.randn(R, C, std=1.5)}
        if op == "softmax_rows":
            return {"x": m.randn(R, C, std=3.0)}
        if op == "rope_qk":
            t = {"x": m.randn(R, C), "a": m.randn(R, C)}
            t["cos"], t["sin"] = _rope_tables(R, 128, True)
            return t
        t = {"x": m.stream(R, C)}
        if op not in ("rms_norm_modulate_bf16", "layer_norm"):
            t["a"] = m.stream(R, C)
        for n in ("v1", "v2", "v3", "v4"):  # norm weights, 1 + scale, shift, gate
            t[n] = m.randn(C, mean=1.0 if n in ("v1", "v3") else 0.0, std=0.3)
        return t
    if kind == "dit_ffn":
        return {"x": m.randn(c["rows"], c["dim"]), "w1": m.linear(c["hidden"], c["dim"]).bfloat16(),
                "w3": m.linear(c["hidden"], c["dim"]).bfloat16(), "w2": m.linear(c["dim"], c["hidden"]).bfloat16()}
    if kind == "dit_attention":
        D = 128 * c["heads"]
        t = {n: m.stream(c["S"], D)[None] for n in ("q", "k", "v")}
        t.update(gq=m.randn(128, mean=1.0, std=0.1), gk=m.randn(128, mean=1.0, std=0.1))
        t["cos"], t["sin"] = _rope_tables(c["S"], 128, True)
        return t
    if kind == "unet_ff":
        return {"x": m.randn(c["rows"], c["dim"]), "w": m.linear(8 * c["dim"], c["dim"]),
                "b": m.randn(8 * c["dim"], std=0.02)}
    if kind == "unet_attention":
        D = c["heads"] * c["d"]
        return {"q": m.randn(c["N"], c["Sq"], D, std=1.5), "k": m.randn(c["N"], c["Skv"], D, std=1.5),
                "v": m.randn(c["N"], c["Skv"], D)}
    if kind == "unet_resnet":
        return _resnet_inputs(m, c["N"], c["cin"], c["cout"], c["H"], c["W"], True, c["down"])
    if kind == "vae_norm":
        return {"x": m.randn(1, c["C"], c["H"], c["W"], std=2.0), "g": m.randn(c["C"], mean=1.0, std=0.1),
                "b": m.randn(c["C"], std=0.1)}
    if kind == "vae_resnet":
        return _resnet_inputs(m, 1, c["cin"], c["cout"], c["H"], c["W"], False, c["up"])
    if kind == "vae_attention":
        t = {"x": m.randn(1, 512, c["H"], c["W"]), "g": m.randn(512, mean=1.0, std=0.1), "b": m.randn(512, std=0.1)}
        for n in "qkvo":
            t["w" + n], t["b" + n] = m.linear(512, 512) * (2.0 if n in "qk" else 1.0), m.randn(512, std=0.02)
        return t
    raise ValueError(kind)


def _outputs(c):
    """name -> (shape, dtype) of the device arrays that run() writes besides its inputs."""
    kind = c["kind"]
    f, h = np.float32, np.uint16  # h: the bits of a bfloat16
    if kind == "timestep_mlp":
        return {"h": ((c["rows"], c["hidden"]), f), "y": ((c["rows"], c["cout"]), f)}
    if kind == "text_attention":
        return {"y": ((1, c["S"], c["heads"] * c["d"]), f)}
    if kind == "rows":
        op, shape = c["op"], (c["rows"], c["C"])
        if op in ("softmax_rows", "rope_qk"):
            return {}
        return {"y": (shape, h if op.endswith("bf16") else f)}
    if kind == "dit_ffn":
        return {"h": ((c["rows"], c["hidden"]), f), "y": ((c["rows"], c["dim"]), f)}
    if kind == "dit_attention":
        return {"y": ((1, c["S"], 128 * c["heads"]), f)}
    if kind == "unet_ff":
        return {"h": ((c["rows"], 8 * c["dim"]), f), "y": ((c["rows"], 4 * c["dim"]), f)}
    if kind == "unet_attention":
        return {"y": ((c["N"], c["Sq"], c["heads"] * c["d"]), f)}
    if kind == "vae_norm":
        return {"y": ((1, c["C"], c["H"], c["W"]), f)}
    if kind == "vae_attention":
        S = c["H"] * c["W"]
        t = {n: ((1, S, 512), f) for n in ("h", "q", "k", "v", "a")}
        t.update(n=((1, 512, c["H"], c["W"]), f), y=((1, 512, c["H"], c["W"]), f))
        return t
    N, cin, cout, H, W = c.get("N", 1), c["cin"], c["cout"], c["H"], c["W"]
    t = {"n1": ((N, cin, H, W), f), "h1": ((N, cout, H, W), f), "n2": ((N, cout, H, W), f), "y": ((N, cout, H, W), f)}
    if cin != cout:
        t["s"] = ((N, cout, H, W), f)
    if c.get("down"):
        t["e"] = ((N, cout, (H - 1) // 2 + 1, (W - 1) // 2 + 1), f)
    if c.get("up"):
        t.update(u=((N, cout, 2 * H, 2 * W), f), e=((N, cout, 2 * H, 2 * W), f))
    return t


def prepare(case, seed):
    be = _be()
    st = {"case": case, "be": be, "d": {}}
    if case["kind"] == "zimage_forward":
        rng = np.random.default_rng(seed)
        st["model"] = sdhip.ZImage.random(noise_refiners=1, context_refiners=1, layers=case["layers"], seed=seed)
        st["x"] = rng.standard_normal((1, 16, case["H"], case["W"]), dtype=np.float32)
        st["cap"] = rng.standard_normal((1, case["L"], 2560), dtype=np.float32)
        st["t"] = float(rng.uniform(0.05, 0.95))
        return st
    for n, t in _inputs(case, seed).items():
        a = sdhip.DArray(be, t.shape, dtype=np.uint16 if t.dtype == torch.bfloat16 else np.float32)
        _view(a).copy_(t)
        st["d"][n] = a
    for n, (shape, dtype) in _outputs(case).items():
        st["d"][n] = sdhip.DArray(be, shape, dtype=dtype)
    torch.cuda.synchronize()  # the library works on a stream of its own
    st["out"] = {n: _view(st["d"][n]) for n in _returned(case)}
    return st


def _returned(c):
    """The arrays that a pass computes and its caller reads, updates in place among them."""
    kind = c["kind"]
    if kind in ("text_attention", "dit_attention"):
        return ("y", "q") if kind == "dit_attention" or c["qknorm"] else ("y",)
    if kind == "rows":
        return {"softmax_rows": ("x",), "rope_qk": ("x", "a"), "add_rms_norm": ("x", "y"),
                "rms_norm_gated_add_modulate_bf16": ("x", "y"), "ln_modulate_gate": ("a", "y")}.get(c["op"], ("y",))
    if kind == "timestep_mlp":
        return ("h", "y")
    return ("e", "y") if c.get("up") or c.get("down") else ("y",)


# ------------------------------------------------------------------------ runs
def _resnet(be, d, N, cin, cout, H, W, eps, down, up):
    HW = H * W
    be.group_norm(d["x"], d["n1"], N, cin, HW, 32, d["g1"], d["b1"], eps, silu=True)
    be.conv2d(d["n1"], N, cin, H, W, d["w1"], cout, 3, 3, d["c1"], 1, 1, d["h1"], H, W)
    if "temb" in d:
        be.add_channel_bias(d["h1"], d["temb"], N, cout, HW)
    be.group_norm(d["h1"], d["n2"], N, cout, HW, 32, d["g2"], d["b2"], eps, silu=True)
    be.conv2d(d["n2"], N, cout, H, W, d["w2"], cout, 3, 3, d["c2"], 1, 1, d["y"], H, W)
    skip = d["x"]
    if cin != cout:
        be.conv2d(d["x"], N, cin, H, W, d["ws"], cout, 1, 1, d["cs"], 1, 0, d["s"], H, W)
        skip = d["s"]
    be.add(d["y"], skip, N * cout * HW)
    if down:
        be.conv2d(d["y"], N, cout, H, W, d["we"], cout, 3, 3, d["ce"], 2, 1, d["e"], (H - 1) // 2 + 1,
                  (W - 1) // 2 + 1)
    if up:
        be.upsample_nearest2x(d["y"], d["u"], N * cout, H, W)
        be.conv2d(d["u"], N, cout, 2 * H, 2 * W, d["we"], cout, 3, 3, d["ce"], 1, 1, d["e"], 2 * H, 2 * W)


def run(state):
    c, be, d = state["case"], state["be"], state["d"]
    kind = c["kind"]
    if kind == "zimage_forward":
        return {"y": state["model"].forward(state["x"], state["t"], state["cap"])}
    if kind == "timestep_mlp":
        R, I, H, O = c["rows"], c["cin"], c["hidden"], c["cout"]
        be.gemm_nt_f32(R, H, I, d["x"], I, d["w1"], I, d["h"], H, d["b1"])
        be.silu(d["h"], R * H)
        be.gemm_nt_f32(R, O, H, d["h"], H, d["w2"], H, d["y"], O, d["b2"])
    elif kind == "text_attention":
        S, hd = c["S"], c["d"]
        kv = c["kv_heads"] or c["heads"]
        if c["qknorm"]:
            be.qknorm_rope(d["q"], c["heads"] * hd, d["k"], kv * hd, 1, S, hd, d["gq"], d["gk"], 1e-6, d["cos"],
                           d["sin"], False)
        be.attention(d["q"], d["k"], d["v"], d["y"], 1, S, S, c["heads"], kv, hd, True)
    elif kind == "rows":
        R, C, op = c["rows"], c["C"], c["op"]
        if op == "swiglu":
            be.swiglu(d["x"], d["a"], d["y"], R * C)
        elif op == "softmax_rows":
            be.softmax_rows(d["x"], R, C, 0.125)
        elif op == "rope_qk":
            be.rope_qk(d["x"], C, d["a"], C, 1, R, 128, d["cos"], d["sin"], True)
        elif op == "add_rms_norm":
            be.add_rms_norm(d["x"], d["a"], d["y"], R, C, d["v1"], 1e-6)
        elif op == "layer_norm":
            be.layer_norm(d["x"], d["y"], R, C, d["v1"], d["v2"], 1e-5)
        elif op == "ln_modulate_gate":
            be.ln_modulate_gate(d["x"], d["a"], d["v2"], d["v4"], d["v2"], d["y"], R, C, 1e-6)
        elif op == "rms_norm_modulate_bf16":
            be.rms_norm_modulate_bf16(d["x"], d["y"], R, C, d["v1"], d["v3"], 1e-5)
        else:
            be.rms_norm_gated_add_modulate_bf16(d["x"], d["a"], d["y"], R, C, d["v1"], d["v2"], d["v3"], d["v3"], 1e-5)
    elif kind == "dit_ffn":
        R, D, F = c["rows"], c["dim"], c["hidden"]
        be.linear_swiglu(d["x"], d["w1"], d["w3"], d["h"], R, D, F)
        be.gemm_nt_bf16(R, D, F, d["h"], F, d["w2"], F, d["y"], D)
    elif kind == "dit_attention":
        be.qknorm_rope_attention(d["q"], d["k"], d["v"], d["y"], 1, c["S"], c["heads"], 128, d["gq"], d["gk"], 1e-5,
                                 d["cos"], d["sin"])
    elif kind == "unet_ff":
        R, D = c["rows"], c["dim"]
        be.gemm_nt_f32(R, 8 * D, D, d["x"], D, d["w"], D, d["h"], 8 * D, d["b"])
        be.geglu(d["h"], d["y"], R, 4 * D)
    elif kind == "unet_attention":
        be.attention(d["q"], d["k"], d["v"], d["y"], c["N"], c["Sq"], c["Skv"], c["heads"], c["heads"], c["d"])
    elif kind == "unet_resnet":
        _resnet(be, d, c["N"], c["cin"], c["cout"], c["H"], c["W"], 1e-5, c["down"], False)
    elif kind == "vae_norm":
        be.group_norm(d["x"], d["y"], 1, c["C"], c["H"] * c["W"], 32, d["g"], d["b"], 1e-6, silu=True)
    elif kind == "vae_resnet":
        _resnet(be, d, 1, c["cin"], c["cout"], c["H"], c["W"], 1e-6, False, c["up"])
    elif kind == "vae_attention":
        S = c["H"] * c["W"]
        be.group_norm(d["x"], d["n"], 1, 512, S, 32, d["g"], d["b"], 1e-6)
        be.nchw_to_nlc(d["n"], d["h"], 1, 512, S)
        for n in "qkv":
            be.gemm_nt_f32(S, 512, 512, d["h"], 512, d["w" + n], 512, d[n], 512, d["b" + n])
        be.attention(d["q"], d["k"], d["v"], d["a"], 1, S, S, 1, 1, 512)
        be.gemm_nt_f32(S, 512, 512, d["a"], 512, d["wo"], 512, d["h"], 512, d["bo"])
        be.nlc_to_nchw(d["h"], d["y"], 1, 512, S)
        be.add(d["y"], d["x"], 512 * S)
    else:
        raise ValueError(kind)
    return state["out"]


# ------------------------------------------------------------ what a pass needs
def work(c):
    """Bytes of a pass's inputs (weights among them) and outputs, each once, and its operations."""
    kind = c["kind"]
    if kind == "timestep_mlp":
        R, I, H, O = c["rows"], c["cin"], c["hidden"], c["cout"]
        return {"bytes": 4 * (R * I + H * I + H + O * H + O + R * O), "flops": 2 * R * H * (I + O)}
    if kind == "text_attention":
        S, d, h = c["S"], c["d"], c["heads"]
        kv = c["kv_heads"] or h
        n = S * d * (2 * h + 2 * kv) + (S * d * (h + kv) + 2 * S * d if c["qknorm"] else 0)
        return {"bytes": 4 * n, "flops": 4 * d * h * S * (S + 1) // 2}
    if kind == "rows":
        n = c["rows"] * c["C"]
        per = {"rms_norm_gated_add_modulate_bf16": 14, "rms_norm_modulate_bf16": 6, "add_rms_norm": 16,
               "ln_modulate_gate": 16, "layer_norm": 8, "swiglu": 12, "rope_qk": 16, "softmax_rows": 8}[c["op"]]
        more = 8 * c["rows"] * 128 if c["op"] == "rope_qk" else 0 if c["op"] in ("swiglu", "softmax_rows") else 12 * c["C"]
        return {"bytes": per * n + more, "flops": 8 * n}
    if kind == "dit_ffn":
        R, D, F = c["rows"], c["dim"], c["hidden"]
        return {"bytes": 8 * R * D + 6 * D * F, "flops": 6 * R * D * F}
    if kind == "dit_attention":
        S, D = c["S"], 128 * c["heads"]
        return {"bytes": 4 * (5 * S * D + 2 * S * 128), "flops": 4 * S * S * D}
    if kind == "unet_ff":
        R, D = c["rows"], c["dim"]
        return {"bytes": 4 * (R * D + 8 * D * D + 8 * D + R * 4 * D), "flops": 16 * R * D * D}
    if kind == "unet_attention":
        D = c["heads"] * c["d"]
        return {"bytes": 8 * c["N"] * D * (c["Sq"] + c["Skv"]), "flops": 4 * c["N"] * c["Sq"] * c["Skv"] * D}
    if kind == "vae_norm":
        n = c["C"] * c["H"] * c["W"]
        return {"bytes": 8 * n, "flops": 10 * n}
    if kind == "vae_attention":
        S = c["H"] * c["W"]
        return {"bytes": 4 * (2 * S * 512 + 4 * 512 * 513), "flops": 8 * S * 512 * 512 + 4 * S * S * 512}
    if kind == "zimage_forward":
        D, F, I, T = 3840, 10240, c["H"] * c["W"] // 4, 0
        I, T = -(-I // 32) * 32, -(-c["L"] // 32) * 32  # rows are padded to 32 tokens
        per = 4 * D * D + 3 * D * F
        f = sum(n * (2 * S * per + 4 * S * S * D) for n, S in ((1, I), (1, T), (c["layers"], I + T)))
        return {"bytes": 2 * per * (2 + c["layers"]) + 8 * 16 * c["H"] * c["W"] + 4 * c["L"] * 2560, "flops": f}
    N, ci, co, H, W = c.get("N", 1), c["cin"], c["cout"], c["H"], c["W"]
    HW, sc = H * W, 0 if ci == co else 1
    n, f = N * HW * (ci + co) + 9 * co * (ci + co) + sc * ci * co, 2 * N * HW * co * (9 * (ci + co) + sc * ci)
    if c.get("down"):
        o = ((H - 1) // 2 + 1) * ((W - 1) // 2 + 1)
        n, f = n + N * o * co + 9 * co * co, f + 2 * N * o * co * 9 * co
    if c.get("up"):
        n, f = n + 4 * N * HW * co + 9 * co * co, f + 8 * N * HW * co * 9 * co
    return {"bytes": 4 * n, "flops": f}


def tolerance(c):
    """fp32 sums in another order lie about 1e-6 apart (measured against exact(): 3e-8 to 1.5e-6); where a value is
    rounded to bf16 on the way, a last-bit change upstream moves some roundings by one step (2^-8 of the value)."""
    kind = c["kind"]
    if kind == "zimage_forward":
        return {"rel": 6e-3, "max": 0.1}  # bf16 roundings in every layer: a 1e-7 change of the input gives 1.5e-3
    if kind == "dit_ffn":
        return {"rel": 3e-4, "max": 0.02}  # measured against exact(): 5e-5, the bf16 hidden rows' roundings
    if kind == "rows" and c["op"].endswith("bf16"):
        return {"rel": 5e-4, "max": 8e-3}
    return {"rel": 6e-6, "max": 2e-4}


# --------------------------------------------------------------------- 64 bits
def _gn64(x, g, b, eps, silu):
    y = torch.nn.functional.group_norm(x, 32, g, b, eps)
    return y * torch.sigmoid(y) if silu else y


def _conv64(x, w, cout, k, bias, stride, pad):
    """A convolution as one matrix product per kernel tap."""
    N, ci, H, W = x.shape
    Ho, Wo = (H + 2 * pad - k) // stride + 1, (W + 2 * pad - k) // stride + 1
    xp = torch.nn.functional.pad(x, (pad, pad, pad, pad))
    w = w.reshape(cout, ci, k, k)
    out = []
    for n in range(N):
        y = bias[:, None].expand(cout, Ho * Wo).clone()
        for i in range(k):
            for j in range(k):
                s = xp[n, :, i:i + stride * (Ho - 1) + 1:stride, j:j + stride * (Wo - 1) + 1:stride]
                y += w[:, :, i, j].contiguous() @ s.reshape(ci, Ho * Wo)
        out.append(y.reshape(cout, Ho, Wo))
    return torch.stack(out)


def _attn64(q, k, v, heads, kv_heads, causal):
    N, Sq, D = q.shape
    Skv, d = k.shape[1], D // heads
    y = torch.empty_like(q)
    for n in range(N):
        for h in range(heads):
            g = h // (heads // kv_heads)
            s = (q[n, :, h * d:(h + 1) * d] @ k[n, :, g * d:(g + 1) * d].t().contiguous()) / math.sqrt(d)
            if causal:
                s.masked_fill_(torch.ones(Sq, Skv, dtype=torch.bool, device="cuda").triu(1), -math.inf)
            y[n, :, h * d:(h + 1) * d] = torch.softmax(s, dim=1) @ v[n, :, g * d:(g + 1) * d]
    return y


def _rms64(x, g, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * g


def _rope64(x, dim, cos, sin, interleaved):
    """x [..., S, heads * dim] rotated by tables [S, dim]."""
    y = x.reshape(x.shape[-2], -1, dim)
    c, s = cos[:, None], sin[:, None]
    if interleaved:
        a, b = y[..., 0::2], y[..., 1::2]
        r = torch.stack((a * c[..., 0::2] - b * s[..., 0::2], b * c[..., 0::2] + a * s[..., 0::2]), dim=-1)
    else:
        a, b = y.chunk(2, dim=-1)
        ca, cb = c.chunk(2, dim=-1)
        sa, sb = s.chunk(2, dim=-1)
        r = torch.cat((a * ca - b * sa, b * cb + a * sb), dim=-1)
    return r.reshape(x.shape)


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "zimage_forward":
        return None  # its weights exist only inside the model, and its bf16 roundings have no 64-bit counterpart
    f32 = _inputs(c, seed)
    t = {n: v.double() for n, v in f32.items()}
    if kind == "timestep_mlp":
        h = t["x"] @ t["w1"].t() + t["b1"]
        h = h * torch.sigmoid(h)
        return {"h": h, "y": h @ t["w2"].t() + t["b2"]}
    if kind in ("text_attention", "dit_attention"):
        dit = kind == "dit_attention"
        d = 128 if dit else c["d"]
        kv = c["heads"] if dit else c["kv_heads"] or c["heads"]
        if dit or c["qknorm"]:
            eps = 1e-5 if dit else 1e-6
            for n in "qk":
                x = t[n]
                x = _rms64(x.reshape(1, c["S"], -1, d), t["g" + n], eps).reshape(x.shape)
                t[n] = _rope64(x, d, t["cos"], t["sin"], dit)
        y = _attn64(t["q"], t["k"], t["v"], c["heads"], kv, not dit)
        return {"y": y, "q": t["q"]} if dit or c["qknorm"] else {"y": y}
    if kind == "rows":
        op, x = c["op"], t["x"]
        if op == "swiglu":
            return {"y": x * torch.sigmoid(x) * t["a"]}
        if op == "softmax_rows":
            return {"x": torch.softmax(x * 0.125, dim=1)}
        if op == "rope_qk":
            return {n: _rope64(t[n], 128, t["cos"], t["sin"], True) for n in ("x", "a")}
        if op == "add_rms_norm":
            x = x + t["a"]
            return {"x": x, "y": _rms64(x, t["v1"], 1e-6)}
        if op == "layer_norm":
            return {"y": torch.nn.functional.layer_norm(x, (c["C"],), t["v1"], t["v2"], 1e-5)}
        if op == "ln_modulate_gate":
            y = torch.nn.functional.layer_norm(x, (c["C"],), None, None, 1e-6) * (1 + t["v2"]) + t["v4"]
            return {"a": t["a"] + torch.tanh(t["v2"]) * y, "y": y}
        if op == "rms_norm_modulate_bf16":
            return {"y": _rms64(x, t["v1"], 1e-5) * t["v3"]}
        x = x + t["v2"] * _rms64(t["a"], t["v1"], 1e-5)
        return {"x": x, "y": _rms64(x, t["v3"], 1e-5) * t["v3"]}
    if kind == "dit_ffn":  # the entry points round the products' left operands to bf16
        x = f32["x"].bfloat16().double()
        g = x @ t["w1"].t().contiguous()
        h = g * torch.sigmoid(g) * (x @ t["w3"].t().contiguous())
        return {"y": h.float().bfloat16().double() @ t["w2"].t().contiguous()}
    if kind == "unet_ff":
        h = t["x"] @ t["w"].t().contiguous() + t["b"]
        a, b = h.chunk(2, dim=1)
        return {"y": a * 0.5 * b * (1 + torch.erf(b / math.sqrt(2.0)))}
    if kind == "unet_attention":
        return {"y": _attn64(t["q"], t["k"], t["v"], c["heads"], c["heads"], False)}
    if kind == "vae_norm":
        return {"y": _gn64(t["x"], t["g"], t["b"], 1e-6, True)}
    if kind == "vae_attention":
        S = c["H"] * c["W"]
        h = _gn64(t["x"], t["g"], t["b"], 1e-6, False).reshape(512, S).t().contiguous()
        q, k, v = (h @ t["w" + n].t().contiguous() + t["b" + n] for n in "qkv")
        o = _attn64(q[None], k[None], v[None], 1, 1, False)[0] @ t["wo"].t().contiguous() + t["bo"]
        return {"y": t["x"] + o.t().reshape(t["x"].shape)}
    eps = 1e-5 if kind == "unet_resnet" else 1e-6
    co = c["cout"]
    h = _conv64(_gn64(t["x"], t["g1"], t["b1"], eps, True), t["w1"], co, 3, t["c1"], 1, 1)
    if "temb" in t:
        h = h + t["temb"][:, :, None, None]
    y = _conv64(_gn64(h, t["g2"], t["b2"], eps, True), t["w2"], co, 3, t["c2"], 1, 1)
    y = y + (_conv64(t["x"], t["ws"], co, 1, t["cs"], 1, 0) if "ws" in t else t["x"])
    if c.get("down"):
        return {"e": _conv64(y, t["we"], co, 3, t["ce"], 2, 1), "y": y}
    if c.get("up"):
        u = y.repeat_interleave(2, dim=2).repeat_interleave(2, dim=3)
        return {"e": _conv64(u, t["we"], co, 3, t["ce"], 1, 1), "y": y}
    return {"y": y}
