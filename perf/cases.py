"""Performance cases of the upscaler: what its users run, over the range of sizes they run it at.

A case is one call of a public entry point of ``aeisu_amd.runtime``:

* ``frames``: ``Upscaler.run`` on frames that already lie in device memory (a video player, a
  capture pipeline or a batch job).  A stream keeps its output buffer and does not wait for the
  finite check (``stream`` true); a single call allocates its output and checks it.
* ``photo``: ``upscale(model, image, tile)`` on an image in host memory, as ``infer.py`` and
  ``evaluate.py`` call it for every file.
* ``controller`` / ``head``: the two halves alone, for programs that keep or edit the coefficients.

``listed`` holds the benchmark's configurations and sizes of the tests; ``draw`` gives further
sizes of the same ranges (sides from 32 to 2,560 pixels, odd ones among them).
"""
from __future__ import annotations

import functools
import math
from pathlib import Path

import torch
from torch.nn import functional as F

from aeisu_amd.runtime import load_model, upscale

WEIGHTS = Path(__file__).resolve().parent.parent / "weights"
# (file, FP32 checkpoint it was made from) of each policy and model
FILES = {
    ("fp32", "area"): ("aeisu_area.pt", "aeisu_area.pt"),
    ("fp16", "area"): ("aeisu_area.pt", "aeisu_area.pt"),
    ("mixed", "area"): ("aeisu_area_mixed_fp8.bin", "aeisu_area.pt"),
    ("int8", "area"): ("aeisu_int8_fp16.pt", "aeisu_area.pt"),
    ("fp32", "div2k"): ("aeisu_div2k_l1.pt", "aeisu_div2k_l1.pt"),
    ("fp16", "div2k"): ("aeisu_div2k_l1.pt", "aeisu_div2k_l1.pt"),
    ("mixed", "div2k"): ("aeisu_div2k_l1_mixed_fp8.bin", "aeisu_div2k_l1.pt"),
}
DTYPE = {"f16": torch.float16, "f32": torch.float32}
BYTES = {"f16": 2, "f32": 4}
# per LR pixel: 11,520 multiply-adds of the controller, 1,900 of the head
CONTROLLER_FLOPS, HEAD_FLOPS = 2 * 11520, 2 * 1900


def _frames(name, policy, h, w, batch=1, model="area", din="f16", dout="f16", stream=True):
    return {"name": name, "kind": "frames", "policy": policy, "model": model, "batch": batch, "h": h, "w": w,
            "in": din, "out": dout, "stream": stream}


def listed():
    return [
        # the headline workload: live 1080p video to 4K on the shipped FP8/FP16 artifact
        _frames("mixed-1080p", "mixed", 1080, 1920),
        # a batch job: four 1440p frames a call, the DIV2K model
        _frames("mixed-div2k-1440p-b4", "mixed", 1440, 2560, batch=4, model="div2k"),
        # a low-resolution stream, bound by latency
        _frames("mixed-540p", "mixed", 540, 960),
        # the smallest call: the 64 x 48 frame that the runtime test starts with
        _frames("mixed-48x64", "mixed", 48, 64),
        # eight 540p streams in one batch on the INT8 route
        _frames("int8-540p-b8", "int8", 540, 960, batch=8),
        # 1080p video on the FP16 policy
        _frames("fp16-1080p", "fp16", 1080, 1920),
        # one still of odd size with FP32 frames and the finite check, as a quality comparison runs it
        _frames("fp16-613x837-f32", "fp16", 613, 837, din="f32", dout="f32", stream=False),
        # the FP32 policy (the arithmetic of the PyTorch path): a crop, and a whole 1080p frame
        _frames("fp32-256", "fp32", 256, 256, din="f32", dout="f32"),
        _frames("fp32-1080p", "fp32", 1080, 1920, din="f32", dout="f32"),
        # an image file of the evaluation set's half resolution through the default tiling
        {"name": "photo-fp16-678x1020", "kind": "photo", "policy": "fp16", "model": "area", "batch": 1, "h": 678,
         "w": 1020, "tile": 128},
        # coefficients alone, and the head alone on given coefficients with FP32 output for post-processing
        {"name": "controller-fp16-720p", "kind": "controller", "policy": "fp16", "model": "area", "batch": 1, "h": 720,
         "w": 1280, "in": "f16"},
        {"name": "head-fp16-1080p", "kind": "head", "policy": "fp16", "model": "area", "batch": 1, "h": 1080, "w": 1920,
         "in": "f16", "out": "f32"},
    ]


# most LR pixels of a drawn call: such a call costs no more than the largest listed one
_MOST = {"mixed": 14_000_000, "int8": 14_000_000, "fp16": 4_000_000, "fp32": 1_000_000}


def draw(rng):
    kind = rng.choice(("frames",) * 6 + ("photo", "controller", "head"))
    policy = rng.choice(("mixed", "mixed", "int8", "fp16", "fp32") if kind == "frames" else
                        ("fp16", "mixed") if kind == "photo" else ("fp16",))
    model = "area" if policy == "int8" else rng.choice(("area", "div2k"))
    top = 1000 if kind == "photo" else 1440
    h = round(math.exp(rng.uniform(math.log(32), math.log(top))))
    w = min(2560, round(h * rng.uniform(0.75, 1.8)))
    most = min(_MOST[policy] // (h * w), 8)
    batch = 1 if kind == "photo" else rng.choice([b for b in (1, 1, 1, 2, 3, 4, 8) if b <= max(1, most)])
    case = {"kind": kind, "policy": policy, "model": model, "batch": batch, "h": h, "w": w}
    if kind == "photo":
        case["tile"] = rng.choice((0, 128, 128, 256))
        return case
    case["in"] = rng.choice(("f16", "f32")) if policy in ("fp16", "fp32") else "f16"
    if kind != "controller":
        case["out"] = rng.choice(("f16", "f32")) if policy == "fp16" else case["in"]
    if kind == "frames":
        case["stream"] = rng.choice((True, True, False))
    return case


# ---- inputs ------------------------------------------------------------------------------------------
def _images(case, seed):
    """[B,3,H,W] float32 in [0, 1] on the GPU: colour noise with a falling spectrum (octaves of bilinear
    value noise), flat regions with hard edges cut into it, and 2 % of sensor noise."""
    b, h, w = case["batch"], case["h"], case["w"]
    g = torch.Generator("cuda").manual_seed(seed)

    def octave(cell, channels):
        grid = torch.rand(b, channels, -(-h // cell) + 1, -(-w // cell) + 1, generator=g, device="cuda") - 0.5
        return F.interpolate(grid, size=(h, w), mode="bilinear", align_corners=True)

    img = sum(octave(cell, 3) * amp for cell, amp in ((128, 0.7), (32, 0.35), (8, 0.15))) + 0.45
    mask = octave(48, 1) + 0.3 * octave(12, 1)
    img = torch.where(mask > 0.15, octave(256, 3) + 0.5, img)
    img += 0.02 * (2 * torch.rand(b, 3, h, w, generator=g, device="cuda") - 1)
    return img.clamp_(0, 1)


def _padded(h, w):
    """(Hp, Wp, py, px): replicate padding to a multiple of 32 and a halo of 16 pixels."""
    ey, ex = -h % 32, -w % 32
    return h + 32 + ey, w + 32 + ex, 16 + ey // 2, 16 + ex // 2


def _coefficients(case, seed):
    """Packed coefficients [B,Hp/2,Wp/2,64] FP16 with the spread that the controller gives (a few per
    cent beyond the clamp's knee at 2)."""
    hp, wp, _, _ = _padded(case["h"], case["w"])
    g = torch.Generator("cuda").manual_seed(seed + 1)
    return torch.randn(case["batch"], hp // 2, wp // 2, 64, generator=g, device="cuda").half()


@functools.lru_cache(maxsize=None)
def _model(policy, model):
    return load_model(WEIGHTS / FILES[policy, model][0], "cuda", policy)


def prepare(case, seed):
    state = {"case": case, "model": _model(case["policy"], case["model"])}
    img = _images(case, seed)
    if case["kind"] == "photo":
        state["image"] = img[0].cpu()
        return state
    state["frames"] = img.to(DTYPE[case["in"]]).contiguous()
    if case["kind"] == "head":
        state["meta"] = _coefficients(case, seed)
    if case["kind"] == "frames" and case["stream"]:
        b, h, w = case["batch"], case["h"], case["w"]
        state["buffer"] = torch.empty(b, 3, 2 * h, 2 * w, dtype=DTYPE[case["out"]], device="cuda")
    return state


def run(state):
    case, model = state["case"], state["model"]
    if case["kind"] == "photo":
        return upscale(model, state["image"], case["tile"])
    if case["kind"] == "controller":
        return model.controller(state["frames"])
    if case["kind"] == "head":
        return model.head(state["frames"], state["meta"], out_dtype=DTYPE[case["out"]])
    if case["stream"]:
        return model.run(state["frames"], out=state["buffer"], check_finite=False)
    return model.run(state["frames"], out_dtype=DTYPE[case["out"]])


def work(case):
    px = case["batch"] * case["h"] * case["w"]
    hp, wp, _, _ = _padded(case["h"], case["w"])
    coefficients = case["batch"] * hp * wp // 4 * 64 * 2
    frame_in, frame_out = 3 * px * BYTES[case.get("in", "f32")], 12 * px * BYTES[case.get("out", "f32")]
    if case["kind"] == "controller":
        return {"bytes": frame_in + coefficients, "flops": px * CONTROLLER_FLOPS}
    if case["kind"] == "head":
        return {"bytes": frame_in + coefficients + frame_out, "flops": px * HEAD_FLOPS}
    return {"bytes": frame_in + frame_out, "flops": px * (CONTROLLER_FLOPS + HEAD_FLOPS)}


def tolerance(case):
    """About four times what another rounding of the sums moves, measured with inputs changed by one part in
    10^6 and against ``exact``.  Mixed and INT8: a sum that crosses a rounding midpoint changes an E4M3 or INT8
    code, which the four 3x3 layers spread (1.0e-3 of the result, single pixels by 0.08; the DIV2K model 1.6e-3
    and 0.2, INT8 1.1e-3 and 0.15).  FP16: 1.6e-5 and 1.3e-3, its coefficients 6.3e-4 and 0.026.  FP32 and the
    head: 1.2e-7 and 8.5e-7; with FP16 output, values at a rounding midpoint move by 2^-10."""
    if case["policy"] in ("mixed", "int8") and case["kind"] != "head":
        return {"rel": 6e-3, "max": 0.8} if case["model"] == "div2k" else {"rel": 4e-3, "max": 0.5}
    if case["kind"] == "controller":
        return {"rel": 2.5e-3, "max": 0.1}
    if case["kind"] == "head" or case["policy"] == "fp32":
        half = case.get("out") == "f16"
        if case["kind"] == "head":
            return {"rel": 1e-4, "max": 2e-3} if half else {"rel": 4e-6, "max": 7e-5}
        return {"rel": 3e-5, "max": 2e-3} if half else {"rel": 1e-6, "max": 2e-5}
    return {"rel": 1e-4, "max": 8e-3}


# ---- the same in 64 bits -----------------------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _weights64(model):
    payload = torch.load(WEIGHTS / FILES["fp32", model][1], map_location="cpu", weights_only=True)
    w = {k: v.cuda().double() for k, v in payload["model"].items()}
    raw = w["basis_raw"]                                             # [16 coefficients, 4 phases, 25 taps]
    raw = raw - raw.mean(-1, keepdim=True)
    w["basis"] = (raw * (float(payload.get("basis_l1_scale", 0.5)) / raw.abs().sum(-1, keepdim=True).clamp_min(1e-6)))
    return w


def _conv64(x, w, b):
    """3x3 (zero padding) or 1x1 convolution of [H,W,Cin] by [Cout,Cin,k,k]."""
    k = w.shape[-1]
    h, wd, _ = x.shape
    x = F.pad(x, (0, 0, k // 2, k // 2, k // 2, k // 2))
    out = b.expand(h * wd, -1).clone()
    for i in range(k):
        for j in range(k):
            out += x[i:i + h, j:j + wd].reshape(h * wd, -1) @ w[:, :, i, j].t().contiguous()
    return out.view(h, wd, -1)


def _leaky(x):
    return torch.where(x >= 0, x, 0.1 * x)


def _unshuffle(x):
    h, w, c = x.shape
    return x.view(h // 2, 2, w // 2, 2, c).permute(0, 2, 4, 1, 3).reshape(h // 2, w // 2, 4 * c)


def _shuffle(x):
    h, w, c = x.shape
    return x.view(h, w, c // 4, 2, 2).permute(0, 3, 1, 4, 2).reshape(2 * h, 2 * w, c // 4)


def _controller64(src, w):
    """Coefficients [Hp/2,Wp/2,64] of one padded frame [3,Hp,Wp]."""
    rgb = [src[c] for c in range(3)]
    maps = [sum(w["analysis_rgb_basis"][i, c] * rgb[c] for c in range(3)) for i in range(3)]
    luma = sum(w["analysis_rgb_mix"][c] * rgb[c] for c in range(3))
    p = F.pad(luma[None, None], (1, 1, 1, 1), mode="replicate")[0, 0]
    h, wd = luma.shape
    at = {(y, x): p[1 + y:1 + y + h, 1 + x:1 + x + wd] for y in (-1, 0, 1) for x in (-1, 0, 1)}
    across, down = at[0, 1] - at[0, -1], at[1, 0] - at[-1, 0]
    a, b, d, e = (w["analysis_" + n] for n in ("dx_rows", "dy_cols", "diag45", "diag135"))
    maps += [luma,
             a[0] * (at[-1, 1] - at[-1, -1]) + a[1] * across + a[2] * (at[1, 1] - at[1, -1]),
             b[0] * (at[1, -1] - at[-1, -1]) + b[1] * down + b[2] * (at[1, 1] - at[-1, 1]),
             d[0] * (at[1, 1] - at[-1, -1]) + d[1] * down + d[2] * across,
             e[0] * (at[-1, 1] - at[1, -1]) - e[1] * down + e[2] * across]
    layer = lambda x, n: _conv64(x, w[n + ".weight"], w[n + ".bias"])  # noqa: E731
    skip = _leaky(layer(_unshuffle(torch.stack(maps, -1)), "project_540"))
    low = _leaky(layer(_unshuffle(skip), "compress_270"))
    halves = [low[..., :32], low[..., 32:]]
    for i in range(1, 5):
        halves = [_leaky(layer(x, "bottleneck_270_%s%d" % (n, i))) for x, n in zip(halves, "ab")]
    work_ = skip + _shuffle(_leaky(layer(torch.cat(halves, -1), "expand_270")))
    return layer(_leaky(layer(work_, "refine_540")), "metadata_head")


def _head64(src, meta, w):
    """Clipped [3,2H,2W] of one frame [3,H,W] and its packed coefficients [Hp/2,Wp/2,64]."""
    h, wd = src.shape[1:]
    hp, wp, py, px = _padded(h, wd)
    c = meta.view(hp // 2, wp // 2, 2, 2, 16).permute(0, 2, 1, 3, 4).reshape(hp, wp, 16)[py:py + h, px:px + wd]
    mag = c.abs()
    c = torch.where(mag <= 2, c, torch.sign(c) * (2 + 0.05 * (mag - 2)).clamp(max=2.5)).reshape(h * wd, 16)
    p = F.pad(src[None], (2, 2, 2, 2), mode="replicate")[0]
    out = src.new_zeros(3, h, 2, wd, 2)
    for t in range(25):
        taps = (c @ w["basis"][:, :, t].contiguous() + w["base_kernel"][t]).view(h, wd, 4)
        window = p[:, t // 5:t // 5 + h, t % 5:t % 5 + wd]
        for ph in range(4):
            out[:, :, ph >> 1, :, ph & 1] += window * taps[..., ph]
    return out.reshape(3, 2 * h, 2 * wd).clamp(0, 1)


def exact(case, seed):
    w = _weights64(case["model"])
    img = _images(case, seed)
    if case["kind"] != "photo":
        img = img.to(DTYPE[case["in"]])
    metas = _coefficients(case, seed).double() if case["kind"] == "head" else None
    hp, wp, py, px = _padded(case["h"], case["w"])
    outs = []
    for i, src in enumerate(img.double()):
        if metas is not None:
            meta = metas[i]
        else:
            pad = (px, wp - px - case["w"], py, hp - py - case["h"])
            meta = _controller64(F.pad(src[None], pad, mode="replicate")[0], w)
        outs.append(meta if case["kind"] == "controller" else _head64(src, meta, w))
    return outs[0] if case["kind"] == "photo" else torch.stack(outs)
