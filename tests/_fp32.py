"""FP32 arithmetic and hi / lo FP16 splits restated for the tests of the FP32 policy (test-side only)."""
from __future__ import annotations

import torch
from torch.nn import functional as F

SLOPE = 0.1


def leaky(y, slope=SLOPE):
    return torch.where(y >= 0, y, slope * y)


def chain(acc, pairs):
    """acc + the products of `pairs`, one FP32 fused multiply-add after the other (a product of two FP32 values is
    exact in 64 bits, where the sum's own rounding is 2^-29 of the FP32 one)."""
    for a, b in pairs:
        acc = (acc.double() + a.double() * b.double()).float()
    return acc


def conv_chain(x, w, b):
    """Convolution of [B,Cin,H,W] with one FP32 FMA chain per output, the bias first."""
    k, (bs, _, hh, ww) = w.shape[-1], x.shape
    x = F.pad(x, (k // 2,) * 4)
    acc = b.view(1, -1, 1, 1).expand(bs, -1, hh, ww)
    return chain(acc, ((x[:, i:i + 1, dy:dy + hh, dx:dx + ww], w[:, i, dy, dx].view(1, -1, 1, 1))
                       for dy in range(k) for dx in range(k) for i in range(w.shape[1])))


def split(v, dim, bits=11):
    """v as hi + lo: both FP16 after scaling the largest magnitude over `dim` to [2^14, 2^15); lo keeps `bits` bits
    of its significand (0: no lo at all)."""
    e = 14 - torch.floor(torch.log2(v.abs().amax(dim, keepdim=True).clamp_min(1e-38)))
    s = (v.double() * 2 ** e).float()
    hi = s.half().float()
    lo = (s - hi).half().float()
    if bits < 11:
        step = 2 ** (torch.floor(torch.log2(lo.abs().clamp_min(1e-30))) - bits + 1)
        lo = torch.round(lo / step) * step if bits else torch.zeros_like(lo)
    return hi.double() / 2 ** e, lo.double() / 2 ** e


def conv_split(x, w, b, bits=11):
    """Convolution by hi hi' + hi lo' + lo hi', the weights scaled by output and the operands by pixel, sums exact."""
    p = w.shape[-1] // 2
    (xh, xl), (wh, wl) = split(x, (1,), bits), split(w, (1, 2, 3), bits)
    return (F.conv2d(xh, wh, padding=p) + F.conv2d(xl, wh, padding=p) + F.conv2d(xh, wl, padding=p)
            + b.double().view(1, -1, 1, 1)).float()


def conv_size(x, w, b):
    """Sum of the magnitudes of an output's terms."""
    return F.conv2d(x.double().abs(), w.double().abs(), b.double().abs(), padding=w.shape[-1] // 2)


def rms(err, size):
    """Root mean square of an error relative to the magnitude of each output's terms."""
    return (err.double() / size.clamp_min(1e-300)).square().mean().sqrt().item()
