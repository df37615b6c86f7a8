"""FP32 policy: every stage against the same stage in 64 bits on the GPU's own input, at the edges of the
kernels' tiles and over FP32's range.

The layers from compress to the tail run as hi / lo FP16 splits on the MFMA (k_fp32.hip).  The bound of an output is
2^-22 P sum |w||x| with P = 3 + 4 K / 8 at K products: each operand is held to 2^-22 (two operands and the
dropped lo lo' product: 3), and the FP32 accumulators round once per 8 products, in three chains of which
one is at the main sum's magnitude (2^-24 a rounding, taken as 2^-22 for terms that the MFMA cuts off when it
aligns them).  That is the worst case of an output, 100 times and more what is seen, so the error over all outputs is
also held to that of FP32 FMA chains, which a split that loses bits exceeds.
"""
from __future__ import annotations

import pytest
import torch
from torch.nn import functional as F

from oracle import model as M
from tests._fp32 import chain, conv_chain, conv_size, leaky, rms
from tests._util import WEIGHTS, crop_output, pad_frame

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def R(gpu):
    from aeisu_amd import runtime
    return runtime


@pytest.fixture(scope="module", params=["aeisu_area", "aeisu_div2k_l1"])
def model(R, request):
    return R.load_model(WEIGHTS / f"{request.param}.pt", precision="fp32"), M.load_folded(WEIGHTS / f"{request.param}.pt")


def stages(model, frames):
    """skip, low0..4, work, meta of a run that keeps them (NCHW, CPU)."""
    from aeisu_amd import _lib as L
    b, _, h, w = frames.shape
    flags = L.FLAG_KEEP_INTERMEDIATES
    hd = model.handle(b, h, w, torch.float32, torch.float32, flags)
    model.run(frames.cuda().contiguous(), flags=flags, check_finite=False)
    torch.cuda.synchronize()
    _, _, _, _, hq, wq = model.geometry(hd)

    def fetch(which, hh, ww, c):
        t = model.intermediate(hd, which).cpu().view(torch.float32)
        return t.reshape(b, hh, ww, c).permute(0, 3, 1, 2).contiguous()

    return (fetch(L.BUF_SKIP, hq, wq, 32), [fetch(L.BUF_LOW0 + i, hq // 2, wq // 2, 64) for i in range(5)],
            fetch(L.BUF_WORK, hq, wq, 32), fetch(L.BUF_META, hq, wq, 64))


def conv64(x, state, name, slope=0.1):
    """(LeakyReLU of the convolution in 64 bits, its error bound)."""
    w, b = state[name + ".weight"].double(), state[name + ".bias"].double()
    pad, k = w.shape[-1] // 2, w[0].numel()
    y = F.conv2d(x.double(), w, b, padding=pad)
    return leaky(y, slope), 2.0 ** -22 * (3 + 4 * k / 8) * conv_size(x, w, b)


def no_worse(name, got, ref, chains, size, values):
    """The error of all outputs, relative to the magnitude of each one's terms, is at most that of FP32 FMA chains
    (`chains` is what those give), but for chance: 10 % (expand's and the project's largest rounding is the same in
    both, so that their errors come out alike), a factor of 2 for a frame of one value, whose `values` distinct
    outputs are few.  Splits have 0.3 to 0.7 of it; with 6 bits in the lo halves they have more than twice it
    (tests/test_fp32_split_cpu.py)."""
    ours, theirs = rms(got.double() - ref, size), rms(chains.double() - ref, size)
    print(f"  {name}: {ours:.3g} of the terms, FMA chains {theirs:.3g}", flush=True)
    assert ours <= (1.1 if values > 1 else 2) * theirs, name


def check(name, got, ref, bound, chains, size, values):
    """Every output within its bound, and all of them no worse than FMA chains."""
    over = (got.double() - ref).abs() - bound
    assert torch.isfinite(got).all(), name
    assert over.max().item() <= 0, f"{name}: {over.max().item():.3g} over the bound"
    no_worse(name, got, ref, chains, size, values)


def conv_fp32(x, state, name, slope=0.1):
    """The layer with FP32 FMA chains (on the GPU: 64-bit arithmetic on the CPU takes a minute per size)."""
    y = conv_chain(x.cuda(), state[name + ".weight"].cuda(), state[name + ".bias"].cuda()).cpu()
    return torch.where(y >= 0, y, y * slope)


def compare(model, state, frames):
    skip, low, work, meta = stages(model, frames)
    values = frames[0, 0].numel()

    def layer(x, name):
        return (*conv64(x, state, name), conv_fp32(x, state, name), conv_size(x, state[name + ".weight"], state[name + ".bias"]))

    check("compress", low[0], *layer(F.pixel_unshuffle(skip, 2), "compress_270"), values)
    for i in range(1, 5):
        for n, part in (("a", slice(0, 32)), ("b", slice(32, 64))):
            check(f"bottleneck {i}{n}", low[i][:, part], *layer(low[i - 1][:, part], f"bottleneck_270_{n}{i}"), values)
    up, bound, one, size = (F.pixel_shuffle(t, 2) for t in layer(low[4], "expand_270"))
    ref = skip.double() + up
    check("expand", work, ref, bound + 2.0 ** -23 * ref.abs(), skip + one, size + skip.double().abs(), values)
    r, rb, one, size = layer(work, "refine_540")
    w = state["metadata_head.weight"].double()
    ref, tb = conv64(r, state, "metadata_head", slope=1.0)
    check("refine + tail", meta, ref, tb + F.conv2d(rb, w.abs()), conv_fp32(one, state, "metadata_head", slope=1.0),
          conv_size(size, w, state["metadata_head.bias"]), values)


# one tile and less, ragged tiles, tile multiples, many frames (the large-launch variants), long rows, the grouped
# layers' 8-row tiles in one round
SIZES = [(1, 1, 1), (1, 33, 65), (2, 96, 128), (1, 97, 31), (40, 70, 90), (3, 150, 1030), (1, 350, 640)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_stages_against_64_bits(model, size):
    b, h, w = size
    print(f"case: FP32 stages {size}", flush=True)
    compare(*model, torch.rand(b, 3, h, w, generator=torch.Generator().manual_seed(h * w)))


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_project_against_64_bits(model, size):
    """Analysis features and project, against the oracle's FP32 features and FMA chains."""
    b, h, w = size
    m, state = model
    print(f"case: FP32 project {size}", flush=True)
    frames = torch.rand(b, 3, h, w, generator=torch.Generator().manual_seed(h * w))
    skip = stages(m, frames)[0]
    wide = {k: v.double() if torch.is_tensor(v) else v for k, v in state.items()}
    features = lambda x, st: F.pixel_unshuffle(M.rgb_to_feature8(x, st), 2)  # noqa: E731
    exact = features(pad_frame(frames).double(), wide)
    ref = conv64(exact, state, "project_540")[0]
    one = conv_fp32(features(pad_frame(frames), state), state, "project_540")
    size_ = conv_size(exact, state["project_540.weight"], state["project_540.bias"])
    no_worse("project", skip, ref, one, size_, h * w)


@pytest.mark.parametrize("gain", [0.0, 1e-30, 1e-6, 3e5, 1e12])
def test_stages_over_the_range(model, gain):
    """Frames far outside [0, 1]: the scaled splits neither overflow FP16 nor lose the small values."""
    print(f"case: FP32 stages, frame values up to {gain:g}", flush=True)
    frames = gain * (2 * torch.rand(1, 3, 45, 70, generator=torch.Generator().manual_seed(5)) - 1)
    frames[:, :, :20] *= 1e-3                       # tiles that hold both
    compare(*model, frames)


@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan")])
def test_nonfinite_input_stays_local(model, bad):
    """A non-finite pixel makes its own surroundings non-finite and leaves pixels that it cannot reach (32 or
    more away) at their values: it does not enter the scale of the tiles that it lies in."""
    m, _ = model
    print(f"case: FP32 frame with one pixel at {bad}", flush=True)
    frames = torch.rand(1, 3, 80, 150, generator=torch.Generator().manual_seed(7))
    clean = m.run(frames.cuda(), check_finite=False).cpu()
    frames[0, 1, 40, 70] = bad
    got = m.run(frames.cuda(), check_finite=False).cpu()
    with pytest.raises(FloatingPointError):
        m.run(frames.cuda())
    far = torch.ones(160, 300, dtype=torch.bool)
    far[2 * (40 - 32):2 * (40 + 33), 2 * (70 - 32):2 * (70 + 33)] = False
    assert (got - clean).abs()[..., far].max().item() <= 2e-5


# the second size takes the large-launch variants
@pytest.mark.parametrize("size", [(1, 80, 150), (3, 150, 1030)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("value", [1e4, 1e6, 1e8, -1e12, 1e30])
def test_finite_outlier_stays_local(model, size, value):
    """A large finite pixel leaves the pixels that it cannot reach (32 or more away) at their values but for the
    rounding of splits with another scale (2^-22 or so, as between regions of upscale())."""
    m, _ = model
    print(f"case: FP32 frames {size} with one pixel at {value:g}", flush=True)
    b, h, w = size
    frames = torch.rand(b, 3, h, w, generator=torch.Generator().manual_seed(7))
    clean = m.run(frames.cuda(), check_finite=False).cpu()
    y, x = h // 2, w // 2
    frames[b // 2, 1, y, x] = value
    got = m.run(frames.cuda(), check_finite=False).cpu()
    far = torch.ones(b, 1, 2 * h, 2 * w, dtype=torch.bool)
    far[b // 2, :, max(0, 2 * (y - 32)):2 * (y + 33), 2 * (x - 32):2 * (x + 33)] = False
    assert ((got - clean).abs() * far).max().item() <= 4e-6


@pytest.mark.parametrize("size", [(1, 45, 70), (3, 150, 1030)], ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("values", [(30.0,), (500.0, -5e3), (2e4,), (1e8,), (-1e12, 3e5), (1e30, 1e-30, 1e10)], ids=str)
def test_stages_with_outliers(model, size, values):
    """Pixels far apart in magnitude within a tile: every stage within the bound of each pixel's own window."""
    print(f"case: FP32 stages {size} with pixels at {values}", flush=True)
    b, h, w = size
    frames = torch.rand(b, 3, h, w, generator=torch.Generator().manual_seed(9))
    for i, v in enumerate(values):
        frames[0, :, h // 2 + 9 * i, w // 2 - 13 * i] = v
    compare(*model, frames)


def with_weights(R, path, change):
    """(model, folded state) of area's checkpoint with change(layer, weight, bias) for its layers' FP32 weights."""
    from aeisu_amd import artifacts as A
    records, header = A.read_records(A.load_blob(WEIGHTS / "aeisu_area.pt")[0])
    state, arrays = M.load_folded(WEIGHTS / "aeisu_area.pt"), {r[0]: i for i, r in enumerate(records)}
    for layer in A.LAYERS:
        iw, ib = arrays[layer + ".weight_fp32"], arrays[layer + ".bias"]
        w, b = change(layer, torch.from_numpy(records[iw][3]).clone(), torch.from_numpy(records[ib][3]).clone())
        for i, t in ((iw, w), (ib, b)):
            records[i] = (*records[i][:3], t.numpy())
        names = [f"bottleneck_270_{n}{int(layer[-1]) + 1}" for n in "ab"] if layer.startswith("bottleneck") else [A.FOLDED_NAMES[layer]]
        for name, pw, pb in zip(names, w.chunk(len(names)), b.chunk(len(names))):
            state[name + ".weight"], state[name + ".bias"] = pw.contiguous(), pb.contiguous()
    path.write_bytes(A.write(records, **header))
    return R.load_model(path, precision="fp32"), state


def test_weights_over_the_range(R, tmp_path):
    """Layers whose weights and activations are scaled by powers of two that the next layer takes back: the FP32
    policy's arithmetic is the same up to those powers, so the outputs are the same bits."""
    print("case: FP32 policy, layers scaled by 2^-100 to 2^80", flush=True)
    scale, last = {"compress": -50, "bottleneck0": 30, "bottleneck1": -70, "bottleneck2": 10, "bottleneck3": -20, "refine": 45}, {}

    def change(layer, w, b):
        before = {"bottleneck0": "compress", "bottleneck1": "bottleneck0", "bottleneck2": "bottleneck1",
                  "bottleneck3": "bottleneck2", "expand": "bottleneck3", "tail": "refine"}.get(layer)
        own = scale.get(layer, 0)
        return w * 2.0 ** (own - scale.get(before, 0)), b * 2.0 ** own

    m, _ = with_weights(R, tmp_path / "scaled.bin", change)
    frames = torch.rand(2, 3, 70, 90, generator=torch.Generator().manual_seed(2)).cuda()
    plain = R.load_model(WEIGHTS / "aeisu_area.pt", precision="fp32")
    assert torch.equal(m.run(frames), plain.run(frames))


def test_rows_of_small_weights(R, tmp_path):
    """Outputs whose weights are far below their layer's largest: every channel within FP32 error of its own
    magnitude (the 2-norm of its error below 2e-6 of its own; 64 x 2^-24 per sum would be 4e-6)."""
    print("case: FP32 policy, every other output's weights at 2^-30", flush=True)

    def change(layer, w, b):
        if layer not in ("project", "expand"):                # expand is added to skip
            w[1::2] *= 2.0 ** -30
            b[1::2] *= 2.0 ** -30
        return w, b

    m, state = with_weights(R, tmp_path / "rows.bin", change)
    skip, low, work, meta = stages(m, torch.rand(1, 3, 100, 130, generator=torch.Generator().manual_seed(4)))
    pairs = {"compress": (low[0], conv64(F.pixel_unshuffle(skip, 2), state, "compress_270")[0])}
    for i in range(1, 5):
        pairs[f"bottleneck {i}"] = (low[i], torch.cat([conv64(low[i - 1][:, 32 * j:32 * j + 32], state, f"bottleneck_270_{n}{i}")[0]
                                                       for j, n in enumerate("ab")], 1))
    pairs["refine + tail"] = (meta, conv64(conv64(work, state, "refine_540")[0], state, "metadata_head", slope=1.0)[0])
    for name, (got, ref) in pairs.items():
        size = lambda x: x.double().square().sum((0, 2, 3)).sqrt()  # noqa: E731
        worst = (size(got - ref) / size(ref)).max().item()
        print(f"  {name}: worst channel {worst:.3g}", flush=True)
        assert worst <= 2e-6, name


@pytest.mark.parametrize("dtypes", [("f32", "f32"), ("f16", "f32"), ("f32", "f16"), ("f16", "f16")], ids="-".join)
@pytest.mark.parametrize("size", [(1, 1, 1), (1, 4, 64), (2, 5, 65), (1, 7, 31), (1, 33, 130), (3, 250, 331)],
                         ids=lambda s: "x".join(map(str, s)))
def test_head_against_64_bits(model, size, dtypes):
    """The head on the GPU's own coefficients, at ragged widths and heights, in every pair of layouts.  An
    output is 25 filter weights (sums of 16 products of exact parts, of which the 4 MFMA passes at the main terms'
    magnitude cut off up to 2^-24 in each of their 8 terms and the sum, 36 x 2^-24; the base; the clamp rounds a
    coefficient twice) applied to the window (25 roundings): 64 x 2^-24 of the terms, and the output's rounding."""
    from aeisu_amd import _lib as L
    kind = {"f16": torch.float16, "f32": torch.float32}
    m, state = model
    b, h, w = size
    print(f"case: FP32 head {size} {dtypes}", flush=True)
    frames = (1.4 * torch.rand(b, 3, h, w, generator=torch.Generator().manual_seed(h + w)) - 0.2).to(kind[dtypes[0]])
    flags = L.FLAG_KEEP_INTERMEDIATES
    got = m.run(frames.cuda(), out_dtype=kind[dtypes[1]], flags=flags).cpu().double()
    hd = m.handle(b, h, w, kind[dtypes[0]], kind[dtypes[1]], flags)
    _, _, _, _, hq, wq = m.geometry(hd)
    meta = m.intermediate(hd, L.BUF_META).cpu().view(torch.float32).reshape(b, hq, wq, 64).permute(0, 3, 1, 2).double()
    padded = pad_frame(frames).double()
    base, basis = state["base"].double(), state["basis"].double()
    ref = crop_output(M.reconstruct(padded, meta, base, basis), h, w)
    size_ = crop_output(M.reconstruct(padded.abs(), meta.abs(), base.abs(), basis.abs()), h, w)
    bound = 64 * 2.0 ** -24 * size_ + 1e-12
    if dtypes[1] == "f16":
        bound = bound + 2.0 ** -11 * ref.abs() + 2.0 ** -25
    over = (got - ref.clamp(0, 1)).abs() - bound
    assert over.max().item() <= 0, f"{over.max().item():.3g} over the bound"


def head_chain(padded, meta, base, basis, y0, x0, h, w):
    """The head of an h x w frame at (y0, x0) of its padded grid with one FP32 FMA chain per filter weight (the
    base added last) and per output."""
    c = F.pixel_shuffle(meta.view(meta.shape[0], 4, 16, *meta.shape[2:]).transpose(1, 2).flatten(1, 2), 2)
    c = c[..., y0:y0 + h, x0:x0 + w]
    mag = c.abs()
    c = torch.where(mag <= 2, c, torch.sign(c) * (2 + 0.05 * (mag - 2)).clamp(max=2.5))
    src = padded[..., y0 - 2:y0 + h + 2, x0 - 2:x0 + w + 2]
    phases = []
    for ph in range(4):
        u = torch.zeros(c.shape[0], 3, h, w)
        for tap in range(25):
            wt = chain(torch.zeros(c.shape[0], 1, h, w), ((c[:, k:k + 1], basis[tap, k, ph]) for k in range(16)))
            wt = wt + base[tap, ph]
            u = chain(u, [(wt, src[..., tap // 5:tap // 5 + h, tap % 5:tap % 5 + w])])
        phases.append(u)
    return F.pixel_shuffle(torch.stack(phases, 2).flatten(1, 2), 2).clamp(0, 1)


def test_head_no_further_from_64_bits_than_fma_chains(model):
    """The error over a whole frame, not only a bound of every value: its norm is at most that of FP32 FMA chains
    (0.91 to 0.93 of it on the GPU), and its mean at most a tenth of its root mean square, a share of 0.5 % of the
    norm.  Sums that all cut bits off in one direction have a mean of a quarter of it."""
    from aeisu_amd import _lib as L
    from aeisu_amd import frames as scenes
    m, state = model
    h, w = 150, 150
    print("case: FP32 head against FMA chains", flush=True)
    frames = scenes.scene(h, w, 11, texture=True)[None].float()
    flags = L.FLAG_KEEP_INTERMEDIATES
    got = m.run(frames.cuda(), flags=flags).cpu()
    hd = m.handle(1, h, w, torch.float32, torch.float32, flags)
    _, _, _, _, hq, wq = m.geometry(hd)
    meta = m.intermediate(hd, L.BUF_META).cpu().view(torch.float32).reshape(1, hq, wq, 64).permute(0, 3, 1, 2)
    padded = pad_frame(frames)
    ref = crop_output(M.reconstruct(padded.double(), meta.double(), state["base"].double(), state["basis"].double()), h, w).clamp(0, 1)
    one = head_chain(padded, meta, state["base"], state["basis"], 16 + -h % 32 // 2, 16 + -w % 32 // 2, h, w)
    ours, theirs = got.double() - ref, one.double() - ref
    print(f"  error norm {ours.norm():.4g}, FMA chains {theirs.norm():.4g}; mean {ours.mean():.3g}, {theirs.mean():.3g}", flush=True)
    assert ours.norm() <= theirs.norm()
    assert ours.mean().abs() <= 0.1 * ours.square().mean().sqrt()
