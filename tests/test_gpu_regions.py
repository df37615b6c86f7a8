"""upscale() with tiles joined into regions, and its copy to the host, against the whole frame and .cpu()."""
from __future__ import annotations

import pytest
import torch

from tests._util import WEIGHTS

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def R(gpu):
    from aeisu_amd import runtime
    return runtime


FILES = {"fp16": "aeisu_area.pt", "fp32": "aeisu_area.pt", "mixed": "aeisu_area_mixed_fp8.bin", "int8": "aeisu_int8_fp16.pt"}


@pytest.mark.parametrize("precision", sorted(FILES))
@pytest.mark.parametrize("size,tile,region", [((70, 90), 32, 64), ((97, 161), 32, 96), ((33, 300), 64, 128), ((64, 64), 96, 32),
                                              ((70, 90), 32, 2048), ((1, 1), 32, 32)])
def test_regions_equal_whole(R, monkeypatch, precision, size, tile, region):
    """Regions of one or several tiles, cut inside the frame, in its padding and with cores that hold padding
    only, against one run of the whole frame: the per-pixel arithmetic is the same but for the FP32 policy's
    tile scales, whose rounding moves an output by at most some 2^-22."""
    print(f"case: {precision} {size} tile {tile} region {region}", flush=True)
    monkeypatch.setattr(R, "_REGION", region)
    model = R.load_model(WEIGHTS / FILES[precision], precision=precision)
    src = torch.rand(3, *size, generator=torch.Generator().manual_seed(3))
    whole, got = R.upscale(model, src, 0), R.upscale(model, src, tile)
    assert got.shape == (3, 2 * size[0], 2 * size[1]) and got.device.type == "cpu" and got.dtype == torch.float32
    assert (whole - got).abs().max().item() <= (4e-6 if precision == "fp32" else 0)
    bad = src.clone()
    bad[0, size[0] // 2, size[1] // 2] = float("nan")
    with pytest.raises(FloatingPointError):
        R.upscale(model, bad, tile)


@pytest.mark.parametrize("size", [(150, 333), (65, 500), (200, 60)])
def test_one_scratch_for_all_regions(R, monkeypatch, size):
    """Every region of an image has the same shape, at the edges too: one geometry, and the scratch of one region of
    at most the region's side and its halo."""
    print(f"case: regions of {size}", flush=True)
    monkeypatch.setattr(R, "_REGION", 64)
    model = R.load_model(WEIGHTS / "aeisu_area.pt", precision="fp32")
    R.upscale(model, torch.rand(3, *size, generator=torch.Generator().manual_seed(6)), 32)
    other = R.load_model(WEIGHTS / "aeisu_area.pt", precision="fp32")
    other.run(torch.rand(1, 3, 128, 128, device="cuda"), pad=False)
    assert model.persistent_bytes() <= other.persistent_bytes()


def test_small_tiles_take_less_scratch(R):
    """A caller short of memory still has it with a smaller tile."""
    print("case: scratch of upscale() by tile", flush=True)
    src = torch.rand(3, 700, 1100, generator=torch.Generator().manual_seed(8))
    used = {}
    for tile in (32, 64, 128):
        model = R.load_model(WEIGHTS / "aeisu_area.pt", precision="fp32")
        weights = model.persistent_bytes()
        R.upscale(model, src, tile)
        used[tile] = model.persistent_bytes() - weights
    assert used[32] < used[64] < used[128]
    assert used[32] <= 576 * 576 * 200


@pytest.mark.parametrize("numel", [1, 2 << 20, (2 << 20) + 1, (4 << 20) + 3, 9_000_001])
def test_copy_to_host(R, numel):
    """One chunk and less, chunk boundaries and a short last chunk; results are ordinary pageable tensors."""
    x = torch.rand(numel, device="cuda")
    got = R._to_host(x)
    assert not got.is_pinned() and torch.equal(got, x.cpu())
