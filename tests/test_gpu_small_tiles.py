"""The quantized policies' small body tiles (8x8 and 12x12 low pixels, compress exchange) against the per-layer
path, bit for bit: one tile and less, the largest frames of each tile side, ragged grids, batches, both frame
layouts, with the exchange and with every tile on its fallback."""
from __future__ import annotations

import pytest
import torch

from tests._util import WEIGHTS

pytestmark = pytest.mark.gpu

FILES = {"mixed": "aeisu_area_mixed_fp8.bin", "mixed-fp8mma": "aeisu_area_mixed_fp8.bin", "int8": "aeisu_int8_fp16.pt"}


@pytest.mark.parametrize("precision", sorted(FILES))
@pytest.mark.parametrize("b,h,w,tile", [(1, 1, 1, 8), (1, 48, 64, 8), (2, 70, 102, 8), (3, 33, 200, 8), (1, 20, 2000, 8),
                                        (1, 480, 480, 8), (1, 512, 480, 12), (2, 240, 426, 12), (1, 100, 2300, 12), (1, 480, 854, 12)])
def test_small_tiles_equal_layers(gpu, precision, b, h, w, tile):
    from aeisu_amd import _lib as L
    from aeisu_amd.runtime import load_model
    model = load_model(WEIGHTS / FILES[precision], precision=precision)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    for dtype in (torch.float16, torch.float32):
        frames = torch.rand(b, 3, h, w, generator=torch.Generator().manual_seed(h * w)).to(dtype).cuda()
        want = model.run(frames, flags=L.FLAG_UNFUSED)
        for flags in (0, L.FLAG_BODY_EXCHANGE_FALLBACK):
            print(f"case: {precision} {b}x{h}x{w} {dtype} flags {flags}", flush=True)
            hd = model.handle(b, h, w, dtype, dtype, flags)
            if cus == 256:
                assert int(hd.report().split("body_exchange_tile=")[1].split()[0]) == tile
            for _ in range(3):                       # the exchange's counters grow from launch to launch
                assert torch.equal(model.run(frames, flags=flags), want)
