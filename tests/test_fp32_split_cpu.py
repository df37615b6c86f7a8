"""What the FP32 policy's stage tests can see, on the CPU: hi / lo splits hold the limit that test_gpu_fp32_split.py sets
(the error of FP32 FMA chains) and splits that lost bits do not."""
from __future__ import annotations

import pytest
import torch
from torch.nn import functional as F

from oracle import model as M
from tests._fp32 import conv_chain, conv_size, conv_split, leaky, rms
from tests._util import WEIGHTS, pad_frame


@pytest.fixture(scope="module", params=["aeisu_area", "aeisu_div2k_l1"])
def state(request):
    return M.load_folded(WEIGHTS / f"{request.param}.pt")


@pytest.fixture(scope="module")
def work(state):
    """The refine layer's input for a random frame, and compress's."""
    x = pad_frame(torch.rand(1, 3, 33, 65, generator=torch.Generator().manual_seed(1)))
    skip = M.leaky(M.conv(F.pixel_unshuffle(M.rgb_to_feature8(x, state), 2), state, "project_540"))
    return skip, F.pixel_unshuffle(skip, 2)


def layer(state, name):
    return state[name + ".weight"], state[name + ".bias"]


def test_one_layer(state, work):
    for name, x in (("refine_540", work[0]), ("compress_270", work[1])):
        w, b = layer(state, name)
        ref, size = F.conv2d(x.double(), w.double(), b.double(), padding=w.shape[-1] // 2), conv_size(x, w, b)
        limit = rms(conv_chain(x, w, b).double() - ref, size)
        assert rms(conv_split(x, w, b).double() - ref, size) <= 0.8 * limit
        for bits in (0, 3, 6):
            assert rms(conv_split(x, w, b, bits).double() - ref, size) > 2 * limit, (name, bits)


def test_refine_and_tail(state, work):
    """A tail or a refine layer without its lo halves shows in the coefficients."""
    (w, b), (tw, tb), x = layer(state, "refine_540"), layer(state, "metadata_head"), work[0]
    r = F.conv2d(x.double(), w.double(), b.double(), padding=1)
    ref = F.conv2d(leaky(r), tw.double(), tb.double())
    size = conv_size(conv_size(x, w, b), tw, tb)
    limit = rms(conv_chain(leaky(conv_chain(x, w, b)), tw, tb).double() - ref, size)
    error = lambda refine, tail: rms(conv_split(leaky(conv_split(x, w, b, refine)), tw, tb, tail).double() - ref, size)  # noqa: E731
    assert error(11, 11) <= 0.8 * limit
    for refine, tail in ((0, 11), (11, 0), (0, 0), (3, 11), (11, 3)):
        assert error(refine, tail) > 2 * limit, (refine, tail)
