"""Convolutions too wide for a tile in LDS (640 channels on lines of 8 voxels and more): the
kernel without staging, with its reduction split over work-groups and whole."""
import numpy as np
import pytest
import torch

from oracle import unet_ref as U
from test_gpu_unet_conv_tiles import _shifting_params, test_gpu_unet_conv_tiles as check_against_oracle

pytestmark = pytest.mark.gpu

GRID, BASE = (5, 5, 57), 80  # bottleneck 1x1x8 voxels of 640 channels


def test_gpu_unet_wide_split():
    """Forward and gradients of one sample: every wide convolution is split over work-groups."""
    check_against_oracle(GRID, BASE, 1)


def test_gpu_unet_wide_whole():
    """110 samples: the 640 -> 320 decoder convolution has waves enough for whole sums.  The
    sums of small integers are exact, so each sample equals its own forward pass to the bit."""
    from platoanalyze_amd.unet import UNet

    print(f"case: wide unet {GRID} base {BASE} batch 110", flush=True)
    net = UNet(GRID, BASE)
    net.set_params(torch.from_numpy(_shifting_params(U.UNetRef(GRID, BASE)).astype(np.float32)))
    rng = np.random.default_rng(9)
    x = torch.from_numpy(rng.integers(0, 3, (3, *GRID, U.IN_CH)).astype(np.float32)).cuda()
    one = [net.forward(x[k:k + 1].contiguous()).clone() for k in range(3)]
    y = net.forward(x.repeat(37, 1, 1, 1, 1)[:110].contiguous())
    assert int(torch.count_nonzero(one[0])) > one[0].numel() // 20
    for k in range(110):
        assert torch.equal(y[k], one[k % 3][0]), k
