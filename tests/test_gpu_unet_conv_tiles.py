"""Forward and data-gradient convolutions of the U-Net at the edges of their voxel tiles:
partial tiles of one to four 16-voxel rows, z runs, several lines a tile, the parity classes
of odd grids, K steps with chunks past the last tap, split and whole reductions."""
import numpy as np
import pytest
import torch

from oracle import unet_ref as U

pytestmark = pytest.mark.gpu


def _shifting_params(ref):
    """Each channel is passed on through a tap of its own (all 27 in use from 32 channels on,
    every axis and sign from 8), zero biases."""
    p = []
    for i, l in enumerate(ref.L):
        cin, cout = l[2], l[5]
        W = np.zeros((27, cin, cout))
        for k in range(max(cin, cout)):
            W[(13 + i + 5 * k) % 27, k % cin, k % cout] = 1.0
        p += [W.reshape(-1), np.zeros(cout)]
    return np.concatenate(p)


@pytest.mark.parametrize("grid,base,batch", [((5, 5, 5), 8, 1), ((17, 17, 17), 8, 4), ((33, 33, 33), 8, 1),
                                             ((9, 33, 17), 8, 3), ((5, 5, 133), 24, 1), ((33, 17, 9), 24, 2)])
def test_gpu_unet_conv_tiles(grid, base, batch):
    """Weights of 0 and 1 and small integers as inputs: activations up to 256 are exact in
    BF16 and their sums in FP32, so the forward pass equals the oracle to the bit.  The data
    gradients are rounded to BF16 once per layer, by at most one place (2^-8) apart; 2e-2
    covers five such layers in a row, and a misplaced tap or voxel is an error of order one."""
    from platoanalyze_amd.unet import UNet

    print(f"case: unet convolution tiles {grid} base {base} batch {batch}", flush=True)
    ref = U.UNetRef(grid, base)
    p = _shifting_params(ref)
    net = UNet(grid, base)
    net.set_params(torch.from_numpy(p.astype(np.float32)))
    rng = np.random.default_rng(7)
    V = int(np.prod(grid))
    x = rng.integers(0, 3, (batch, V, U.IN_CH)).astype(np.float32)
    t = rng.integers(0, 13, (batch, V, U.OUT_CH)).astype(np.float32)
    y_ref, acts = ref.forward(x.astype(np.float64), p)
    assert max(float(np.abs(a).max()) for a in acts if a is not None) <= 256
    assert np.count_nonzero(y_ref) > y_ref.size // 20
    xt = torch.from_numpy(x).reshape(batch, *grid, U.IN_CH).cuda()
    tt = torch.from_numpy(t).reshape(batch, *grid, U.OUT_CH).cuda()
    y = net.forward(xt).cpu().numpy().reshape(y_ref.shape)
    assert np.array_equal(y, y_ref.astype(np.float32))
    loss_ref, g_ref, _ = ref.loss_grad(x.astype(np.float64), t.astype(np.float64), p)
    loss, g = net.gradient(xt, tt)
    assert abs(loss - loss_ref) <= 1e-6 * abs(loss_ref)
    g = g.cpu().numpy()
    off = 0
    for k, l in enumerate(ref.L):
        for n in (27 * l[2] * l[5], l[5]):
            a, b = g[off:off + n], g_ref[off:off + n]
            off += n
            assert float(np.linalg.norm(a - b)) <= 2e-2 * float(np.linalg.norm(b)), k
