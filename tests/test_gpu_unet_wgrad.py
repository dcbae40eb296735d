"""Weight and bias gradients of the U-Net at the edges of their tiles: 8-channel tails,
24 channels (one and a half blocks), z runs of more than one tile, the smallest grid."""
import numpy as np
import pytest
import torch

from oracle import unet_ref as U

pytestmark = pytest.mark.gpu


def _copying_params(ref):
    """Weights that pass channels on unchanged through the centre tap (input channel ci to
    the output channels equal to it modulo the smaller width), zero biases."""
    p = []
    for l in ref.L:
        cin, cout = l[2], l[5]
        W = np.zeros((27, cin, cout))
        for k in range(max(cin, cout)):
            W[13, k % cin, k % cout] = 1.0
        p += [W.reshape(-1), np.zeros(cout)]
    return np.concatenate(p)


@pytest.mark.parametrize("grid,base,batch", [((5, 5, 5), 8, 1), ((9, 13, 5), 24, 2), ((5, 5, 133), 8, 1),
                                             ((5, 37, 9), 16, 3), ((17, 17, 17), 8, 2)])
def test_gpu_unet_wgrad_tiles(grid, base, batch):
    """Every layer against the NumPy oracle on a network whose activations are small
    integers and whose data gradients are sums of few BF16 values, so no activation or
    gradient is rounded differently on the two sides and only the FP32 sums over up to
    10000 voxels differ: sqrt(1e4) 2^-24 of the terms' sum is 6e-6, 1e-4 leaves room for
    cancellation.  The sums are ordered: a second call gives the same bits."""
    from platoanalyze_amd.unet import UNet

    print(f"case: unet weight gradients {grid} base {base} batch {batch}", flush=True)
    ref = U.UNetRef(grid, base)
    p = _copying_params(ref)
    net = UNet(grid, base)
    net.set_params(torch.from_numpy(p.astype(np.float32)))
    rng = np.random.default_rng(11)
    V = int(np.prod(grid))
    x = rng.integers(1, 4, (batch, V, U.IN_CH)).astype(np.float32)
    y = rng.integers(0, 13, (batch, V, U.OUT_CH)).astype(np.float32)
    loss_ref, g_ref, _ = ref.loss_grad(x.astype(np.float64), y.astype(np.float64), p)
    xt = torch.from_numpy(x).reshape(batch, *grid, U.IN_CH).cuda()
    yt = torch.from_numpy(y).reshape(batch, *grid, U.OUT_CH).cuda()
    loss, g = net.gradient(xt, yt)
    assert abs(loss - loss_ref) <= 1e-6 * abs(loss_ref)
    _, again = net.gradient(xt, yt)
    assert torch.equal(g, again)
    g = g.cpu().numpy()
    off = 0
    for k, l in enumerate(ref.L):
        for n, what in ((27 * l[2] * l[5], "weights"), (l[5], "biases")):
            a, b = g[off:off + n], g_ref[off:off + n]
            off += n
            assert np.linalg.norm(b) > 0, (k, what)
            err = float(np.linalg.norm(a - b) / np.linalg.norm(b))
            assert err < 1e-4, (k, what, err)
