"""Weight gradients whose workgroups take two, three and more units, so that their
sums go to memory halfway (layers with 64 outputs per workgroup; 16 samples of 128
x 128 give 192 -> 64 three units a workgroup, 288 -> 128 three, 64 -> 64 one).
Against the mean of the samples' gradients, whose workgroups take one unit or two;
tolerance as in test_gpu_unet_dw.py for a batch that is a power of two."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_unet import note, perturbed_params, sample

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,B", [(128, 128, 8), (128, 128, 16), (256, 128, 16), (256, 256, 16)])
def test_sums_in_two_halves(H, W, B):
    note("weight gradients in halves %dx%d batch %d" % (H, W, B))
    terrain, params, target = sample(H + 3 * W, B, H, W)
    with fa.UNet(H, W, max_batch=B, seed=43) as net:
        net.set_params(perturbed_params(net, 44))
        g = net.loss_grad(terrain, params, target)[1].astype(np.float64)
        mean = np.mean([net.loss_grad(terrain[b:b + 1], params[b:b + 1], target[b:b + 1])[1]
                        .astype(np.float64) for b in range(B)], axis=0)
        layers = net.layers()
    off = 0
    for i, (ci, co, _) in enumerate(layers):
        for what, n in (("W", 9 * ci * co), ("b", co)):
            a, m = g[off:off + n], mean[off:off + n]
            off += n
            assert np.linalg.norm(a - m) <= 2e-4 * np.linalg.norm(m), (i, what)
