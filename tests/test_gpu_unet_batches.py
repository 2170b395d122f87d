"""The convolution takes 16 x 8 pixel tiles per wave where there are enough of
them and 16 x 2 ones elsewhere, so a sample's output comes from other tiles
alone than in a batch.  Every accumulator adds the same products in the same
order at either height, so the outputs are the same bits; sizes whose deep
levels are narrower than a tile or no multiple of it among them."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_unet import note, perturbed_params, sample

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,B", [(32, 32, 64), (32, 96, 40), (96, 160, 24), (160, 64, 24),
                                   (256, 256, 16)])
def test_a_batch_gives_each_samples_bits(H, W, B):
    note("unet batch %d of %dx%d against single samples" % (B, H, W))
    terrain, params, _ = sample(H * W, B, H, W)
    with fa.UNet(H, W, max_batch=B, seed=31) as net:
        net.set_params(perturbed_params(net, 32))
        y = net.forward(terrain, params)
        for b in (0, 1, B // 2, B - 1):
            one = net.forward(terrain[b:b + 1], params[b:b + 1])
            np.testing.assert_array_equal(one[0], y[b])


@pytest.mark.parametrize("H,W", [(32, 32), (64, 64), (96, 224), (128, 128), (256, 256)])
def test_batches_on_either_side_of_the_single_waves(H, W):
    """Levels with up to a wave per CU go to single waves, larger ones to
    workgroups: batches from one sample on pass that line level by level."""
    note("unet batches 1, 2, 3, 5, 8 of %dx%d" % (H, W))
    terrain, params, _ = sample(H + W, 8, H, W)
    with fa.UNet(H, W, max_batch=8, seed=33) as net:
        net.set_params(perturbed_params(net, 34))
        y = net.forward(terrain, params)
        for B in (1, 2, 3, 5):
            np.testing.assert_array_equal(net.forward(terrain[:B], params[:B]), y[:B])
