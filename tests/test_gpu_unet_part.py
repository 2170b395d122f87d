"""A batch whose weight gradients take more chunks than those of the largest batch
(352 x 352: level 2 is 88 x 88, 65 chunks for 22 samples, 64 for 32).  The weight
gradients are the same bits as those of a network made for that batch: no sum's
order depends on max_batch."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_unet import note, perturbed_params, sample

pytestmark = pytest.mark.gpu


def test_smaller_batch_with_more_chunks():
    H = W = 352
    B = 22
    note("352x352, 22 of up to 32 samples")
    terrain, params, target = sample(5, B, H, W)
    out = []
    for max_batch in (32, B):
        with fa.UNet(H, W, max_batch=max_batch, seed=3) as net:
            net.set_params(perturbed_params(net, 4))
            out.append(net.loss_grad(terrain, params, target)[1])
            layers = net.layers()
    off = 0
    for i, (ci, co, _) in enumerate(layers):
        n = 9 * ci * co
        np.testing.assert_array_equal(out[0][off:off + n], out[1][off:off + n], err_msg=str(i))
        assert np.any(out[0][off:off + n] != 0)
        off += n + co
