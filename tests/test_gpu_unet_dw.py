"""The weight-gradient kernel's split of the pixels: strips that do not pair up,
levels that leave some workgroups no unit, one sample and many, sizes whose
levels go to it and to the per-tap kernel.  Gradients of a batch are the mean of
its samples' gradients, which come from other strips and chunks: the sums differ
by their order alone.  Each of the up to n = B*H*W products added in FP32 costs
at most one rounding of the running sum, so a gradient is off by at most n *
2^-24 of the sum of its terms' magnitudes in the worst case and by about sqrt(n)
* 2^-24 in practice: 2e-4 of the layer's norm bounds n = 1e6."""
import numpy as np
import pytest

import fastscape_amd as fa
from test_gpu_unet import note, perturbed_params, sample

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,W,B", [(32, 32, 3), (32, 96, 5), (64, 160, 7), (96, 64, 2),
                                   (224, 32, 3), (128, 128, 9)])
def test_batch_gradient_is_the_mean_of_the_samples(H, W, B):
    note("weight gradients %dx%d batch %d" % (H, W, B))
    terrain, params, target = sample(H + 7 * W, B, H, W)
    with fa.UNet(H, W, max_batch=B, seed=41) as net:
        net.set_params(perturbed_params(net, 42))
        loss, g = net.loss_grad(terrain, params, target)
        ones = [net.loss_grad(terrain[b:b + 1], params[b:b + 1], target[b:b + 1])
                for b in range(B)]
        layers = net.layers()
    assert abs(loss - np.mean([o[0] for o in ones])) <= 1e-5 * abs(loss)
    mean = np.mean([o[1].astype(np.float64) for o in ones], axis=0)
    off = 0
    for i, (ci, co, _) in enumerate(layers):
        for what, n in (("W", 9 * ci * co), ("b", co)):
            a, m = g[off:off + n].astype(np.float64), mean[off:off + n]
            off += n
            # activations' gradients are rounded to BF16 at scale 1/B, so they
            # differ from the samples' by their own roundings unless B is a
            # power of two: 2^-8 a value, averaging out over the pixels
            tol = 2e-4 if B & (B - 1) == 0 else 2e-2
            assert np.linalg.norm(a - m) <= tol * np.linalg.norm(m), (i, what)


@pytest.mark.parametrize("H,W,B", [(32, 32, 1), (32, 96, 5), (256, 256, 9)])
def test_loss_and_head_bias_against_64_bits(H, W, B):
    """Sums over all pixels, in FP32: a term is rounded three times, and is part
    of at most (terms of a thread + 6 shuffles + 3 + one addition per workgroup,
    at most 2048) additions: that many times 2^-24 of the sum of magnitudes."""
    note("loss %dx%d batch %d" % (H, W, B))
    terrain, params, target = sample(2 * H + W, B, H, W)
    with fa.UNet(H, W, max_batch=B, seed=43) as net:
        net.set_params(perturbed_params(net, 44))
        y = net.forward(terrain, params).astype(np.float64).ravel()
        loss, g = net.loss_grad(terrain, params, target)
    M = B * H * W
    e = y - target.astype(np.float64).ravel()
    groups = min((4 * M + 255) // 256, 2048)
    eps = (3 + -(-4 * M // (256 * groups)) + 9 + groups) * 2.0 ** -24
    assert abs(loss - np.sum(e * e) / M) <= eps * np.sum(e * e) / M
    assert abs(g[-1] - np.sum(2 * e) / M) <= eps * np.sum(2 * np.abs(e)) / M


@pytest.mark.parametrize("H,W", [(32, 64), (256, 256)])
def test_calls_after_each_other_keep_their_targets(H, W):
    """Targets and gradients are copied beside the kernels: every call of a
    sequence with changing batches and targets gives what it gives on a new
    network (the same kernels on the same inputs; sums by atomics, a handful of
    whose orders differ, agree within 1e-5 of a layer's norm)."""
    note("loss and gradients in sequence %dx%d" % (H, W))
    calls = [(4, 1), (1, 2), (4, 3), (3, 4), (4, 1)]
    with fa.UNet(H, W, max_batch=4, seed=45) as net:
        p0 = perturbed_params(net, 46)
        net.set_params(p0)
        got = []
        for B, k in calls:
            terrain, params, target = sample(k, B, H, W)
            got.append(net.loss_grad(terrain, params, k * target))
    for (B, k), (loss, g) in zip(calls, got):
        terrain, params, target = sample(k, B, H, W)
        with fa.UNet(H, W, max_batch=4, seed=45) as net:
            net.set_params(p0)
            l1, g1 = net.loss_grad(terrain, params, k * target)
        assert abs(loss - l1) <= 1e-5 * abs(l1)
        assert np.linalg.norm(g - g1) <= 1e-5 * np.linalg.norm(g1)
