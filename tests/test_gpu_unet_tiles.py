"""The U-Net's convolution takes more output tiles per wave where there are enough
positions: 8 samples at 32^3 run the wide kernels (2 position tiles, 2 and 3 channel
tiles), one sample the narrow ones.

Bar: an output's products are summed in the same order in all of them, so a batch
predicts each sample bit for bit as that sample alone.  The gradient of the mean loss
is the mean of the samples' gradients: with 8 samples the factor 1/8 is exact in BF16,
so only FP32 sums over positions are ordered differently (chains of a few thousand
terms, sqrt(4096) * 2^-24 = 4e-6 of the norm; bar 2e-5)."""
import numpy as np
import pytest

import ouranos_amd as ou

pytestmark = pytest.mark.gpu


def test_wide_and_narrow_tiles_agree():
    B, G = 8, 32
    rng = np.random.default_rng(4)
    feat = np.zeros((B, G ** 3, 12), np.float32)
    feat[..., 0:10] = rng.standard_normal((B, G ** 3, 10))
    feat[..., 10] = 1.0
    target = rng.standard_normal((B, G ** 3, 8)).astype(np.float32)
    net = ou.UNet(grid=G, max_batch=B, seed=11)
    rest = net.get_params()
    head = slice(rest.size - 264, rest.size)  # so that the head is not zero
    rest[head] = rng.normal(scale=0.1, size=264)
    net.set_params(rest)
    out = net.predict(feat)
    _, grad = net.loss_grad(feat, target)
    mean = np.zeros_like(grad, dtype=np.float64)
    for b in range(B):
        assert np.array_equal(net.predict(feat[b:b + 1])[0], out[b])
        mean += np.asarray(net.loss_grad(feat[b:b + 1], target[b:b + 1])[1], np.float64) / B
    assert np.linalg.norm(mean) > 0
    assert np.linalg.norm(grad - mean) <= 2e-5 * np.linalg.norm(mean)
    net.close()
