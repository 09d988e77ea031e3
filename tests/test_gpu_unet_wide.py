"""The U-Net's convolution where a wave takes two tiles of output channels: the
64-channel layers, from 131072 positions on (two samples at 64^3, both signs of each;
with four samples also two tiles of positions).

Bar: an output's products are summed in the same order however many tiles a wave takes,
so a batch predicts each sample bit for bit as that sample alone."""
import numpy as np
import pytest

import ouranos_amd as ou

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,B", [(60, 4), (64, 2), (64, 4)])
def test_two_channel_tiles_agree_with_one(G, B):
    rng = np.random.default_rng(7)
    feat = np.zeros((B, G ** 3, 12), np.float32)
    feat[..., 0:10] = rng.standard_normal((B, G ** 3, 10), dtype=np.float32)
    feat[..., 10] = 1.0
    net = ou.UNet(grid=G, max_batch=B, seed=12)
    params = net.get_params()
    head = slice(params.size - 264, params.size)  # so that the head is not zero
    params[head] = rng.normal(scale=0.1, size=264)
    net.set_params(params)
    out = net.predict(feat)
    assert np.linalg.norm(out) > 0
    for b in range(B):
        assert np.array_equal(net.predict(feat[b:b + 1])[0], out[b]), b
    net.close()
