"""The strip sweep (OU_SWEEP_TILES in 2D up to 10 moments) where it can go wrong:
one strip and a ring of several, strips with one column left over, strips shorter
than a phase, groups of several rounds, empty direction slots, and materials that
change along a strip.

Bar: the sums are formed in the level sweep's order, so at equal direction groups
the results equal the level launches bit for bit.  Every case sweeps twice: the
second sweep meets the first one's words in the ring."""
import numpy as np
import pytest

import ouranos_amd as ou
from ouranos_amd import problems as P

pytestmark = pytest.mark.gpu


def _strip(n, p, prec, L, block=None):
    quad = ou.Quadrature(ou.PRODUCT_GLC, 2, n_polar=8, n_azim=20, L_max=L)
    i, j = np.meshgrid(np.arange(n[0]), np.arange(n[1]), indexing="xy")
    b = block or max(n)
    mat = (i // b + -(-n[0] // b) * (j // b)).reshape(-1)
    sigma_t = np.random.default_rng(5).uniform(1.0, 10.0, mat.max() + 1)
    sigma_s = np.stack([0.5 * sigma_t * 0.5 ** l for l in range(L + 1)], 1)
    return ou.RadiativeTransfer(2, p, n, [1.0 / max(n)] * 2, quad, sigma_t, sigma_s, mat,
                                precision=prec)


def _both(op, shape, x):
    op.sweep_mode = ou.SWEEP_TILES
    op.sweep_shape = shape
    op.Apply(-x)
    tiles = op.Apply(x)
    op.sweep_mode = ou.SWEEP_LEVELS
    op.sweep_shape = (4, shape[1])
    return tiles, op.Apply(x)


@pytest.mark.parametrize("prec", [ou.FP64, ou.FP32], ids=["fp64", "fp32"])
@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("n,L,block", [((1, 1), 0, None), ((9, 1), 1, None), ((1, 9), 0, None),
                                       ((7, 17), 1, None), ((8, 8), 3, None), ((17, 9), 3, None),
                                       ((24, 40), 3, 8), ((40, 16), 1, 8)])
def test_strips_equal_levels(n, L, block, p, prec):
    op = _strip(n, p, prec, L, block=block)
    x = np.random.default_rng(3).standard_normal(op.n)
    ran = 0
    for shape in [(1, 1), (2, 1), (2, 3), (4, 1), (4, 2)]:
        try:
            op.sweep_mode = ou.SWEEP_TILES
            op.sweep_shape = shape
        except ou.OuError:
            assert shape[0] == 4 and p == 2 and prec == ou.FP64  # 2 step waves at most
            continue
        tiles, levels = _both(op, shape, x)
        assert np.array_equal(tiles, levels), shape
        ran += 1
    assert ran >= 3
    op.close()


def test_strip_wait_limit():
    """Without any time to wait a sweep of several strips reports the timeout and
    ends; with its limit back the plan sweeps as before."""
    op = P.hetero_2d(n=64, block=8, n_polar=4, n_azim=8, L=1).operator(ou.FP64)
    assert op.sweep_mode == ou.SWEEP_TILES
    x = np.random.default_rng(3).standard_normal(op.n)
    y = op.Apply(x)
    op.set_sweep_wait_limit(0.0)
    with pytest.raises(ou.OuError) as e:
        op.Apply(x)
    assert e.value.code == -8  # OU_ERR_TIMEOUT
    op.set_sweep_wait_limit(10.0)
    assert np.array_equal(op.Apply(x), y)
    op.close()
