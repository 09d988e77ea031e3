"""The strip sweep (OU_SWEEP_TILES in 2D up to 10 moments) at the edges of what it
accepts: direction groups without directions, and a source that overflows.

Bar: the sums are formed in the level sweep's order, so at equal direction groups the
results equal the level launches bit for bit, whatever an earlier shape or mode left in
the partial moments."""
import numpy as np
import pytest

import ouranos_amd as ou
from ouranos_amd import problems as P

pytestmark = pytest.mark.gpu

PRECISIONS = pytest.mark.parametrize("prec", [ou.FP64, ou.FP32], ids=["fp64", "fp32"])


class _Subset:
    """Some directions of a quadrature (the operator takes any omega / M2D / D2M)."""

    def __init__(self, q, keep):
        self.omega = np.ascontiguousarray(q.omega[keep])
        self.M2D = np.ascontiguousarray(q.M2D[keep])
        self.D2M = np.ascontiguousarray(q.D2M[:, keep])
        self.mom_l = q.mom_l
        self.most_normal = np.ascontiguousarray(q.most_normal[:, keep])
        self.weight_sum = q.weight_sum
        self.n_dir = int(self.omega.shape[0])
        self.n_mom = q.n_mom


def _operator(quad, p, prec, n=(21, 10), h=0.05):
    L = int(quad.mom_l.max())
    sigma_t = np.array([2.0])
    sigma_s = np.array([[1.0 * 0.5 ** l for l in range(L + 1)]])
    return ou.RadiativeTransfer(2, p, n, [h] * 2, quad, sigma_t, sigma_s,
                                np.zeros(n[0] * n[1], np.int32), precision=prec)


def _quads():
    glc = lambda a, b, L: ou.Quadrature(ou.PRODUCT_GLC, 2, n_polar=a, n_azim=b, L_max=L)
    full = glc(8, 16, 1)  # 16 directions per quadrant; one is left in the (-,-) quadrant
    minus = np.flatnonzero((full.omega[:, 0] < 0) & (full.omega[:, 1] < 0))
    keep = np.setdiff1d(np.arange(full.n_dir), minus[1:])
    # quadrature, groups, groups of the level sweep before it
    return {"4_in_3_groups": (glc(4, 8, 1), 3, 2), "4_in_8_groups": (glc(4, 8, 3), 8, 2),
            "6_in_4_groups": (ou.Quadrature(ou.LS, 2, sn=6, L_max=0), 4, 2),
            "9_in_4_groups": (glc(6, 12, 1), 4, 2),
            "1_and_16_in_4_groups": (_Subset(full, keep), 4, 5)}


@PRECISIONS
@pytest.mark.parametrize("p", [1, 2])
@pytest.mark.parametrize("name", sorted(_quads()))
def test_groups_without_directions(name, p, prec):
    quad, groups, before = _quads()[name]
    op = _operator(quad, p, prec)
    x = np.random.default_rng(8).standard_normal(op.n)
    op.sweep_mode = ou.SWEEP_TILES
    op.sweep_shape = (1, groups)
    op.sweep_mode = ou.SWEEP_LEVELS
    op.sweep_shape = (4, before)
    op.Apply(-x)  # leaves its moments where the strips' layout has empty groups
    op.sweep_mode = ou.SWEEP_TILES
    tiles = op.Apply(x)
    assert np.array_equal(op.Apply(x), tiles)
    op.sweep_mode = ou.SWEEP_LEVELS
    op.sweep_shape = (4, groups)
    assert np.array_equal(op.Apply(x), tiles)
    op.close()


def test_overflow_in_the_last_moment():
    """A source term that overflows FP32 in one dof of the last moment of three (padded
    to four) is an infinity there, as in the level launches, and no NaN."""
    quad = ou.Quadrature(ou.PRODUCT_GLC, 2, n_polar=8, n_azim=16, L_max=1)
    assert quad.n_mom == 3
    # large cells: nothing but the overflowed source term leaves FP32's range
    op = _operator(quad, 1, ou.FP32, h=100.0)
    n_dofs = op.n // 3
    M = ou.fe_matrices(2, 1, [100.0] * 2)[0]
    x = np.zeros(op.n)
    # sigma_s M x: 1.5 times the largest FP32 in its own dof, half of it beside it
    x[2 * n_dofs + 4 * 50] = 1.5 * float(np.finfo(np.float32).max) / (0.5 * M[0, 0])
    op.sweep_mode = ou.SWEEP_TILES
    op.sweep_shape = (1, 2)
    tiles = op.Apply(x)
    op.sweep_mode = ou.SWEEP_LEVELS
    op.sweep_shape = (4, 2)
    levels = op.Apply(x)
    assert np.isinf(levels).any()
    assert np.array_equal(tiles, levels, equal_nan=True)
    op.close()
