"""The bounded waits of the strip sweep (OU_SWEEP_TILES in 2D up to 10 moments) and the
reports of those that give up.

Bar: a zero limit gives up at the first wait that finds its upwind strip unfinished, a
sweep that gave up is reported once by the next call that can, whatever mode comes in
between, and afterwards results equal the earlier ones bit for bit."""
import numpy as np
import pytest

import ouranos_amd as ou
from ouranos_amd import problems as P

pytestmark = pytest.mark.gpu

TIMEOUT = -8  # OU_ERR_TIMEOUT


def _uniform(n=(48, 2)):
    quad = ou.Quadrature(ou.PRODUCT_GLC, 2, n_polar=4, n_azim=8, L_max=0)
    return ou.RadiativeTransfer(2, 1, n, [1.0 / max(n)] * 2, quad, np.array([1.0]),
                                np.array([[0.5]]), np.zeros(n[0] * n[1], np.int32))


@pytest.mark.parametrize("rows", [1, 2, 7])
def test_zero_limit_gives_up_at_the_first_wait(rows):
    """Short strips: a wait lasts a few microseconds, fewer than 16 polls."""
    op = _uniform((48, rows))
    assert op.sweep_mode == ou.SWEEP_TILES
    x = np.random.default_rng(3).standard_normal(op.n)
    y = op.Apply(x)
    op.set_sweep_wait_limit(0.0)
    for _ in range(3):
        with pytest.raises(ou.OuError) as e:
            op.Apply(x)
        assert e.value.code == TIMEOUT
    op.set_sweep_wait_limit(10.0)
    assert np.array_equal(op.Apply(x), y)
    op.close()


def _device_apply(op, x):
    """ou_apply_device, which reports nothing, awaited through another buffer's copy."""
    dx, dy = ou.DeviceBuffer(x.nbytes), ou.DeviceBuffer(x.nbytes)
    dx.upload(x)
    op.apply_device(dx, dy)
    ou._check(ou.lib().ou_device_synchronize())
    y = dy.download(np.empty(x.size))
    dx.free()
    dy.free()
    return y


@pytest.mark.parametrize("first,second", [(ou.SWEEP_PERSISTENT, ou.SWEEP_TILES),
                                          (ou.SWEEP_TILES, ou.SWEEP_PERSISTENT)],
                         ids=["persistent_then_strips", "strips_then_persistent"])
def test_timeout_is_reported_once_across_modes(first, second):
    """A sweep that gave up in one mode is reported in the other: never NaN without an
    error, and not a second time."""
    spec = P.hetero_2d(n=64, block=8, n_polar=16, n_azim=32, L=1)
    op = spec.operator(ou.FP64)
    x = P.seeded_vector(spec.size, 5)
    want = {}
    for mode in (first, second):
        op.sweep_mode = mode
        op.sweep_shape = (4, 1) if mode == ou.SWEEP_PERSISTENT else (2, 1)
        want[mode] = op.Apply(x)
    op.sweep_mode = first
    op.set_sweep_wait_limit(0.0)
    assert np.isnan(_device_apply(op, x)).all()
    op.set_sweep_wait_limit(10.0)
    op.sweep_mode = second
    with pytest.raises(ou.OuError) as e:
        op.Apply(x)
    assert e.value.code == TIMEOUT
    for mode in (second, first, second):
        op.sweep_mode = mode
        assert np.array_equal(op.Apply(x), want[mode]), mode
        op.sweep_status()
    op.close()


def _batch(limit):
    specs = [P.hetero_2d(n=n, block=8, seed=s, n_polar=8, n_azim=16, L=1)
             for n, s in ((64, 1), (48, 2))]
    ops = [s.operator(ou.FP64) for s in specs]
    for op in ops:
        op.set_sweep_wait_limit(limit)
    return specs, ops


def test_batch_reports_a_strip_timeout():
    """apply raises instead of returning NaN; an application that only enqueues is
    reported by the status call or by the next one; level launches are not affected."""
    specs, ops = _batch(0.0)
    xs = [P.seeded_vector(s.size, i) for i, s in enumerate(specs)]
    batch = ou.Batch(ops, waves=4, dir_groups=1)
    want = batch.apply(xs)
    batch.set_sweep_mode(ou.SWEEP_TILES)
    batch.set_shape(2, 1)
    for _ in range(2):
        with pytest.raises(ou.OuError) as e:
            batch.apply(xs)
        assert e.value.code == TIMEOUT
        batch.sweep_status()  # reported and cleared
    dx = [ou.DeviceBuffer(x.nbytes) for x in xs]
    dy = [ou.DeviceBuffer(x.nbytes) for x in xs]
    for b, x in zip(dx, xs):
        b.upload(x)
    for report in (batch.sweep_status, lambda: batch.apply_device(dx, dy),
                   lambda: batch.sweep_device(dy)):
        batch.apply_device(dx, dy)
        ou._check(ou.lib().ou_device_synchronize())
        with pytest.raises(ou.OuError) as e:
            report()
        assert e.value.code == TIMEOUT
        batch.sweep_status()
    batch.set_sweep_mode(ou.SWEEP_LEVELS)
    for y, w in zip(batch.apply(xs), want):
        assert np.array_equal(y, w)
    batch.close()


def test_batch_tuner_passes_over_shapes_that_give_up():
    specs, ops = _batch(0.0)
    xs = [P.seeded_vector(s.size, i) for i, s in enumerate(specs)]
    batch = ou.Batch(ops)
    table = batch.tune(reps=1)
    assert table and all(e["mode"] == ou.SWEEP_LEVELS for e in table)
    assert batch.sweep_mode == ou.SWEEP_LEVELS
    assert all(np.isfinite(y).all() for y in batch.apply(xs))
    batch.close()
