"""GPU: batches with the strip height left to the launch (chosen from the sources still
running), on grids from a few rows to more than a strip and to one
that fills the device with its deeper launches, with sources that stop at
different steps so that the height changes between launches: each source's final state and
gauge series equal those of the same source stepped alone, one step per launch, bit for
bit (both precisions)."""
import numpy as np
import pytest

from ptha_amd.batch import UnitSourceBatch
from ptha_amd.domain import Domain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32k"])
@pytest.mark.parametrize("nx,ny,steps", [(7, 5, (3, 9)), (56, 13, (23, 7, 1)), (130, 97, (40, 12, 0, 33, 21)),
                                         (611, 300, (17, 6)), (1300, 1200, (14, 9, 14, 3))])
def test_rows_chosen_per_launch(precision, nx, ny, steps):
    print("CASE batch rows", precision, nx, ny, steps, flush=True)
    rng = np.random.default_rng(nx + ny)
    lw, ll = (nx / 60.0, ny / 60.0), (150.0, -30.0)
    elev = -4000.0 + 500.0 * rng.random((ny, nx))
    elev[:, -1] = elev[0, :] = 1e6
    stages = [np.where(elev < 0, rng.standard_normal((ny, nx)), 0.0) for _ in steps]
    xy = np.stack([ll[0] + lw[0] * rng.random(6), ll[1] + lw[1] * rng.random(6)], axis=1)
    dt, every = 3.0, 4
    with UnitSourceBatch(nx, ny, lw, ll, len(steps), precision=precision) as b:
        b.set_elevation(elev)
        b.set_nsteps(np.array(steps, dtype=np.int32))
        b.setup_point_gauges(xy, every=every, max_samples=max(steps) // every + 1)
        for k, s in enumerate(stages):
            b.set_source(k, s)
        b.evolve(dt, max(steps))
        for k, n in enumerate(steps):
            with Domain(nx, ny, lw, ll, "linear", precision=precision, spherical=True, max_U_variables=()) as d:
                d.set_launch(128, 16, 32)
                U = np.zeros((4, ny, nx))
                U[0], U[3] = stages[k], elev
                d.U = U
                d.setup_point_gauges(xy, max_samples=n // every + 1)
                for m in range(n + 1):
                    if m % every == 0:
                        d.sample_gauges()
                    if m < n:
                        d.evolve_one_step(dt)
                assert np.array_equal(b.get_source(k), d.U[:3]), k
                assert np.array_equal(b.gauge_series(k), d.gauge_series()[1]), k


def test_autotune_keeps_what_no_fixed_shape_beats():
    """One small source needs strips of a few rows, shorter than any fixed shape that the tuner
    tries (2.5 us a step against 8.6 with the best of those): tuning must not leave
    the batch slower than it found it. The allowance, a half, covers the clock's scatter."""
    print("CASE autotune keeps automatic", flush=True)
    nx, ny, dt, steps = 300, 300, 3.0, 300
    rng = np.random.default_rng(1)
    elev = -4000.0 + 500.0 * rng.random((ny, nx))
    with UnitSourceBatch(nx, ny, (5.0, 5.0), (150.0, -30.0), 1, precision="fp32k") as b:
        b.set_elevation(elev)
        b.set_nsteps(np.array([20 * steps], dtype=np.int32))
        b.set_source(0, rng.standard_normal((ny, nx)))
        b.evolve(dt, steps)
        before = min(b.evolve_timed(dt, steps) for _ in range(4))
        state = b.get_source(0)
        (bx, rows, variant), ms = b.autotune(dt)
        assert np.array_equal(b.get_source(0), state) and ms > 0
        after = min(b.evolve_timed(dt, steps) for _ in range(4))
        assert after <= 1.5 * before, (before, after)
        b.set_launch(bx, rows, variant)   # what is returned is a shape that can be set
        b.evolve(dt, 3)
