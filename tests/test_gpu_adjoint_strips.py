"""GPU: the transposed leapfrog step on grids from five cells (the smallest domain) to several wavefronts wide and
several strips high (grids without and with interior wavefronts, narrower and wider than the
61 columns that one owns, odd strips at the north edge), with land: <y, F x> = <F' y, x> over
three steps, with Coriolis and without, FP64 and FP32.

The bar: a step forms each value from at most 30 operations in either direction, so over n
steps each side is off by at most 30 n eps of the terms' sizes, taken as the sums of the
products' sizes, with a factor of 4 for the cancellation inside the values."""
import numpy as np
import pytest

from ptha_amd.adjoint import GaugeMap

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(5, 5), (5, 64), (62, 9), (63, 70), (124, 131), (190, 33), (260, 47)])
@pytest.mark.parametrize("precision,spherical", [("fp64", True), ("fp32k", True), ("fp64", False)])
def test_transpose_of_steps(nx, ny, precision, spherical):
    print("CASE adjoint strips", nx, ny, precision, spherical, flush=True)
    rng = np.random.default_rng(nx * 1000 + ny)
    lw, ll = ((nx / 30.0, ny / 30.0), (150.0, -40.0)) if spherical else ((nx * 3000.0, ny * 3000.0), (0.0, 0.0))
    elev = -3000.0 + 1500.0 * rng.random((ny, nx))
    elev[rng.random((ny, nx)) < 0.05] = 10.0
    xy = np.array([[ll[0] + 0.5 * lw[0], ll[1] + 0.5 * lw[1]]])
    n, eps = 3, 2.0 ** -53 if precision == "fp64" else 2.0 ** -24
    g = GaugeMap(nx, ny, lw, ll, elev, 2.0, n, n, xy, precision=precision, spherical=spherical)
    x = rng.standard_normal((3, ny, nx)).astype(np.float32).astype(np.float64)
    y = rng.standard_normal((3, ny, nx)).astype(np.float32).astype(np.float64)
    x[1:] *= 16.0
    Fx, Fty = g.forward_steps(x, n), g.transpose_steps(y, n)
    g.close()
    size = np.abs(y * Fx).sum() + np.abs(x * Fty).sum()
    assert abs((y * Fx).sum() - (x * Fty).sum()) <= 4 * 30 * n * eps * size
