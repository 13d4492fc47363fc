"""GPU: the finite-volume flux pass by strip heights from one row up (the default of a grid is
chosen from its size), on grids narrower and wider than a strip's 61 columns: rk2 steps give
the same bits, in FP64 and FP32, wet and dry."""
import numpy as np
import pytest

from ptha_amd.domain import Domain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(7, 9), (61, 40), (131, 67)])
@pytest.mark.parametrize("precision", ["fp64", "fp32k"])
def test_strip_heights_same_bits(nx, ny, precision):
    ref = None
    for rows in (8, 0, 1, 2, 3, 5, 64):
        print("CASE fv strips", nx, ny, precision, rows, flush=True)
        rng = np.random.default_rng(nx + ny)
        with Domain(nx, ny, (nx * 50.0, ny * 50.0), (0.0, 0.0), "rk2", precision=precision, spherical=False) as d:
            if rows:
                d.set_launch(128, rows, 0)
            U = np.zeros((4, ny, nx))
            U[3] = -3.0 + 4.0 * rng.random((ny, nx))
            U[0] = np.maximum(U[3], 0.3 * rng.standard_normal((ny, nx)))
            d.set_manning_squared(0.03 ** 2)
            d.U = U
            for _ in range(4):
                d.evolve_one_step()
            got = (d.U.copy(), d.scalars()["time"])
        if ref is None:
            ref = got
        assert np.array_equal(got[0], ref[0]) and got[1] == ref[1], rows
