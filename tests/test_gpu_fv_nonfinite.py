"""GPU: one fixed-step 'euler' step of a wet grid with one infinite value: the limited gradient
between infinite differences of both signs is NaN, as in the reference's form (inf * 0), not
zero, so no cell leaves the finite range that the oracle keeps in it, and cells that are
finite on both sides are the same bits. (Fewer cells may be lost than in the oracle: the
device's minima and maxima pass over a NaN operand.)"""
import numpy as np
import pytest

import pyoracle
from ptha_amd.domain import Domain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("var", [0, 1, 2])
@pytest.mark.parametrize("bad", [np.inf, -np.inf])
def test_infinite_value_spreads_as_in_the_oracle(oracle_built, var, bad):
    print("CASE fv nonfinite", var, bad, flush=True)
    nx, ny, lw = 70, 31, (3500.0, 1550.0)
    rng = np.random.default_rng(3)
    U = np.zeros((4, ny, nx))
    U[3] = -3.0 - rng.random((ny, nx))
    U[0] = 0.3 * rng.standard_normal((ny, nx))
    U[1:3] = 0.2 * rng.standard_normal((2, ny, nx))
    U[var, 15, 30] = bad
    o = pyoracle.CpuDomain("oracle", nx, ny, lw, (0.0, 0.0), method="euler")
    o.set_U(U)
    o.evolve(0.5, 1)
    with Domain(nx, ny, lw, (0.0, 0.0), "euler", max_U_variables=()) as d:
        d.U = U
        d.evolve_one_step(0.5)
        Ug = d.U
    Uo = o.get_U()
    fo, fg = np.isfinite(Uo), np.isfinite(Ug)
    assert not (fo & ~fg).any(), np.argwhere(fo & ~fg)[:5]
    assert np.array_equal(Uo[fo & fg], Ug[fo & fg])
