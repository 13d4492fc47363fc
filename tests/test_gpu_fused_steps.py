"""GPU: several leapfrog steps of a single grid per launch (swh_evolve_steps and the gauge
schedule), with max_stage and the boundary fluxes inside, against one step per launch:
states, maxima, gauge samples and times are the same bits, the boundary-flux integrals agree
to 1e-13 of the gross flux (both are double-double sums, in another order). Grids from a few
cells to several wavefronts wide and several strips high, step counts that leave remainders,
max_stage every step, every third step and not at all."""
import numpy as np
import pytest

from ptha_amd import backend as B
from ptha_amd.domain import Domain

pytestmark = pytest.mark.gpu


def _make(nx, ny, precision, method, tl, lfc, spherical, maxu, freq, seed=0):
    lw, ll = ((nx / 30.0, ny / 30.0), (150.0, -40.0)) if spherical else ((nx * 2000.0, ny * 2000.0), (0.0, 0.0))
    rng = np.random.default_rng(nx * 1000 + ny + seed)
    d = Domain(nx, ny, lw, ll, method, precision=precision, spherical=spherical, linear_solver_is_truely_linear=tl,
               linear_friction_coeff=lfc, max_U_variables=maxu, max_U_update_frequency=freq)
    U = rng.standard_normal((4, ny, nx))
    U[1:3] *= 20.0
    U[3] = -3000.0 + 1500.0 * rng.random((ny, nx))
    U[3][rng.random((ny, nx)) < 0.03] = 5.0
    if method != "linear":
        d.set_manning_squared(0.03 ** 2)
    d.U = U
    return d


CASES = [  # nx, ny, precision, method, truely linear, linear friction, spherical
    (5, 5, "fp32k", "linear", True, 0.0, True),
    (5, 9, "fp64", "linear", True, 0.0, False),
    (56, 40, "fp32k", "linear", True, 0.0, True),
    (112, 17, "fp32k", "linear", True, 1e-4, False),
    (221, 131, "fp32k", "leapfrog_linear_plus_nonlinear_friction", True, 0.0, True),
    (59, 33, "fp64", "linear", True, 0.0, True),
    (119, 70, "fp64", "leapfrog_linear_plus_nonlinear_friction", True, 1e-5, False),
    (60, 37, "fp64", "linear", False, 0.0, False),
    (61, 140, "fp32k", "linear", False, 1e-4, True),
]


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("maxu,freq", [(("max_stage",), 1), (("max_stage",), 3), ((), 1)])
def test_fused_equals_single_steps(case, maxu, freq):
    print("CASE fused", case, maxu, freq, flush=True)
    nx, ny, precision, method, tl, lfc, spherical = case
    a = _make(nx, ny, precision, method, tl, lfc, spherical, maxu, freq)
    b = _make(nx, ny, precision, method, tl, lfc, spherical, maxu, freq)
    b.set_launch(128, 4, 32)
    dt, gross = 2.0, 0.0
    for n in (1, 2, 3, 4, 5, 7, 8, 16):
        a.evolve_steps(dt, n)
        b.evolve_steps(dt, n)
        assert np.array_equal(a.U, b.U), n
        if maxu:
            assert np.array_equal(a.max_U("max_stage"), b.max_U("max_stage")), n
        sa, sb = a.scalars(), b.scalars()
        for k in ("time", "evolve_step_dt", "dt_last_update", "nsteps_advanced"):
            assert sa[k] == sb[k], (n, k)
        gross = max(gross, float(np.abs(sb["boundary_flux_store"]).sum()) * dt * 50)
        assert np.allclose(sa["boundary_flux_store"], sb["boundary_flux_store"], rtol=0, atol=1e-13 * gross)
        for k in ("boundary_flux_evolve_integral", "boundary_flux_time_integral"):
            assert abs(sa[k] - sb[k]) <= 1e-13 * gross, (n, k)
    a.close()
    b.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32k"])
@pytest.mark.parametrize("method,steps", [("linear", [0, 1, 2, 4, 9, 13, 14, 21, 34, 40]), ("linear", [3, 8, 13, 16, 18]),
                                          ("leapfrog_linear_plus_nonlinear_friction", [0, 5, 11, 12, 30])])
def test_gauge_schedule_inside_fused_steps(precision, method, steps):
    print("CASE fused gauges", precision, method, steps, flush=True)
    nx, ny = 131, 77
    ij = np.array([[3, 3], [3, 40], [66, 12], [131, 77], [1, 1], [66, 50]])
    out = []
    for one in (False, True):
        d = _make(nx, ny, precision, method, True, 0.0, True, ("max_stage",), 1)
        if one:
            d.set_launch(128, 4, 32)
        d.setup_point_gauges(ij=ij, max_samples=len(steps))
        s = np.array(steps, dtype=np.int64)
        B.check(d._lib.swh_evolve_record_gauges_schedule(d._h, 2.0, len(s), s.ctypes.data_as(B._PI64)), "schedule")
        out.append((d.gauge_series(), d.U, d.max_U("max_stage"), d.scalars()["nsteps_advanced"]))
        d.close()
    (ta, va), Ua, Ma, na = out[0]
    (tb, vb), Ub, Mb, nb = out[1]
    assert na == nb == steps[-1]
    assert np.array_equal(ta, tb) and np.array_equal(va, vb)
    assert np.array_equal(Ua, Ub) and np.array_equal(Ma, Mb)
