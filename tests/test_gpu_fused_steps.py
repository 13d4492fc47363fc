"""GPU: several leapfrog steps of a single grid per launch (swh_evolve_steps and the gauge
schedule), with max_stage and the boundary fluxes inside, against one step per launch:
states, maxima, gauge samples and times are the same bits. Grids from a few cells to several
wavefronts wide and several strips high, step counts that leave remainders and that make runs of
fused launches long enough to be taken, max_stage every step, every third step and not at all,
boundary-flux lines at other distances from the edge, forcing that begins and ends between
fused launches, gauge samples inside a launch after each of its steps.

The boundary fluxes are double-double sums in another order (equal to 2^-90 of their terms),
then rounded: a side's sum and its product with the edge length by half a unit of 2^-53 each,
their total times dt by five more, the running integral by one per step. With S the sum of the sides'
sizes, the two runs' stores agree to 2 units of S, a step's integral to 8 units of S dt,
the time integral over n steps to 10 n units of S dt, S at most four times its largest sampled
value, plus n units of the largest running integral."""
import numpy as np
import pytest

from ptha_amd import backend as B
from ptha_amd.domain import Domain

pytestmark = pytest.mark.gpu


def _make(nx, ny, precision, method, tl, lfc, spherical, maxu, freq, seed=0, ext=2):
    lw, ll = ((nx / 30.0, ny / 30.0), (150.0, -40.0)) if spherical else ((nx * 2000.0, ny * 2000.0), (0.0, 0.0))
    rng = np.random.default_rng(nx * 1000 + ny + seed)
    d = Domain(nx, ny, lw, ll, method, precision=precision, spherical=spherical, linear_solver_is_truely_linear=tl,
               linear_friction_coeff=lfc, max_U_variables=maxu, max_U_update_frequency=freq,
               exterior_cells_width=ext)
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


def _compare(a, b, dt, counts, maxu):
    u, S, largest, steps = 2.0 ** -53, 0.0, 0.0, 0
    for n in counts:
        a.evolve_steps(dt, n)
        b.evolve_steps(dt, n)
        steps += n
        assert np.array_equal(a.U, b.U), n
        if maxu:
            assert np.array_equal(a.max_U("max_stage"), b.max_U("max_stage")), n
        sa, sb = a.scalars(), b.scalars()
        for k in ("time", "evolve_step_dt", "dt_last_update", "nsteps_advanced"):
            assert sa[k] == sb[k], (n, k)
        s = float(np.abs(sb["boundary_flux_store"]).sum())
        S, largest = max(S, s), max(largest, abs(sb["boundary_flux_time_integral"]))
        assert np.allclose(sa["boundary_flux_store"], sb["boundary_flux_store"], rtol=0, atol=2 * u * s)
        k = "boundary_flux_evolve_integral"
        assert abs(sa[k] - sb[k]) <= 8 * u * s * dt, (n, k)
        k = "boundary_flux_time_integral"
        assert abs(sa[k] - sb[k]) <= steps * u * (40 * S * dt + largest), (n, k)


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("maxu,freq", [(("max_stage",), 1), (("max_stage",), 3), ((), 1)])
def test_fused_equals_single_steps(case, maxu, freq):
    print("CASE fused", case, maxu, freq, flush=True)
    a = _make(*case, maxu, freq)
    b = _make(*case, maxu, freq)
    b.set_launch(128, 4, 32)
    _compare(a, b, 2.0, (1, 2, 3, 4, 5, 7, 8, 16, 40), maxu)
    a.close()
    b.close()


@pytest.mark.parametrize("nx,ny,ext", [(9, 5, 1), (40, 23, 5), (119, 64, 12), (301, 355, 60)])
@pytest.mark.parametrize("precision", ["fp64", "fp32k"])
def test_boundary_lines_at_other_widths(nx, ny, ext, precision):
    print("CASE fused lines", nx, ny, ext, precision, flush=True)
    case = (nx, ny, precision, "linear", True, 0.0, True, ("max_stage",), 1)
    a, b = _make(*case, ext=ext), _make(*case, ext=ext)
    b.set_launch(128, 4, 32)
    _compare(a, b, 2.0, (3, 12, 19), ("max_stage",))
    a.close()
    b.close()


@pytest.mark.parametrize("precision", ["fp64", "fp32k"])
@pytest.mark.parametrize("t0,t1", [(31.0, 55.0), (36.0, 37.0), (0.0, 30.0), (117.0, 300.0)])
def test_forcing_between_fused_launches(precision, t0, t1):
    print("CASE fused forcing", precision, t0, t1, flush=True)
    case = (131, 77, precision, "linear", True, 0.0, True, ("max_stage",), 1)
    a, b = _make(*case), _make(*case)
    b.set_launch(128, 4, 32)
    work = np.random.default_rng(5).standard_normal((1, 20, 30))
    for d in (a, b):
        d.set_forcing_patch(t0, t1, 11, 40, 21, 40, 1, 1, work)
    _compare(a, b, 2.0, (60, 3, 33), ("max_stage",))
    a.close()
    b.close()


IJ = [[3, 3], [3, 40], [66, 12], [131, 77], [1, 1], [66, 50]]
# two gauges in one column and strip, at each side of the edges of wavefronts (59 columns) and strips of
# 3 to 47 rows; three in one cell, which do not fit the lanes
EDGES = [[66, 30], [66, 30], [59, 12], [60, 12], [118, 76], [119, 76]] + [[20 + r, r] for r in (3, 4, 6, 7, 48, 49)]
CROWD = [[70, 41], [70, 41], [70, 41], [5, 9]]


@pytest.mark.parametrize("precision", ["fp64", "fp32k"])
@pytest.mark.parametrize("method,tl,lfc,spherical", [
    ("linear", True, 0.0, True), ("linear", True, 1e-4, False), ("linear", False, 0.0, True),
    ("leapfrog_linear_plus_nonlinear_friction", True, 0.0, True)])
@pytest.mark.parametrize("maxu", [(), ("max_stage",)])
@pytest.mark.parametrize("ij", [IJ, EDGES, CROWD])
@pytest.mark.parametrize("steps", [
    [0, 1, 2, 4, 9, 13, 14, 21, 34, 40], [3, 8, 13, 16, 18], [0, 5, 11, 12, 30],
    list(range(4, 85, 4)),       # after the first, second and third step of a launch in turn
    [17, 34, 51, 68, 85, 96],    # (every 17, then the end of a launch)
    list(range(2, 61, 2)), [36]])
def test_gauge_schedule_inside_fused_steps(precision, method, tl, lfc, spherical, maxu, ij, steps):
    print("CASE fused gauges", precision, method, tl, lfc, spherical, maxu, len(ij), steps, flush=True)
    nx, ny = 131, 77
    ij = np.array(ij)
    out = []
    for one in (False, True):
        d = _make(nx, ny, precision, method, tl, lfc, spherical, maxu, 1)
        if one:
            d.set_launch(128, 4, 32)
        d.setup_point_gauges(ij=ij, max_samples=len(steps))
        s = np.array(steps, dtype=np.int64)
        B.check(d._lib.swh_evolve_record_gauges_schedule(d._h, 2.0, len(s), s.ctypes.data_as(B._PI64)), "schedule")
        out.append((d.gauge_series(), d.U, d.max_U("max_stage") if maxu else 0.0, d.scalars()["nsteps_advanced"]))
        d.close()
    (ta, va), Ua, Ma, na = out[0]
    (tb, vb), Ub, Mb, nb = out[1]
    assert na == nb == steps[-1]
    assert np.array_equal(ta, tb) and np.array_equal(va, vb)
    assert np.array_equal(Ua, Ub) and np.array_equal(Ma, Mb)
