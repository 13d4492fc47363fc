"""GPU: the tridiagonal walks of the dispersive solve at the sizes where their phases,
blocks of lines and transposing tiles begin and end (16 lines per workgroup, 64 elements
per phase of the substitution, 8 of the elimination, 16 per unrolled block, 32 x 32 tiles),
on a bed of random depth jumps, where the elimination swaps rows, and with a state so small
that the back substitution leaves the range of its reciprocal; and the smaller work buffer
(taken where device memory is short), whose results are the same bits. FP64 'linear' steps are
bit-identical to the oracle, whose elimination is LAPACK's dgtsv."""
import numpy as np
import pytest

import helpers as H
from ptha_amd import backend as B
from ptha_amd import configs as C

pytestmark = pytest.mark.gpu

SIZES = [(6, 5), (17, 67), (18, 19), (33, 65), (66, 18), (81, 34), (131, 50)]


def _rough(nx, ny, scale):
    cfg = C.gaussian_hump_cartesian(nx=nx, ny=ny, dx=8.0, sigma=40.0)
    rng = np.random.default_rng(1000 * nx + ny)
    U = np.zeros((4, ny, nx))
    U[3] = rng.choice([-20.0, -19.0, -6.0, -0.2, 2.0], size=(ny, nx), p=[0.4, 0.2, 0.2, 0.1, 0.1])
    U[0] = np.where(U[3] < 0, scale * rng.standard_normal((ny, nx)), 0.0)
    return dict(cfg, U=U)


@pytest.mark.parametrize("scale", [1.0, 1e-299])
@pytest.mark.parametrize("nx,ny", SIZES)
def test_walk_edges_fp64_bitexact(oracle_built, nx, ny, scale):
    print("CASE dispersion walk", nx, ny, scale, flush=True)
    cfg = _rough(nx, ny, scale)
    o, dt, _ = H.cpu_run("oracle", cfg, 0)
    o.dispersion_setup(0.0, -1.0, 2)
    g = H.gpu_domain(cfg)
    g.dispersion_enable(0.0, -1.0, 2)
    for _ in range(5):
        o.dispersive_step(0.3 * dt, 1)
        g.dispersive_step(0.3 * dt, 1)
    Uo, Ug = o.get_U(), g.U
    for k in range(4):
        assert np.array_equal(Ug[k], Uo[k]), (k, np.abs(Ug[k] - Uo[k]).max())
    assert np.abs(Ug[1]).max() > 0 and np.isfinite(Ug).all()
    g.close()


@pytest.mark.parametrize("method", ["linear", "midpoint"])
@pytest.mark.parametrize("precision", ["fp64", "fp32k"])
@pytest.mark.parametrize("nx,ny", [(6, 5), (33, 65), (131, 50)])
def test_compact_work_buffer_same_bits(nx, ny, precision, method):
    print("CASE dispersion compact", nx, ny, precision, method, flush=True)
    cfg, out = dict(_rough(nx, ny, 1.0), method=method), []
    for compact in (False, True):
        g = H.gpu_domain(cfg, precision=precision)
        if compact:
            B.check(g._lib.swh_probe_dispersion_compact(g._h), "compact")
        g.dispersion_enable(0.0, -1.0, 2)
        for _ in range(4):
            g.dispersive_step(0.05, 1)
        out.append(g.U)
        g.close()
    assert np.array_equal(out[0], out[1], equal_nan=True) and np.abs(out[0][1]).max() > 0
