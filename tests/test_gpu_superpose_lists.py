"""GPU: events summed from lists of their sources against sums in NumPy FP64 of the same
recorded series: source counts at the edges of the two tile widths (16 and 8 lanes an event)
and past them (matrix product), gauges and samples that leave partial tiles, events of one
source, of none, with a source named twice and of nearly all sources; with and without
weights, series and maxima, and a source whose series holds NaN.

The bar: each side's sum of n terms rounds by at most n units of 2^-53 of the sum of the
terms' sizes, the offset, the scale and the last addition by one each."""
import numpy as np
import pytest

from ptha_amd.batch import UnitSourceBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsrc,gauges,samples,n_events", [
    (5, 1, 3, 1), (37, 17, 9, 65), (200, 33, 8, 300), (639, 16, 5, 130), (640, 5, 4, 70), (1279, 9, 3, 40),
    (1281, 4, 3, 33)])
@pytest.mark.parametrize("weighted", [False, True])
def test_lists_equal_sums(nsrc, gauges, samples, n_events, weighted):
    print("CASE superpose lists", nsrc, gauges, samples, n_events, weighted, flush=True)
    nx, ny, every = 12, 10, 2
    rng = np.random.default_rng(nsrc + n_events)
    with UnitSourceBatch(nx, ny, (2.0, 1.6), (140.0, -30.0), nsrc, precision="fp64") as b:
        b.set_elevation(np.full((ny, nx), -4000.0))
        b.set_nsteps(np.full(nsrc, every * (samples - 1), dtype=np.int32))
        bad = nsrc // 3
        for k in range(nsrc):
            s = rng.standard_normal((ny, nx))
            if k == bad and weighted:
                s[4, 5] = np.nan
            b.set_source(k, s)
        xy = np.stack([140.2 + 1.6 * rng.random(gauges), -29.8 + 1.2 * rng.random(gauges)], axis=1)
        b.setup_point_gauges(xy, every=every, max_samples=samples)
        b.evolve(3.0, every * (samples - 1))
        X = np.stack([b.gauge_series(k) for k in range(nsrc)])
        assert X.shape == (nsrc, samples, 3, gauges)
        events = [[0], [], [nsrc - 1, 0, nsrc - 1], list(range(nsrc - 1))]
        events = (events + [sorted(rng.choice(nsrc, size=int(rng.integers(1, max(2, nsrc // 3))), replace=False).tolist())
                            for _ in range(n_events)])[:max(n_events, 4)]
        w = [rng.normal(size=len(e)).tolist() for e in events] if weighted else None
        slip = None if weighted else rng.uniform(0.5, 8.0, size=len(events))
        msl = 0.3
        series, nv = b.superpose(events, slip=slip, weights=w, msl=msl, summary="series")
        mx, _ = b.superpose(events, slip=slip, weights=w, msl=msl, summary="max_stage")
        assert np.all(nv == samples)
        off = np.array([msl, 0.0, 0.0])[None, :, None]
        for e, ev in enumerate(events):
            we = np.array(w[e]) if weighted else np.ones(len(ev))
            sl = 1.0 if weighted else slip[e]
            Y = X[ev] - off
            ref = np.einsum("k,ksvg->svg", we, Y) * sl + off
            size = np.einsum("k,ksvg->svg", np.abs(we), np.abs(Y) + np.abs(off)) * sl + np.abs(off)
            tol = (2 * len(ev) + 8) * 2.0 ** -53 * size
            fin = np.isfinite(ref)
            assert np.array_equal(np.isfinite(series[e]), fin), e
            assert np.all(np.abs(series[e] - ref)[fin] <= tol[fin]), e
            for g in range(gauges):
                st = ref[:, 0, g]
                if np.isnan(st).any():
                    assert np.isnan(mx[e, g]), (e, g)
                else:
                    assert abs(mx[e, g] - st.max()) <= tol[:, 0, g].max(), (e, g)
