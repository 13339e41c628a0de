"""The scans' plain and dense forms and every threshold group size (4, 8, 16,
24, 32 thresholds) against the oracle, bit for bit: series whose runs are
mostly single steps (noise, the logistic map), smooth ones, and one that
changes between them, in short segments and, by the slab form, in segments
longer than the plain form's stretch of 64 blocks.  Counts are integers, so
the bound is equality."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _series(kind, n, dt):
    rng = np.random.default_rng(21)
    smooth = np.cumsum(rng.standard_normal(n)) * 0.05
    noise = rng.standard_normal(n)
    if kind == "smooth":
        return smooth.astype(dt)
    if kind == "noise":
        return noise.astype(dt)
    if kind == "logistic":
        x, v = np.empty(n), 0.37
        for k in range(n):
            x[k], v = v, 3.97 * v * (1 - v)
        return x.astype(dt)
    return np.where(np.arange(n) // 700 % 2 == 0, smooth, noise).astype(dt)   # changing


@pytest.mark.parametrize("kind", ["noise", "logistic", "smooth", "changing"])
@pytest.mark.parametrize("nt", [3, 7, 13, 20, 24, 25, 32])
@pytest.mark.parametrize("dt,dist,m,slab", [(np.float32, 1, 2, 0), (np.float64, 2, 3, 0), (np.float32, 1, 9, 0),
                                            (np.float32, 2, 1, 4096)])
def test_scan_forms(oracle, kind, nt, dt, dist, m, slab):
    import accrqa_amd as amd
    n = 2700 if slab == 0 else 4700
    x = _series(kind, n, dt)
    thr = (np.linspace(0.03, 1.1, nt) * (1.0 if dist == 2 else np.sqrt(m))).astype(dt)
    thr[nt // 2] = thr[nt // 3]   # an equal pair
    amd.set_slab_rows(slab)
    try:
        both = amd.histograms(x, 1, m, thr, dist)
        det = amd.histograms(x, 1, m, thr, dist, which=2)["det"]
    finally:
        amd.set_slab_rows(0)
    assert np.array_equal(both["det"], det)
    for t in sorted({0, 1, nt // 2, nt - 2, nt - 1}):
        assert int(both["rr"][t]) == oracle.rr_count(x, thr[t], 1, m, dist)
        assert np.array_equal(both["det"][t], oracle.hist("det", x, thr[t], 1, m, dist))
        assert np.array_equal(both["lam"][t], oracle.hist("lam", x, thr[t], 1, m, dist))
