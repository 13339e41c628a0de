"""The byte table of the MFMA form in its rotated LDS place: thresholds whose
buckets span few or all of the table, start at different low bits and wrap
around its end, against the oracle.  Counts are integers and every decision is
the reference's, so the bound is equality."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

RANGES = [(1.0, 1.0001), (1.4, 1.5), (1e-3, 3.0), (0.7, 2.9), (1e-18, 1e18), (0.0, 2.5), (2.0, 1e19), (1.9999, 4.0)]


@pytest.mark.parametrize("lo,hi", RANGES)
@pytest.mark.parametrize("m,nt,dt", [(8, 1, np.float32), (16, 16, np.float32), (20, 32, np.float32), (9, 5, np.float64)])
def test_table_ranges(oracle, lo, hi, m, nt, dt):
    import accrqa_amd as amd
    n = 330
    x = np.cumsum(np.random.default_rng(m).standard_normal(n))
    x = ((x - x.mean()) / x.std()).astype(dt)
    thr = np.linspace(lo, hi, nt).astype(dt) if hi < 10 else np.geomspace(lo, hi, nt).astype(dt)
    nc = n - (m - 1)
    rr = amd.histograms(x, 1, m, thr, 1, which=1)["rr"]
    lam = amd.histograms(x, 1, m, thr, 1, which=4)["lam"]
    amd.set_split(amd.SPLIT_NEVER)
    try:
        det = amd.histograms(x, 1, m, thr, 1, which=2)["det"]
    finally:
        amd.set_split(amd.SPLIT_AUTO)
    for t in range(nt):
        assert int(rr[t]) == oracle.rr_count(x, thr[t], 1, m, 1)
        assert np.array_equal(lam[t], oracle.hist("lam", x, thr[t], 1, m, 1))
        assert np.array_equal(det[t], oracle.hist("det", x, thr[t], 1, m, 1))
    assert nc == lam.shape[1] - 1
