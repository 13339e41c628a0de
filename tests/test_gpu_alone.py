"""RR, DET and LAM asked alone, MFMA form (m >= 8): k_rr_mx and the rank-tile
DET pass against the oracle, bit for bit, at the edges of the 32-row blocks,
64-column bands and threshold groups.  Counts and histograms are integers
and every decision is the reference's, so the bound is equality."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _series(n, dt, seed=11):
    x = np.cumsum(np.random.default_rng(seed).standard_normal(n))
    return ((x - x.mean()) / x.std()).astype(dt)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("nc", [1, 2, 31, 32, 33, 63, 64, 65, 127, 129, 700, 2049])
@pytest.mark.parametrize("tau,m,nt", [(1, 8, 1), (2, 16, 5), (3, 17, 17), (1, 33, 32), (0, 9, 3)])
def test_alone_matches_oracle(oracle, dt, nc, tau, m, nt):
    import accrqa_amd as amd
    x = _series(nc + (m - 1) * tau, dt)
    thr = np.sort(np.random.default_rng(nc).uniform(0.05, 2.5 * np.sqrt(m), nt)).astype(dt)
    rr = amd.histograms(x, tau, m, thr, 1, which=1)["rr"]
    det = amd.histograms(x, tau, m, thr, 1, which=2)["det"]
    lam = amd.histograms(x, tau, m, thr, 1, which=4)["lam"]
    for t in range(nt):
        assert int(rr[t]) == oracle.rr_count(x, thr[t], tau, m, 1)
        assert np.array_equal(det[t], oracle.hist("det", x, thr[t], tau, m, 1))
        assert np.array_equal(lam[t], oracle.hist("lam", x, thr[t], tau, m, 1))


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_alone_non_finite(oracle, bad):
    """A NaN or infinite sample sends every pair to the exact re-decision."""
    import accrqa_amd as amd
    x = _series(300, np.float32)
    x[123] = bad
    thr = np.array([0.5, 2.0, 1e30], np.float32)
    rr = amd.histograms(x, 1, 8, thr, 1, which=1)["rr"]
    det = amd.histograms(x, 1, 8, thr, 1, which=2)["det"]
    for t in range(3):
        assert int(rr[t]) == oracle.rr_count(x, thr[t], 1, 8, 1)
        assert np.array_equal(det[t], oracle.hist("det", x, thr[t], 1, 8, 1))


def test_det_alone_split_modes_identical():
    """DET from the rank tiles and from k_det_mx (no tile store)."""
    import accrqa_amd as amd
    x = _series(5000, np.float32)
    thr = np.linspace(0.2, 6.0, 16).astype(np.float32)
    a = amd.histograms(x, 1, 16, thr, 1, which=2)["det"]
    amd.set_split(amd.SPLIT_NEVER)
    try:
        b = amd.histograms(x, 1, 16, thr, 1, which=2)["det"]
    finally:
        amd.set_split(amd.SPLIT_AUTO)
    assert np.array_equal(a, b)
