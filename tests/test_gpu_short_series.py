"""Short series asked for RR, DET or LAM, on both sides of the lengths where the
segment length changes, against the oracle.  Counts are integers, so the bound
is equality."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _hists(amd, oracle, n, m, nt, dist, dt, which):
    x = np.cumsum(np.random.default_rng(n + m).standard_normal(n))
    x = ((x - x.mean()) / x.std()).astype(dt)
    thr = (np.linspace(0.05, 1.5, nt) * (np.sqrt(m) if dist == 1 else 1.0)).astype(dt)
    got = amd.histograms(x, 1, m, thr, dist, which=which)
    for t in range(0, nt, 2):
        if which & 1:
            assert int(got["rr"][t]) == oracle.rr_count(x, thr[t], 1, m, dist)
        if which & 2:
            assert np.array_equal(got["det"][t], oracle.hist("det", x, thr[t], 1, m, dist))
        if which & 4:
            assert np.array_equal(got["lam"][t], oracle.hist("lam", x, thr[t], 1, m, dist))


@pytest.mark.parametrize("nc", [512, 1000, 2897, 2898, 4096, 4097, 8160, 8193])
@pytest.mark.parametrize("m,dist,dt", [(2, 1, np.float32), (12, 1, np.float32), (3, 2, np.float64)])
def test_rr_alone(oracle, nc, m, dist, dt):
    import accrqa_amd as amd
    _hists(amd, oracle, nc + m - 1, m, 3, dist, dt, 1)


@pytest.mark.parametrize("nc", [63, 64, 65, 127, 129, 2047, 2049, 2080, 3105])
@pytest.mark.parametrize("m,dist,dt", [(2, 1, np.float32), (12, 1, np.float32), (3, 2, np.float64), (9, 1, np.float64)])
@pytest.mark.parametrize("split", [True, False])
def test_segments(oracle, nc, m, dist, dt, split):
    import accrqa_amd as amd
    amd.set_split(amd.SPLIT_AUTO if split else amd.SPLIT_NEVER)
    try:
        _hists(amd, oracle, nc + m - 1, m, 5, dist, dt, 7)
        _hists(amd, oracle, nc + m - 1, m, 3, dist, dt, 2)
    finally:
        amd.set_split(amd.SPLIT_AUTO)
