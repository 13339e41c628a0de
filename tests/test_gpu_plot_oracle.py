"""Recurrence plots of bytes against the reference's decision, row by row, in
every work shape: small blocks, 64- and 256-squares, rows; one, two and more
chunks of 16 dimensions; row ends of every length; both sides of the rules that
choose.  Rows come from numpy in the reference's order and precision (held to
the oracle here, on the CPU); the rest of a plot follows from its symmetry,
which is exact.  Decisions are the reference's, so the bound is equality."""
import numpy as np
import pytest


def _rows(x, nc, tau, m, thr, dist, rows):
    """R[i][j] for i in rows: s summed k = 0 .. m-1 in x's precision, [thr - d >= 0]."""
    with np.errstate(all="ignore"):
        s = np.zeros((len(rows), nc), x.dtype)
        for k in range(m):
            v = x[k * tau:k * tau + nc]
            e = v[rows][:, None] - v[None, :]
            # max as the reference's comparison: a NaN difference is passed over
            s = s + e * e if dist == 1 else np.where(np.abs(e) > s, np.abs(e), s)
        d = np.sqrt(s) if dist == 1 else s
        return (x.dtype.type(thr) - d >= 0).astype(np.int8)


def _series(nc, tau, m, dt, kind, seed):
    n = nc + (m - 1) * tau
    w = np.cumsum(np.random.default_rng(seed).standard_normal(n))
    w = (w - w.mean()) / w.std()
    if kind == "ties":
        w = np.round(4 * w)
    x = w.astype(dt)
    if kind == "tiny":      # subnormal halves if it were not scaled; a NaN keeps the Gram unscaled
        x = (1e-6 * w).astype(dt)
        x[n // 3] = np.nan
    if kind == "mixed":     # ordinary, huge and infinite samples side by side
        x[::61], x[7::67], x[11::301] = 3e4, 1e18, np.inf
    return x


def _thr(x, m, dist, kind):
    f = np.float64 if kind == "mixed" else x.dtype.type
    if kind == "ties":
        return 3.0
    return float(f(1e-6 if kind == "tiny" else 1.0) * f(0.4 if dist == 2 else 0.4 * np.sqrt(m)))


@pytest.mark.parametrize("dist", [1, 2])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["walk", "ties", "tiny", "mixed"])
def test_rows_are_the_oracles(oracle, dt, dist, kind):
    for nc, tau, m in ((1, 1, 1), (97, 2, 5), (130, 1, 17)):
        x = _series(nc, tau, m, dt, kind, 5)
        thr = _thr(x, m, dist, kind)
        want, e = oracle.RP(x, tau, m, dt(thr), dist)
        assert e == 0 and np.array_equal(_rows(x, nc, tau, m, thr, dist, np.arange(nc)), want)


def _check(nc, tau, m, dt, dist, kind="walk", off=0):
    import torch
    import accrqa_amd as amd
    x = _series(nc, tau, m, dt, kind, nc + m)
    thr = _thr(x, m, dist, kind)
    buf = torch.full((nc * nc + off + 64,), 7, dtype=torch.int8, device="cuda")
    dx = torch.from_numpy(x).cuda()
    amd.rp_device(dx.data_ptr(), x.size, tau, m, thr, dist, buf.data_ptr() + off, 0, x.dtype)
    torch.cuda.synchronize()
    assert bool((buf[:off] == 7).all()) and bool((buf[off + nc * nc:] == 7).all())
    got = buf[off:off + nc * nc].view(nc, nc)
    # the first and last rows, the edges of blocks, and others
    edge = [r + d for r in (0, 32, 64, 256, 1024, nc // 64 * 64, nc // 256 * 256, nc) for d in (-1, 0, 1)]
    more = np.random.default_rng(1).integers(0, nc, 40).tolist()
    rows = np.array(sorted({r for r in edge + more if 0 <= r < nc}))
    want = _rows(x, nc, tau, m, thr, dist, rows)
    assert np.array_equal(got[torch.from_numpy(rows).cuda()].cpu().numpy(), want)
    for r in range(0, nc, 4096):
        assert bool((got[r:r + 4096] == got[:, r:r + 4096].t()).all()), r


@pytest.mark.gpu
@pytest.mark.parametrize("tail", range(16))
@pytest.mark.parametrize("nc,m,dist", [(304, 3, 2), (4640, 2, 1), (304, 16, 1), (4640, 17, 1)])
def test_row_ends(nc, m, dist, tail):
    """Every length of a row's last chunk, small blocks and squares, both forms."""
    _check(nc + tail, 1, m, np.float32, dist, off=tail % 5)


@pytest.mark.gpu
@pytest.mark.parametrize("nc,tau,m,dist,dt", [
    # small blocks, and both sides of the rule that leaves a plot to one store per decision
    (2049, 1, 8, 2, np.float32), (3071, 1, 9, 2, np.float64), (3072, 1, 8, 2, np.float64), (3072, 1, 8, 2, np.float32),
    (3072, 1, 7, 2, np.float64), (3072, 1, 16, 1, np.float64), (3072, 1, 15, 1, np.float64), (1024, 1, 1, 1, np.float64),
    (1028, 1, 2, 1, np.float64), (1022, 1, 8, 1, np.float64), (1535, 1, 16, 2, np.float32), (1537, 1, 16, 2, np.float32),
    (1535, 1, 15, 2, np.float32), (1535, 8, 16, 1, np.float32), (2048, 1, 32, 1, np.float32), (2047, 1, 33, 1, np.float32), (4096, 1, 3, 2, np.float32),
    (13312, 1, 1, 1, np.float32),
    # rows of one dimension, 64-squares
    (13313, 1, 1, 2, np.float32), (3328, 1, 8, 2, np.float32), (3329, 1, 8, 2, np.float32), (4224, 1, 3, 2, np.float32),
    (4225, 1, 3, 2, np.float32), (4671, 2, 16, 1, np.float32), (4609, 3, 32, 1, np.float32),
    (4609, 1, 48, 1, np.float32), (4673, 1, 97, 1, np.float32), (4609, 2, 3, 1, np.float64), (16384, 1, 16, 1, np.float32),
    (12288, 1, 17, 1, np.float32), (16512, 1, 33, 1, np.float32),
    (16385, 1, 3, 2, np.float64), (45057, 1, 16, 1, np.float32)])
def test_small_blocks_and_squares(nc, tau, m, dist, dt):
    _check(nc, tau, m, dt, dist, off=4 if nc % 2 else 0)


@pytest.mark.gpu
@pytest.mark.parametrize("nc,off", [(16512, 0), (16512, 16), (16385, 3), (24577, 0), (12289, 1), (12416, 0)])
@pytest.mark.parametrize("tau,m,dist,dt", [(2, 3, 1, np.float32), (1, 4, 1, np.float32), (2, 16, 1, np.float32),
                                           (3, 32, 1, np.float32), (1, 6, 2, np.float64)])
def test_large_squares_and_rows(nc, off, tau, m, dist, dt):
    _check(nc, tau, m, dt, dist, off=off)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["ties", "tiny", "mixed"])
@pytest.mark.parametrize("nc,m", [(2500, 16), (2500, 20), (2500, 40), (4609, 16), (4609, 20), (4609, 40), (16512, 16),
                                  (16512, 20), (16385, 5), (16385, 20)])
def test_special_values(nc, m, kind):
    """Ties at the threshold, and non-finite norms: pairs of ordinary samples
    keep the Gram's decision, unscaled, with their own error bound."""
    _check(nc, 1, m, np.float32, 1, kind)
