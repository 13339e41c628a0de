"""Recurrence plots of bytes in every work shape (small blocks, 64- and
256-squares, rows), at sizes around the shapes' block edges and lines, on
buffers at odd addresses: element for element the plot of one store per
decision, which other tests hold against the oracle; nothing outside the plot
is written.  Decisions are the reference's, so the bound is equality."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _plot(amd, torch, x, nc, tau, m, thr, dist, off):
    buf = torch.full((nc * nc + off + 64,), 7, dtype=torch.int8, device="cuda")
    dx = torch.from_numpy(x).cuda()
    amd.rp_device(dx.data_ptr(), x.size, tau, m, thr, dist, buf.data_ptr() + off, 0, x.dtype)
    torch.cuda.synchronize()
    assert bool((buf[:off] == 7).all()) and bool((buf[off + nc * nc:] == 7).all())
    return buf[off:off + nc * nc]


@pytest.mark.parametrize("nc,off", [(1, 0), (31, 1), (257, 3), (1000, 0), (3073, 5), (3100, 0), (4160, 16),
                                    (16385, 1), (16512, 0), (16512, 16), (24577, 0)])
@pytest.mark.parametrize("tau,m,dist,dt", [(1, 16, 1, np.float32), (3, 33, 1, np.float32), (2, 3, 1, np.float32),
                                           (1, 4, 1, np.float32), (1, 2, 2, np.float32), (1, 9, 2, np.float32),
                                           (5, 3, 1, np.float64)])
def test_plot_shapes(nc, off, tau, m, dist, dt):
    import torch
    import accrqa_amd as amd
    if nc > 3100 and (m, dist) in ((33, 1), (9, 2)) and nc != 24577:
        pytest.skip("one large size is enough for these")
    rng = np.random.default_rng(nc + m)
    x = np.cumsum(rng.standard_normal(nc + (m - 1) * tau))
    x = (np.round(x) if m == 4 else x).astype(dt)   # m = 4: integers, ties at the threshold
    thr = 3.0 if m == 4 else float(np.std(x) * 0.4 * (np.sqrt(m) if dist == 1 else 1.0)) + 0.1
    got = _plot(amd, torch, x, nc, tau, m, thr, dist, off)
    amd.set_rp_sym(0)
    try:
        ref = _plot(amd, torch, x, nc, tau, m, thr, dist, 0)
    finally:
        amd.set_rp_sym(1)
    assert bool((got == ref).all())


@pytest.mark.parametrize("bad", [np.nan, np.inf, 1e20])
@pytest.mark.parametrize("m", [3, 16])
@pytest.mark.parametrize("nc", [900, 5000, 16500])
def test_plot_shapes_special_values(bad, m, nc):
    import torch
    import accrqa_amd as amd
    x = np.cumsum(np.random.default_rng(3).standard_normal(nc + m - 1)).astype(np.float32)
    x[::97] = bad
    got = _plot(amd, torch, x, nc, 1, m, 5.0, 1, 0)
    amd.set_rp_sym(0)
    try:
        ref = _plot(amd, torch, x, nc, 1, m, 5.0, 1, 0)
    finally:
        amd.set_rp_sym(1)
    assert bool((got == ref).all())
