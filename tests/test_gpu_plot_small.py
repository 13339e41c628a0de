"""Small recurrence plots on both sides of the sizes and dimensions where the
work shape changes: element for element the plot of one store per decision."""
import numpy as np
import pytest

from test_gpu_plot_shapes import _plot

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nc", [2048, 2049, 3071, 3072, 3073, 4607, 4608, 4609, 8191, 8193])
@pytest.mark.parametrize("m,dist,dt", [(1, 1, np.float32), (7, 1, np.float64), (8, 1, np.float32), (8, 2, np.float32),
                                       (9, 2, np.float64)])
def test_plot_small(nc, m, dist, dt):
    import torch
    import accrqa_amd as amd
    x = np.cumsum(np.random.default_rng(nc + m).standard_normal(nc + m - 1)).astype(dt)
    thr = float(np.std(x) * 0.4 * (np.sqrt(m) if dist == 1 else 1.0))
    got = _plot(amd, torch, x, nc, 1, m, thr, dist, nc % 3)
    amd.set_rp_sym(0)
    try:
        ref = _plot(amd, torch, x, nc, 1, m, thr, dist, 0)
    finally:
        amd.set_rp_sym(1)
    assert bool((got == ref).all())
