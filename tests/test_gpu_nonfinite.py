"""Infinities and NaN in the echoes: where they may go and where not."""
import numpy as np
import pytest

import oracle
from us_lab4a_amd import workloads
from us_lab4a_amd.sta import CoherenceFactor, HipSTARFProcessor

from parity import say

pytestmark = pytest.mark.gpu

MM = 1e-3


# 256 lanes; 1024 lanes; 1024 lanes with 16 tiles a wave
@pytest.mark.parametrize("samples", [600, 5000, 9000])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
def test_rf_dead_zone_sample_reaches_its_filter_only(samples, value):
    """A sample q in the dead zone, which the mean leaves out: the outputs 4q - 40
    to 4q + 40 of the 81-tap x 4 filter, and no others, and only in its channel."""
    wl = workloads.Workload2D(name="nonfinite", num_elements=3, num_samples=samples, upsampling=4, dead_zone_m=4 * MM,
                              grid_x=(-1 * MM, 1 * MM), grid_z=(2 * MM, 6 * MM), n_x=8, n_z=8, points=4,
                              point_x=(-1 * MM, 1 * MM), point_z=(2 * MM, 6 * MM), seed_points=7, seed_noise=8)
    echoes = wl.echoes_cpu()
    q = 100
    echoes[1, 2, q] = 0.0
    a64 = oracle.prepare_rf(oracle.cfg_for(wl), echoes, np.float64)
    echoes[1, 2, q] = value
    say("rf", samples, value)
    p = HipSTARFProcessor(wl.sta_config(), None, CoherenceFactor("none", 1.0), 0.0)
    p.set_grid(wl.grid())
    p.process_echoes(echoes)
    a = p.download_analytic()
    p.close()
    reach = np.zeros(a.shape, bool)
    reach[1, 2, 4 * q - 40:4 * q + 41] = True
    assert a.shape == a64.shape
    assert not np.isfinite(a[reach]).any()
    err = float(np.abs(a[~reach] - a64[~reach]).max() / np.abs(a64).max())
    say("error / peak", f"{err:.2e}")
    assert err <= 2e-6
