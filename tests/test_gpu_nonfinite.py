"""Infinities and NaN in the echoes: where they may go and where not."""
import numpy as np
import pytest

import oracle
from us_lab4a_amd import workloads
from us_lab4a_amd.sta import CoherenceFactor, HipSTAProcessor, HipSTARFProcessor, das_batch_device

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


@pytest.mark.parametrize("weight", [np.inf, np.nan])
def test_infinite_weight_of_an_unheard_element(weight):
    """Pixels whose echoes by way of element 0 all lie past the record's end: its
    weight does not matter to them in any form of the kernel."""
    import torch
    wl = workloads.Workload2D(name="unheard", num_elements=32, num_samples=512, upsampling=4, cf="sign_coherence_factor",
                              grid_x=(-4 * MM, 4.5 * MM), grid_z=(8 * MM, 9.6 * MM), n_x=40, n_z=48, points=4,
                              point_x=(-4 * MM, 4 * MM), point_z=(8 * MM, 9.6 * MM), seed_points=9, seed_noise=10)
    n = wl.n_x * wl.n_z
    say("element 0 has weight", weight)

    def processor():
        rx = np.ones(32, np.float32)
        p = HipSTAProcessor(wl.sta_config(), None, 4, CoherenceFactor(wl.cf, 1.0), 0.0, rx)
        p.set_grid(wl.grid())
        p.process_echoes(wl.echoes_cpu())   # tuned
        rx[0] = weight
        p.set_rx_apod(rx)
        return p

    def out():
        return [torch.full((n,), -1.0, dtype=torch.float32, device="cuda") for _ in range(2)]

    p, q = processor(), processor()
    p.set_kernel(1)
    gather = out()
    p.das_device(*gather)
    frames = {}
    for p0 in (0, 1, 6):
        frames["tile", p0] = out()
        p.set_kernel(2 if p0 else 0, p0)
        p.das_device(*frames["tile", p0])
    frames["noalloc"] = out()
    p.das_device_noalloc(*frames["noalloc"])
    frames["batch"], other = out(), out()
    das_batch_device([p, q], [frames["batch"][0], other[0]], [frames["batch"][1], other[1]])
    torch.cuda.synchronize()
    finite = torch.isfinite(gather[0])
    assert 0 < int(finite.sum()) < n
    for name, f in frames.items():
        for got, want in zip(f, gather):
            assert np.array_equal(got.cpu().numpy(), want.cpu().numpy(), equal_nan=True), name
    p.close()
    q.close()
