"""More channels than the 2^32 lanes of one launch take."""
import numpy as np
import pytest

from us_lab4a_amd import workloads
from us_lab4a_amd.sta import CoherenceFactor, HipSTARFProcessor

from parity import say

pytestmark = pytest.mark.gpu

MM = 1e-3


def prepared(elements, d_echoes):
    wl = workloads.Workload2D(name="many", num_elements=elements, num_samples=4, upsampling=4, grid_x=(-1 * MM, 1 * MM),
                              grid_z=(0.01 * MM, 0.05 * MM), n_x=2, n_z=2)
    p = HipSTARFProcessor(wl.sta_config(), None, CoherenceFactor("none", 1.0), 0.0)
    p.set_grid(wl.grid())
    p.prepare_signals_device(d_echoes, 4)
    a = p.download_analytic()
    p.close()
    return a.reshape(-1, 16)


def test_rf_records_of_2_to_the_24_channels():
    import torch
    gen = torch.Generator("cuda").manual_seed(3)
    few = torch.randn(64 * 64, 4, device="cuda", generator=gen)
    say("rf, 4096 x 4096 channels of 4 samples")
    a = prepared(4096, few.repeat(4096, 1).contiguous())
    ref = prepared(64, few)
    assert a.shape == (1 << 24, 16) and np.array_equal(a.reshape(4096, *ref.shape), np.broadcast_to(ref, (4096,) + ref.shape))
