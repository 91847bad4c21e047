"""mista_set_kernel's choices and mista_last_kernel's report of them."""
import numpy as np
import pytest

from us_lab4a_amd import workloads
from us_lab4a_amd.sta import CoherenceFactor, HipSTAProcessor

from parity import say

pytestmark = pytest.mark.gpu

MM = 1e-3


def processor(samples=512):
    """Short windows: every chunking fits."""
    wl = workloads.Workload2D(name="choice", num_elements=20, num_samples=samples, upsampling=4, cf="sign_coherence_factor",
                              grid_x=(-1 * MM, 1 * MM), grid_z=(7.5 * MM, 9 * MM), n_x=70, n_z=90, points=4,
                              point_x=(-1 * MM, 1 * MM), point_z=(7.5 * MM, 9 * MM), seed_points=5, seed_noise=6)
    p = HipSTAProcessor(wl.sta_config(), None, wl.upsampling, CoherenceFactor(wl.cf, wl.cf_param), 0.0, wl.rx_apodization(),
                        storage="f16")
    p.set_grid(wl.grid())
    p.process_echoes(wl.echoes_cpu())
    return p, wl.n_x * wl.n_z


def image(p, n):
    import torch
    v, f = (torch.full((n,), -1.0, dtype=torch.float32, device="cuda") for _ in range(2))
    p.das_device(v, f)
    torch.cuda.synchronize()
    return v.cpu().numpy(), f.cpu().numpy()


WIDE = [(9, 4 | 80 << 16), (9, 4 | 80 << 16 | 1 << 24), (9, 4 | 80 << 16 | 2 << 24)]


def test_report_names_the_kernel():
    """What is reported, set again, runs and reports the same; the kernels of 2048-point
    tiles differ in the report."""
    p, n = processor()
    p.set_kernel(1)
    gv, gf = image(p, n)
    reports = []
    for p0, p1 in WIDE + [(9, 8 | 160 << 16), (9, 4 | 160 << 16 | 2 << 24), (9, 0), (8, 8 | 80 << 16), (6, 16 | 150 << 16), (5, 0), (1, 0)]:
        p.set_kernel(2, p0, p1)
        image(p, n)
        ran = p.last_kernel()
        p.set_kernel(2, *ran)
        v, f = image(p, n)
        say("asked", p0, hex(p1), "ran", ran[0], hex(ran[1]))
        assert ran[0] == p0 and p.last_kernel() == ran
        assert np.array_equal(v, gv) and np.array_equal(f, gf)
        reports.append(ran)
    p.close()
    assert len(set(reports[:len(WIDE)])) == len(WIDE)


@pytest.mark.parametrize("p0", [1, 2, 3])
def test_eight_pairs_on_256_points_run_tiled(p0):
    p, n = processor()
    p.set_kernel(1)
    gv, gf = image(p, n)
    for p1 in (8, 8 | 52 << 16, 8 | 2 << 8 | 76 << 16):
        p.set_kernel(2, p0, p1)
        v, f = image(p, n)
        say("asked", p0, hex(p1), "ran", p.last_kernel())
        assert p.last_kernel()[0] == p0
        assert np.array_equal(v, gv) and np.array_equal(f, gf)
    p.close()


def test_first_frame_does_not_time_what_cannot_win():
    """256 elements over 512 x 512 points, frames of some 22 ms: the first one, which
    times tile shapes and chunkings, takes no more than 5.5 of them and 15 ms (the
    tables)."""
    import time

    import torch
    wl = workloads.Workload2D(name="first", num_elements=256, num_samples=4096, upsampling=8, cf="phase_coherence_factor",
                              grid_x=(-38 * MM, 38 * MM), grid_z=(5 * MM, 75 * MM), n_x=512, n_z=512)
    e = torch.randn(256 * 256 * 4096, device="cuda")
    v, f = (torch.empty(wl.n_x * wl.n_z, device="cuda") for _ in range(2))
    first, steady = [], []
    for _ in range(3):   # (the first handle also loads the kernels)
        p = HipSTAProcessor(wl.sta_config(), None, wl.upsampling, CoherenceFactor(wl.cf, wl.cf_param), 0.0,
                            wl.rx_apodization(), storage="f16")
        p.set_grid(wl.grid())
        for times in (first, steady):
            torch.cuda.synchronize()
            t = time.perf_counter()
            p.process_device(e, wl.num_samples, v, f)
            torch.cuda.synchronize()
            times.append((time.perf_counter() - t) * 1e3)
        p.close()
    say("first frames", [round(t, 1) for t in first], "steady", [round(t, 1) for t in steady], "ms")
    assert min(first) <= 5.5 * min(steady) + 15.0
