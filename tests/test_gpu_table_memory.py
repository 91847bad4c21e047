"""The tiled DAS where its tables do not fit beside what else is on the device."""
import numpy as np
import pytest

from us_lab4a_amd import workloads
from us_lab4a_amd.serve import Engine, Job2D
from us_lab4a_amd.sta import CoherenceFactor, HipSTAProcessor

from parity import say

pytestmark = pytest.mark.gpu

MM = 1e-3
GIB = 1 << 30


def wide_frame():
    """64 channels a side over 1000 x 2000 points: delay table 0.5 GB; kept whole,
    the tiles' tables and sums take 2 GB."""
    return workloads.Workload2D(name="wide", num_elements=64, num_samples=512, upsampling=4, cf="sign_coherence_factor",
                                tx_apod="hanning", grid_x=(-8 * MM, 8 * MM), grid_z=(1 * MM, 10.8 * MM), n_x=1000, n_z=2000,
                                points=6, point_x=(-7 * MM, 7 * MM), point_z=(2 * MM, 9 * MM), seed_points=41, seed_noise=42)


def processor(wl, storage="f32"):
    p = HipSTAProcessor(wl.sta_config(), None, wl.upsampling, CoherenceFactor(wl.cf, wl.cf_param), 0.0, wl.rx_apodization(),
                        tx_apod=wl.tx_apodization(), storage=storage)
    p.set_grid(wl.grid())
    return p


def das(p, v, f):
    import torch
    p.das_device(v, f)
    torch.cuda.synchronize()
    return v.cpu().numpy(), f.cpu().numpy()


def test_frame_runs_where_its_tables_do_not_fit():
    import torch
    wl = wide_frame()
    n = wl.n_x * wl.n_z
    v, f = (torch.empty(n, dtype=torch.float32, device="cuda") for _ in range(2))
    p = processor(wl)
    p.set_kernel(1)
    p.process_device(torch.from_numpy(wl.echoes_cpu()).cuda(), wl.num_samples, v, f)
    torch.cuda.synchronize()
    gv, gf = v.cpu().numpy(), f.cpu().numpy()
    p.set_kernel(0)
    held = []
    while (free := torch.cuda.mem_get_info()[0]) > 3 * GIB // 2:
        held.append(torch.empty(min(free - 5 * GIB // 4, 32 * GIB), dtype=torch.uint8, device="cuda"))
    say("free bytes left", torch.cuda.mem_get_info()[0])
    try:
        for _ in range(2):   # the tuned frame, then one with the tables' slabs built again
            tv, tf = das(p, v.fill_(-1.0), f.fill_(-1.0))
            assert p.last_kernel()[0] >= 0, "the tiled DAS ran"
            assert np.array_equal(tv, gv) and np.array_equal(tf, gf)
    finally:
        del held
        torch.cuda.empty_cache()
    tv, tf = das(p, v.fill_(-1.0), f.fill_(-1.0))
    assert np.array_equal(tv, gv) and np.array_equal(tf, gf)
    p.close()


def job(wl, storage="f32"):
    n = wl.n_x * wl.n_z
    return Job2D(config=wl.sta_config(), upsampling=wl.upsampling, coherence=CoherenceFactor(wl.cf, wl.cf_param), grid=wl.grid(),
                 rx_apod=wl.rx_apodization(), tx_apod=wl.tx_apodization(), echoes=wl.echoes_cpu(),
                 value=np.zeros(n, np.float32), factor=np.zeros(n, np.float32), storage=storage)


def run_jobs(jobs, budget=0):
    """The jobs one after the other through one handle each; the largest number of
    bytes that the engine counted as resident."""
    most = 0
    with Engine(max_inflight=2, hbm_budget=budget, handles_per_shape=1) as eng:
        tickets = [eng.submit(j) for j in jobs]
        while not all(eng.done(t) for t in tickets):
            most = max(most, eng.stats()["resident_bytes"])
        out = [eng.wait(t) for t in tickets]
        most = max(most, eng.stats()["resident_bytes"])
    return out, most


def test_engine_keeps_to_its_budget():
    """Short records over a large grid, where the tiles' tables and sums are most of a
    handle: two jobs that do not fit together wait for each other; one that does not
    fit with whole tables runs in slabs, to the same images."""
    a, b = wide_frame(), wide_frame()
    b.n_z = 1900
    jobs = [job(a), job(b)]
    (sa, sb), _ = run_jobs(jobs)
    assert sa["ok"] and sb["ok"], (sa, sb)
    ref = [(j.value.copy(), j.factor.copy()) for j in jobs]
    fa, fb = sa["footprint"], sb["footprint"]
    say("footprints", fa, fb)
    for budget in (fa + fb - 1, fa - 1):
        again = [job(a), job(b)]
        stats, most = run_jobs(again, budget)
        say("budget", budget, "resident", most, "footprints", [s["footprint"] for s in stats])
        assert all(s["ok"] for s in stats), stats
        assert most <= budget and max(s["footprint"] for s in stats) <= budget
        for j, (v, f) in zip(again, ref):
            assert np.array_equal(j.value, v) and np.array_equal(j.factor, f)
