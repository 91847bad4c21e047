"""What the first frame of a process loads."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

FIRST_FRAME = """
import torch
from us_lab4a_amd import workloads
from us_lab4a_amd.sta import CoherenceFactor, HipSTAProcessor
wl = workloads.sta2d_32_small()
v, f = (torch.empty(wl.n_x * wl.n_z, device="cuda") for _ in range(2))
e = torch.randn(32 * 32 * 2048, device="cuda")
p = HipSTAProcessor(wl.sta_config(), None, wl.upsampling, CoherenceFactor(wl.cf, wl.cf_param), 0.0, wl.rx_apodization())
p.set_grid(wl.grid())
p.prepare_signals_device(e, 2048)
torch.cuda.synchronize()
before = torch.cuda.mem_get_info()[0]
p.das_device(v, f)
torch.cuda.synchronize()
print("MIB", (before - torch.cuda.mem_get_info()[0]) >> 20)
"""


def test_first_das_does_not_load_the_no_allocation_scratch():
    """A small frame's tables, sums and the kernels: 38 MiB.  The scratch alone is 256."""
    out = subprocess.run([sys.executable, "-c", FIRST_FRAME], cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert out.returncode == 0, out.stderr[-2000:]
    mib = int(out.stdout.split("MIB")[1])
    print("[gpu-test] device memory taken by the first DAS:", mib, "MiB", flush=True)
    assert mib < 128
