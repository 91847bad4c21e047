"""What the speed of this package is measured on: whole frames through its public entry points.

The processors take raw echoes and return an image, so most cases are a
frame as an imaging loop runs it (`process_device`): preparation (upsampling,
DC removal, analytic signal), delay-and-sum, coherence factor, envelope.  The
others are the package's remaining paths: real (RF) samples with the row
envelope, a volume, host buffers, a serving round whose frames share one
delay-and-sum launch, and re-imaging prepared signals on a coarse preview
grid.  Sizes are those of `us_lab4a_amd/workloads.py`, `bench.py --mode serve`
and the tests, or generic.

`exact` restates each path in FP64 with plain torch.  A coherence factor is a
discontinuous function of the per-element sums' phases, so frames with one
compare like with like only while the sums keep their bits; records too long
for the on-chip transforms are taken without one.
"""
import math

import numpy as np
import torch

from us_lab4a_amd import imaging
from us_lab4a_amd.sta import (CoherenceFactor, HipSTA3DProcessor, HipSTAProcessor, HipSTARFProcessor, SA3DConfiguration,
                              STAConfiguration, das_batch_device)

MM = 1e-3
FS, C, PITCH = 40e6, 1540.0, 0.3 * MM
CF = {"none": "none", "pcf": "phase_coherence_factor", "scf": "sign_coherence_factor"}
STORAGE_BYTES = {"f32": 8, "f16": 4, "bf16": 4, "rf": 4}


def _frame(name, elements, samples, up, n_x, n_z, cf, storage, **more):
    c = {"name": name, "kind": "frame", "elements": elements, "first_tx": 0, "num_tx": elements, "samples": samples,
         "up": up, "n_x": n_x, "n_z": n_z, "width_mm": elements * 0.3, "z0_mm": 5.0, "z1_mm": 55.0, "fc": 5e6, "cf": cf,
         "storage": storage, "rx_window": "hanning", "tx_window": "", "peak_offset": 0.0}
    c.update(more)
    return c


def listed():
    return [
        # the small probe of workloads.sta2d_32_small: launches and latency count
        _frame("small_32_f32", 32, 2048, 4, 256, 256, "none", "f32", width_mm=20.0, tx_window="hanning"),
        # the serving mix's short jobs
        _frame("serve_64_pcf_f16", 64, 2048, 8, 128, 128, "pcf", "f16", z1_mm=35.0),
        # the headline frame (workloads.sta2d_128_pcf), in both storages it is quoted for
        _frame("headline_128_pcf_f32", 128, 4096, 8, 512, 1024, "pcf", "f32", width_mm=38.0, z1_mm=65.0),
        _frame("headline_128_pcf_f16", 128, 4096, 8, 512, 1024, "pcf", "f16", width_mm=38.0, z1_mm=65.0),
        # odd sizes everywhere: a transmit sub-range, an odd record, a grid that no tile divides, a pulse-peak offset
        _frame("ragged_100_scf_bf16", 100, 3001, 4, 301, 517, "scf", "bf16", first_tx=7, num_tx=75, width_mm=27.0,
               z1_mm=50.0, peak_offset=1.5),
        # a large aperture: more than 128 transmits
        _frame("large_256_pcf_f16", 256, 4096, 8, 512, 512, "pcf", "f16", z1_mm=65.0),
        # long records: the analytic signal's transforms no longer fit on chip
        _frame("long_192_none_f16", 192, 8192, 8, 256, 512, "none", "f16", z1_mm=65.0),
        # DefaultSTAProcessor's path: real samples, signed values, row envelope
        _frame("rf_128_scf", 128, 2048, 4, 256, 512, "scf", "rf", kind="rf", rx_window="rectangular", z1_mm=35.0),
        # a sparse 3-D acquisition (workloads.sta3d_sparse's array) on a smaller volume
        {"name": "volume_1024x64_scf_f32", "kind": "volume", "array_x": 32, "array_y": 32, "num_tx": 64, "samples": 2048,
         "up": 4, "n_x": 64, "n_y": 64, "n_z": 128, "width_mm": 10.0, "z0_mm": 10.0, "z1_mm": 35.0, "fc": 3e6,
         "cf": "scf", "storage": "f32", "peak_offset": 0.0},
        # a frame from host memory and back, as ArrayProcessor::process callers run it
        _frame("host_64_none_f32", 64, 2048, 4, 256, 256, "none", "f32", kind="host", z1_mm=35.0),
        # one round of a request loop: four jobs prepared, their delay-and-sum in one batch
        _frame("round_4x64_pcf_f16", 64, 4096, 8, 256, 512, "pcf", "f16", kind="round", frames=4, z1_mm=65.0),
        # re-imaging prepared signals on a coarse preview grid (too coarse for the tiles' signal windows)
        _frame("preview_192_scf_f16", 192, 4096, 8, 96, 96, "scf", "f16", kind="image", z1_mm=65.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _pairs(c):
    if c["kind"] == "volume":
        return c["n_x"] * c["n_y"] * c["n_z"] * c["num_tx"] * c["array_x"] * c["array_y"]
    return c["n_x"] * c["n_z"] * c["num_tx"] * c["elements"] * c.get("frames", 1)


def draw(rng):
    kind = rng.choice(["frame"] * 6 + ["long", "rf", "volume", "host", "round", "image"])
    while True:
        z1 = rng.uniform(25.0, 65.0)
        if kind == "volume":
            a = rng.choice([8, 12, 16, 24, 32])
            c = {"kind": "volume", "array_x": a, "array_y": a, "num_tx": rng.randint(4, 64), "samples": _log(rng, 512, 2048),
                 "up": rng.choice([2, 4]), "n_x": rng.randint(12, 64), "n_y": rng.randint(12, 64),
                 "n_z": rng.randint(24, 128), "width_mm": rng.uniform(4.0, 12.0), "z0_mm": 8.0,
                 "z1_mm": min(z1, 35.0), "fc": 3e6, "cf": rng.choice(["none", "scf", "pcf"]),
                 "storage": rng.choice(["f32", "f16"]), "peak_offset": 0.0}
        else:
            long = kind == "long"
            n = _log(rng, 16, 128 if long or kind in ("host", "round") else 256)
            tx = n if rng.random() < 0.6 else rng.randint(max(1, n // 4), n)
            up = 8 if long else rng.choice([2, 4, 8])
            ns = _log(rng, 4500, 8192) if long else _log(rng, 512, 2048 if kind in ("host", "rf") else 4096)
            c = _frame("", n, ns, up, _log(rng, 48, 512), _log(rng, 64, 1024),
                       "none" if long else rng.choice(["none", "pcf", "pcf", "scf"]),
                       rng.choice(["f32", "f16", "bf16"]), kind=kind if kind in ("rf", "host", "round", "image") else "frame",
                       first_tx=rng.randint(0, n - tx), num_tx=tx, z1_mm=min(z1, ns / FS * C / 2 * 900.0),
                       rx_window=rng.choice(["hanning", "rectangular", "blackman"]),
                       tx_window="hanning" if tx > 1 and rng.random() < 0.3 else "",
                       peak_offset=rng.choice([0.0, 0.0, 1.5]), width_mm=n * 0.3 * rng.uniform(0.7, 1.0))
            del c["name"]
            if c["z1_mm"] < 8.0:
                continue
            if kind == "rf":
                c.update(up=4, storage="rf", rx_window="rectangular", tx_window="",
                         cf=rng.choice(["none", "scf"]))
            if kind == "round":
                c["frames"] = rng.randint(2, 4)
            if kind == "image":
                c.update(n_x=_log(rng, 48, 128), n_z=_log(rng, 64, 192))
        if 2e6 < _pairs(c) <= (4e9 if kind == "long" else 1.2e10):
            return c


# ---------------------------------------------------------------- inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _elements(case):
    """(tx positions, rx positions) as FP64 [.][2] arrays (x, y), from the float32 values the processors are given."""
    if case["kind"] == "volume":
        pos = imaging.element_positions_2d_array(PITCH, case["array_x"], 0.0, PITCH, case["array_y"], 0.0).astype(np.float64)
        step = pos.shape[0] / case["num_tx"]
        return pos[[int(k * step) for k in range(case["num_tx"])]], pos
    pitch, n = float(np.float32(PITCH)), case["elements"]
    pos = np.stack([np.arange(n) * pitch - (n - 1) * pitch / 2, np.zeros(n)], axis=-1)
    return pos[case["first_tx"]:case["first_tx"] + case["num_tx"]], pos


def _points(case):
    """Grid points [n][3] (x, y, z) float32, z fastest."""
    half = case["width_mm"] * MM / 2
    if case["kind"] == "volume":
        ax = [np.linspace(-half, half, case["n_x"]), np.linspace(-half, half, case["n_y"]),
              np.linspace(case["z0_mm"] * MM, case["z1_mm"] * MM, case["n_z"])]
        return np.stack(np.meshgrid(*ax, indexing="ij"), axis=-1).reshape(-1, 3).astype(np.float32)
    g = imaging.rectangular_grid(-half, half, case["n_x"], case["z0_mm"] * MM, case["z1_mm"] * MM, case["n_z"])
    return np.stack([g["x"], g["y"], g["z"]], axis=-1).reshape(-1, 3)


def _echoes(case, seed):
    """[tx][rx][samples] float32 on the GPU: point scatterers seen by a Gaussian-modulated pulse, plus white noise at 30 dB."""
    g = _gen(seed)
    tx, rx = (torch.from_numpy(a).cuda() for a in _elements(case))
    ns, fc, count = case["samples"], case["fc"], 24
    half = case["width_mm"] * MM / 2
    u = torch.rand((count, 4), generator=g, device="cuda", dtype=torch.float64)
    sx = (2 * u[:, 0] - 1) * half
    sy = (2 * u[:, 1] - 1) * (half if case["kind"] == "volume" else 0.0)
    sz = (case["z0_mm"] + (case["z1_mm"] - case["z0_mm"]) * u[:, 2]) * MM
    out = torch.zeros((len(tx) * len(rx), ns), dtype=torch.float32, device="cuda")
    a = (math.pi * fc * 0.6) ** 2 / (4 * math.log(10.0 ** 0.3))
    reach = int(math.sqrt(math.log(1e3) / a) * FS) + 1
    k = torch.arange(-reach, reach + 1, device="cuda")
    for s in range(count):
        dist = lambda e: torch.sqrt((sx[s] - e[:, 0]) ** 2 + (sy[s] - e[:, 1]) ** 2 + sz[s] ** 2)  # noqa: E731
        centre = ((dist(tx)[:, None] + dist(rx)[None]) * (FS / C)).reshape(-1, 1)
        i = centre.round().long() + k
        t = (i - centre) / FS
        pulse = ((0.5 + 0.5 * u[s, 3]) * torch.exp(-a * t * t) * torch.cos(2 * math.pi * fc * t)).float()
        pulse = torch.where((i >= 0) & (i < ns), pulse, torch.zeros_like(pulse))
        i = i.clamp(0, ns - 1)
        # one scatterer touches a sample of a channel once, but for the clamped ends, whose pulse is zero
        out.scatter_add_(1, i, pulse)
    rms = float(out.double().square().mean().sqrt())
    for row in out.split(16384):
        row += torch.randn(row.shape, generator=g, device="cuda") * (rms * 10.0 ** -1.5)
    return out.view(len(tx), len(rx), ns)


def _windows(case):
    rx = imaging.window(case["rx_window"], case["elements"])
    return rx, imaging.window(case["tx_window"], case["num_tx"]) if case["tx_window"] else None


def _processor(case):
    cf = CoherenceFactor(CF[case["cf"]], 1.0)
    if case["kind"] == "volume":
        pos = imaging.element_positions_2d_array(PITCH, case["array_x"], 0.0, PITCH, case["array_y"], 0.0)
        step = len(pos) / case["num_tx"]
        cfg = SA3DConfiguration(sampling_frequency=FS, propagation_speed=C, center_frequency=case["fc"], tx_elem_pos=pos,
                                rx_elem_pos=pos, active_tx_elem=[int(k * step) for k in range(case["num_tx"])],
                                active_rx_elem=list(range(len(pos))))
        p = HipSTA3DProcessor(cfg, None, case["up"], cf, case["peak_offset"], np.ones(len(pos), np.float32),
                              storage=case["storage"])
        p.set_grid(_points(case).reshape(case["n_x"] * case["n_y"], case["n_z"], 3), ny=case["n_y"])
        return p
    cfg = STAConfiguration(num_elements=case["elements"], pitch=PITCH, sampling_frequency=FS, propagation_speed=C,
                           center_frequency=case["fc"], first_tx_elem=case["first_tx"],
                           last_tx_elem=case["first_tx"] + case["num_tx"] - 1)
    if case["kind"] == "rf":
        p = HipSTARFProcessor(cfg, None, cf, case["peak_offset"])
    else:
        rx, tx = _windows(case)
        p = HipSTAProcessor(cfg, None, case["up"], cf, case["peak_offset"], rx, tx_apod=tx, storage=case["storage"])
    p.set_grid(_points(case)[:, [0, 2]].reshape(case["n_x"], case["n_z"], 2))
    return p


_STREAM = []


def _stream():
    """The one stream that this program's frames run on."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


def prepare(case, seed):
    """Echoes, the image buffers and a processor whose geometry (grid, tables, tuned tiles) is laid out: one frame has run."""
    n = len(_points(case))
    frames = case.get("frames", 1)
    echoes = [_echoes(case, seed * 8 + k) for k in range(frames)]
    state = {"case": case, "echoes": echoes, "procs": [_processor(case) for _ in echoes],
             "value": [torch.empty(n, device="cuda") for _ in echoes], "factor": [torch.empty(n, device="cuda") for _ in echoes]}
    if case["kind"] == "host":
        state["host"] = echoes.pop().cpu().pin_memory().numpy()
        state["procs"][0].process_echoes(state["host"])
        return state
    torch.cuda.synchronize()
    for p, e, v, f in zip(state["procs"], echoes, state["value"], state["factor"]):
        p.process_device(e, case["samples"], v, f, stream=_stream())
    torch.cuda.synchronize()
    return state


def run(state):
    case, s = state["case"], _stream()
    p, v, f = state["procs"], state["value"], state["factor"]
    kind = case["kind"]
    if kind == "host":
        return p[0].process_echoes(state["host"])
    if kind == "image":
        p[0].das_device(v[0], f[0], stream=s)
    elif kind == "round":
        for q, e in zip(p, state["echoes"]):
            q.prepare_signals_device(e, case["samples"], stream=s)
        das_batch_device(p, v, f, stream=s)
    else:
        p[0].process_device(state["echoes"][0], case["samples"], v[0], f[0], stream=s)
        if kind == "rf":
            p[0].envelope_device(v[0], case["n_x"], case["n_z"], stream=s)
    return {"value": v, "factor": f}


# ---------------------------------------------------------------- what a pass cannot do without

def work(case):
    """Echoes in and images out; about 13 operations a pixel and (tx, rx) pair (position, two interpolations, two weighted
    sums), 108 a complex upsampled sample (27 taps, real) and the two half-size transforms.  Re-imaging reads the prepared
    signals instead."""
    frames = case.get("frames", 1)
    npix = case["n_x"] * case["n_z"] * case.get("n_y", 1)
    nch = case["num_tx"] * (case["array_x"] * case["array_y"] if case["kind"] == "volume" else case["elements"])
    length = case["samples"] * case["up"]
    flops = 13.0 * npix * nch
    byts = npix * 8.0
    if case["kind"] == "image":
        byts += nch * length * STORAGE_BYTES[case["storage"]]
    else:
        byts += nch * case["samples"] * 4.0
        m = (length + 1024) / 2
        flops += nch * (54.0 * length + (0 if case["kind"] == "rf" else 2 * 5 * m * math.log2(m)))
    return {"bytes": byts * frames, "flops": flops * frames}


# ---------------------------------------------------------------- FP64 restatement

def _fast_even(n):
    n += n & 1
    while True:
        m = n
        for q in (2, 3, 5):
            while m % q == 0:
                m //= q
        if m == 1:
            return n
        n += 2


def _kaiser_sinc(periods, n, beta):
    w = np.linspace(-periods, periods, n)
    return np.sinc(w) * np.i0(beta * np.sqrt(np.maximum(0.0, 1 - np.linspace(-1, 1, n) ** 2))) / np.i0(beta)


def _filter(case):
    up = case["up"]
    if case["kind"] == "rf":
        return _kaiser_sinc(10.0, 81, 5.0)
    tol = 80.0
    size = math.ceil((tol - 7.95) / (2.285 * (0.4 / up) * math.pi) + 1.0)
    n = int(math.ceil((size - 1) / (2.0 * up)) * 2 * up) + 1
    return _kaiser_sinc((n - 1) / (2.0 * up), n, 0.1102 * (tol - 8.7))


def _analytic64(x):
    n = x.shape[-1]
    nf = max(2048, _fast_even(n + 1024))
    f = torch.fft.fft(x, n=nf)
    f[..., 1:nf // 2] *= 2
    f[..., nf // 2 + 1:] = 0
    return torch.fft.ifft(f)[..., :n]


def _signals64(case, raw):
    """raw [channels][samples] -> upsampled, DC-free (analytic, or real for RF) signals in FP64."""
    up, taps = case["up"], torch.from_numpy(_filter(case)).cuda()
    x = torch.zeros((raw.shape[0], raw.shape[1] * up), dtype=torch.float64, device="cuda")
    x[:, ::up] = raw.double()
    n = len(taps)
    size = _fast_even(x.shape[1] + n)
    y = torch.fft.irfft(torch.fft.rfft(x, n=size) * torch.fft.rfft(taps, n=size), n=size)
    y = y[:, (n - 1) // 2:(n - 1) // 2 + x.shape[1]]
    y = y - y.mean(dim=1, keepdim=True)
    return y if case["kind"] == "rf" else _analytic64(y)


def _image64(case, echoes):
    up = case["up"]
    p = torch.from_numpy(_points(case)).cuda().double()
    tx, rx = (torch.from_numpy(a).cuda() for a in _elements(case))
    scale = float(np.float32(FS)) * up / float(np.float32(C))
    delay = lambda e: torch.sqrt((p[:, 0] - e[0]) ** 2 + ((p[:, 1] - e[1]) ** 2 if case["kind"] == "volume" else 0.0)  # noqa: E731
                                 + p[:, 2] ** 2) * scale
    offset = FS * up * case["peak_offset"] / case["fc"]
    dtx = torch.stack([delay(e) for e in tx]) + offset
    if case["kind"] in ("volume", "rf"):
        wr, wt = torch.ones(len(rx), dtype=torch.float64, device="cuda"), torch.ones(len(tx), dtype=torch.float64, device="cuda")
    else:
        a, b = _windows(case)
        wr = torch.from_numpy(a).cuda().double()
        wt = torch.ones(len(tx), dtype=torch.float64, device="cuda") if b is None else torch.from_numpy(b).cuda().double()
    n = len(p)
    real = case["kind"] == "rf"
    total = torch.zeros(n, dtype=torch.float64 if real else torch.complex128, device="cuda")
    signs = torch.zeros(n, dtype=torch.float64, device="cuda")
    m = torch.zeros((4, n), dtype=torch.float64, device="cuda")
    step = max(1, min(len(tx), (1 << 25) // n))
    for r in range(len(rx)):
        sig = _signals64(case, echoes[:, r])
        last = sig.shape[1] - 1
        drx = delay(rx[r])
        acc = torch.zeros_like(total)
        for t in range(0, len(tx), step):
            pos = dtx[t:t + step] + drx
            i = pos.long()
            k = pos - i
            i = i.clamp(0, last - 1)
            s = sig[t:t + step]
            v = s.gather(1, i)
            v = v + k * (s.gather(1, i + 1) - v)
            v *= ((pos >= 0) & (pos < last)) * (wt[t:t + step] * wr[r])[:, None]
            acc += v.sum(dim=0)
        total += acc
        if case["cf"] == "pcf":
            phi = acc.angle()
            aux = phi - torch.where(phi < 0, -math.pi, math.pi)
            m += torch.stack([phi, phi * phi, aux, aux * aux])
        signs += torch.where((acc if real else acc.real) >= 0, 1.0, -1.0)
    count = len(rx)
    value = (total if real else total.abs()) / (len(tx) * count)
    if real:
        value = _analytic64(value.view(case["n_x"], case["n_z"])).abs().reshape(-1)
    if case["cf"] == "pcf":
        m /= count
        sigma = torch.sqrt(torch.minimum(m[1] - m[0] ** 2, m[3] - m[2] ** 2).clamp(min=0))
        factor = (1 - sigma * (math.sqrt(3.0) / math.pi)).clamp(min=0)
    elif case["cf"] == "scf":
        q = signs / count
        factor = (1 - torch.sqrt(1 - q * q)).abs()
    else:
        factor = torch.ones_like(value)
    return value, factor


def exact(case, seed):
    images = [_image64(case, _echoes(case, seed * 8 + k)) for k in range(case.get("frames", 1))]
    if case["kind"] == "host":
        v, f = images[0]
        return v.cpu().numpy().reshape(case["n_x"], case["n_z"]), f.cpu().numpy().reshape(case["n_x"], case["n_z"])
    return {"value": [v for v, _ in images], "factor": [f for _, f in images]}
