"""Performance cases of the delay-and-sum framework.

Each case is one call a beamforming program makes through the package's public
entry points: a resident plan run on new channel data (every summed
dimension), the ``DAS`` facade, the MEX matrix contract, a ragged batch, the
analytic signal and the RF-to-IQ front end. Sizes come from the benchmark
acquisitions (``ustb_amd.configs``) and the tests, with odd ones among them.

The channel data are echoes of point scatterers (``ustb_amd.synth``) plus
white noise, made from the seed alone. ``exact`` recomputes every output in
64 bits with plain torch from the definitions: delays and weights are rounded
to single where das.m hands singles to its beamformer, and the angular
frequency of the phase is das_c's single-precision one; all else is FP64.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from ustb_amd import ops, synth
from ustb_amd.batch import Batch
from ustb_amd.das import DAS
from ustb_amd.enums import Dimension, Interpolation, Window
from ustb_amd.geometry import make_plan
from ustb_amd.preprocess import matlab_lowpass, python_lowpass
from ustb_amd.uff import Apodization, ChannelData, LinearArray, LinearScan, MatrixArray, SectorScan, Wave

C = 1540.0
F_NUMBER = 1.7
DIMS = {"none": Dimension.none, "receive": Dimension.receive, "transmit": Dimension.transmit, "both": Dimension.both}
# terms (pixel x channel x wave x frame) of the largest listed case, the volume
MAX_TERMS = 96 * 96 * 128 * 1024 * 25


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def _das(name, entry, setup, N, W, L, nx, nz, F=1, rf=False, cubic=False, dim="both", phase="separable", ny=1):
    return {"name": name, "entry": entry, "setup": setup, "N": N, "W": W, "L": L, "F": F, "nx": nx, "ny": ny, "nz": nz,
            "rf": rf, "cubic": cubic, "dim": dim, "phase": phase}


def listed():
    return [
        # the smallest imaging call: one plane wave on a linear array, a live B-mode frame from RF data
        _das("plane_wave_rf", "plan", "linear", 128, 1, 2048, 256, 256, rf=True),
        # what a script calls: the facade's go() on RF data in hand (analytic signal, cached plan, beamforming)
        _das("facade_rf", "go", "linear", 128, 11, 1600, 193, 321, rf=True),
        # coherent plane-wave compounding of IQ data, fine grid, cubic interpolation (the default benchmark)
        _das("compound_iq_cubic", "plan", "linear", 128, 75, 1024, 512, 1024, cubic=True),
        # a cine loop: every frame of a recording with one plan, odd grid and trace length
        _das("compound_cine", "plan", "linear", 128, 11, 1001, 301, 387, F=16),
        # per-channel images summed over the diverging waves (input of coherence and adaptive methods), das_c's phase
        _das("channel_images", "plan", "phased", 64, 31, 2048, 256, 1024, F=8, dim="transmit", phase="dasc"),
        # per-wave images, then the coherence factor over the waves
        _das("wave_images_cf", "plan_cf", "phased", 64, 31, 1500, 193, 512, F=4, dim="receive"),
        # delayed data of every channel and wave, nothing summed (input of adaptive beamformers)
        _das("delayed_data", "plan", "linear", 128, 5, 1024, 150, 201, dim="none"),
        # the MEX contract on device matrices, as a MATLAB or Python program with delays of its own calls it
        _das("matrix_iq", "matrix", "linear", 128, 25, 1024, 256, 256),
        # one volume of a matrix array, the largest single call
        _das("volume", "plan", "volume", 1024, 25, 512, 96, 128, ny=96),
        # many acquisitions of different sizes in one launch
        _das("ragged_batch", "batch", "linear", 128, 11, 1024, 255, 255, F=1) | {"count": 12},
        # the analytic signal of a recording whose length is no product of small primes
        {"name": "analytic_signal", "entry": "hilbert", "N": 128, "W": 75, "L": 1527, "F": 1},
        # RF to IQ: down-mixing, the MATLAB flavour's filter, decimation by two
        {"name": "rf_to_iq", "entry": "demodulate", "N": 128, "W": 128, "L": 2048, "F": 1, "zero_phase": False, "down": 2},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    entry = rng.choice(["plan", "plan", "plan", "plan", "plan", "plan_cf", "go", "matrix", "matrix", "volume", "batch",
                        "hilbert", "demodulate"])
    if entry == "hilbert":
        L = log(200, 6000)
        return {"entry": entry, "N": log(16, 256), "W": log(1, 75), "F": rng.choice([1, 1, 2]),
                "L": L if rng.random() < 0.5 else 64 * max(4, L // 64)}
    if entry == "demodulate":
        return {"entry": entry, "N": log(16, 192), "W": log(1, 128), "L": log(500, 4000), "F": 1,
                "zero_phase": rng.random() < 0.4, "down": rng.choice([1, 2, 2, 3, 4])}
    if entry == "volume":
        g, m = rng.choice([1, 2, 3, 4, 5]), rng.choice([8, 12, 16, 24, 32])
        return _cap(_das("", "plan", "volume", m * m, g * g, log(300, 800), log(20, 96), log(48, 160), ny=log(20, 96)))
    if entry == "plan_cf":
        return _cap(_das("", entry, rng.choice(["linear", "phased"]), log(32, 128), log(3, 40), log(700, 2100),
                         log(60, 300), log(120, 700), F=log(1, 6), dim="receive"))
    setup = rng.choice(["linear", "linear", "phased"])
    case = _das("", entry, setup, log(32, 192), log(1, 80), log(600, 2300), log(60, 520), log(100, 1024),
                F=rng.choice([1, 1, log(2, 20)]), rf=setup == "linear" and rng.random() < 0.4,
                cubic=rng.random() < 0.3, dim=rng.choice(["both", "both", "both", "transmit", "receive", "none"]),
                phase=rng.choice(["separable", "separable", "dasc"]))
    if entry == "batch":
        case.update(dim="both", F=1, rf=False, phase="separable", W=min(case["W"], 31), count=log(3, 24))
    if entry == "go":
        case.update(phase="separable")
    return _cap(case)


def _terms(case):
    return case["nx"] * case["ny"] * case["nz"] * case["N"] * case["W"] * case["F"] * case.get("count", 1)


def _out_values(case):
    P, dim = case["nx"] * case["ny"] * case["nz"] * case["F"] * case.get("count", 1), case["dim"]
    return P * (case["N"] if dim in ("none", "transmit") else 1) * (case["W"] if dim in ("none", "receive") else 1)


def _cap(case):
    """A drawn case within the cost of the largest listed one: das_c's phase, the matrix contract, dimension none and
    cubic sampling cost several times a term of the volume, so they get fewer."""
    most = MAX_TERMS * (0.08 if case["entry"] == "matrix" or case["dim"] in ("none", "receive") or case["phase"] == "dasc"
                        else 0.25)
    while _terms(case) > most or _out_values(case) > 1.5e8:
        big = max(("nx", "nz", "F", "W"), key=lambda k: case[k])
        case[big] = max(1, int(case[big] * 0.7))
    del case["name"]
    return case


# ---------------------------------------------------------------------------
# Acquisitions
# ---------------------------------------------------------------------------
def _acquisition(case):
    """Probe, waves, scan, apodization and sampling of a case: the benchmark's linear, phased and matrix arrays."""
    N, W, L = case["N"], case["W"], case["L"]
    a = {"waves": [], "sources": None, "angles": None}
    if case["setup"] == "linear":
        a["f0"], fs = 5.2e6, 20.8e6 if case["rf"] else 10.4e6
        zmax = min(50e-3, 0.42 * C * L / fs)
        a["probe"] = LinearArray(N, 0.3e-3)
        a["angles"] = np.deg2rad(np.linspace(-16.0, 16.0, W)) if W > 1 else np.zeros(1)
        a["waves"] = [Wave.plane(t, sound_speed=C) for t in a["angles"]]
        a["axes"] = (np.linspace(-19e-3, 19e-3, case["nx"]), np.zeros(1), np.linspace(5e-3, zmax, case["nz"]))
        a["scan"] = LinearScan(a["axes"][0], a["axes"][2])
    elif case["setup"] == "phased":
        a["f0"], fs = 2.5e6, 10e6
        zmax = min(120e-3, 0.42 * C * L / fs)
        a["probe"] = LinearArray(N, 0.2e-3)
        angles = np.deg2rad(np.linspace(-45.0, 45.0, W)) if W > 1 else np.zeros(1)
        a["sources"] = [(-10e-3 * math.sin(t), 0.0, -10e-3 * math.cos(t)) for t in angles]
        a["axes"] = (np.deg2rad(np.linspace(-45.0, 45.0, case["nx"])), np.zeros(1), np.linspace(1e-3, zmax, case["nz"]))
        a["scan"] = SectorScan(a["axes"][0], a["axes"][2])
    else:
        m, g = math.isqrt(N), math.isqrt(W)
        a["f0"], fs = 3e6, 7.5e6
        zmax = min(35e-3, 0.42 * C * L / fs)
        a["probe"] = MatrixArray(m, m, 0.3e-3)
        grid = np.linspace(-3e-3, 3e-3, g) if g > 1 else np.zeros(1)
        a["sources"] = [(x, y, -10e-3) for x in grid for y in grid]
        a["axes"] = (np.linspace(-10e-3, 10e-3, case["nx"]), np.linspace(-10e-3, 10e-3, case["ny"]),
                     np.linspace(5e-3, zmax, case["nz"]))
        a["scan"] = LinearScan(a["axes"][0], a["axes"][2], a["axes"][1])
    if a["sources"] is not None:
        a["waves"] = [Wave.spherical(*s, sound_speed=C, origin=s) for s in a["sources"]]
    a["zmax"], a["fs"], a["fd"] = zmax, fs, 0.0 if case["rf"] else a["f0"]
    # per-channel and delayed data are kept unweighted in receive, as the benchmark's dimension transmit is
    a["rx"] = case["dim"] in ("both", "receive")
    a["tx"] = case["setup"] == "linear" and not case["rf"]
    return a


def _apodizations(a):
    f = (F_NUMBER, F_NUMBER)
    return (Apodization(Window.tukey25, f_number=f) if a["rx"] else Apodization(),
            Apodization(Window.tukey25, f_number=f) if a["tx"] else Apodization())


def _plan(case, a):
    rx, tx = _apodizations(a)
    return make_plan(a["probe"], a["scan"], a["waves"], n_samples=case["L"], n_frames=case["F"],
                     sampling_frequency=a["fs"], initial_time=0.0, modulation_frequency=a["fd"], sound_speed=C,
                     receive_apodization=rx, transmit_apodization=tx, dimension=DIMS[case["dim"]],
                     interpolation=Interpolation.cubic if case["cubic"] else Interpolation.linear,
                     separable_phase=case["phase"] == "separable")


def _echoes(case, a, seed):
    """(F, W, N, L) channel data of 120 scatterers moving with the frames: float32 RF, or complex64 IQ, plus noise."""
    rng = np.random.default_rng(seed)
    K, F = 120, case["F"]
    depth = rng.uniform(4e-3, 0.95 * a["zmax"], K)
    if case["setup"] == "phased":
        t = rng.uniform(-math.pi / 4, math.pi / 4, K)
        pts = np.stack([depth * np.sin(t), np.zeros(K), depth * np.cos(t)], 1)
    else:
        half = 10e-3 if case["setup"] == "volume" else 19e-3
        pts = np.stack([rng.uniform(-half, half, K), rng.uniform(-half, half, K) * (case["ny"] > 1), depth], 1)
    move = np.stack([np.zeros(F), np.zeros(F), 0.1e-3 * np.arange(F)], 1)
    x = synth.echoes(a["probe"], a["waves"], pts, rng.standard_normal(K), fs=a["fs"], n_samples=case["L"], f0=a["f0"],
                     bandwidth=synth.pulse_bandwidth_for_cycles(2.5), iq=not case["rf"], n_frames=F, frame_offsets=move)
    x = torch.from_numpy(x).to("cuda")
    g = torch.Generator("cuda").manual_seed(int(seed))
    return x + 0.02 * torch.randn(x.shape, dtype=x.dtype, device=x.device, generator=g)


def _analytic(rf):
    """The analytic signal in FP64 (MATLAB's hilbert), one trace per row."""
    L = rf.shape[-1]
    h = torch.zeros(L, dtype=torch.float64, device=rf.device)
    h[0] = 1.0
    h[1:(L + 1) // 2] = 2.0
    if L % 2 == 0:
        h[L // 2] = 1.0
    rows = rf.reshape(-1, L)
    out = torch.empty(rows.shape, dtype=torch.complex128, device=rf.device)
    step = max(1, (1 << 24) // L)
    for i in range(0, rows.shape[0], step):
        out[i:i + step] = torch.fft.ifft(torch.fft.fft(rows[i:i + step].to(torch.float64)) * h)
    return out.reshape(rf.shape)


def _members(case):
    """The acquisitions of a batch: one probe and sequence, square grids of three sizes in turn."""
    if case["entry"] != "batch":
        return [case]
    return [dict(case, nx=max(8, case["nx"] >> k), nz=max(8, case["nz"] >> k)) for k in
            (i % 3 for i in range(case["count"]))]


def _front_end_rf(case, seed):
    """RF traces for the front end: band-limited speckle with the attenuation of depth, float32."""
    g = torch.Generator("cuda").manual_seed(int(seed))
    shape = (case["F"], case["W"], case["N"], case["L"])
    x = torch.randn(shape, dtype=torch.float32, device="cuda", generator=g)
    t = torch.arange(case["L"], dtype=torch.float32, device="cuda")
    fade = torch.exp(-1.5 * t / case["L"])
    carrier = torch.cos(2.0 * math.pi * 0.25 * t)
    return ((x + 4.0 * x.roll(1, -1) * carrier) * fade).contiguous()


def _taps(case):
    """20.8 MHz data around 5.2 MHz: the MATLAB flavour's Kaiser filter or the Python flavour's windowed sinc."""
    fs, f0 = 20.8e6, 5.2e6
    if case["zero_phase"]:
        return fs, f0, python_lowpass(case["L"], 0.5 * f0, fs)
    return fs, f0, matlab_lowpass(0.5 * f0, 1.0 * f0, fs)


# ---------------------------------------------------------------------------
# prepare / run
# ---------------------------------------------------------------------------
def prepare(case, seed):
    entry = case["entry"]
    if entry == "hilbert":
        return {"entry": entry, "rf": _front_end_rf(case, seed)}
    if entry == "demodulate":
        fs, f0, b = _taps(case)
        return {"entry": entry, "rf": _front_end_rf(case, seed), "fs": fs, "f0": f0, "b": b, "down": case["down"],
                "mode": int(case["zero_phase"])}
    if entry == "batch":
        plans, chs, kept = [], [], {}
        for i, member in enumerate(_members(case)):
            key = (member["nx"], member["nz"])
            a = _acquisition(member)
            if key not in kept:
                kept[key] = _plan(member, a)
            if i < 4:
                data = _echoes(member, a, seed * 1000 + i)
            chs.append(data if i < 4 else chs[i % 4].clone())
            plans.append(kept[key])
        batch = Batch(plans)
        return {"entry": entry, "batch": batch, "outs": batch.set_io(chs)}
    a = _acquisition(case)
    x = _echoes(case, a, seed)
    if entry == "go":
        das = DAS()
        das.channel_data = ChannelData(probe=a["probe"], sequence=a["waves"], sampling_frequency=a["fs"],
                                       initial_time=0.0, sound_speed=C, modulation_frequency=a["fd"], device_data=x)
        das.scan = a["scan"]
        das.dimension = DIMS[case["dim"]]
        das.interpolation = Interpolation.cubic if case["cubic"] else Interpolation.linear
        das.receive_apodization, das.transmit_apodization = _apodizations(a)
        return {"entry": entry, "das": das}
    ch = _analytic(x).to(torch.complex64) if case["rf"] else x
    if entry == "matrix":
        td, ta, rd, ra = (t.to(torch.float32) for t in _matrices(case, a, slice(None)))
        return {"entry": entry, "ch": ch, "fs": a["fs"], "fd": a["fd"], "dim": int(DIMS[case["dim"]]), "tx_apo": ta,
                "rx_apo": ra, "tx_delay": td, "rx_delay": rd, "interp": int(case["cubic"])}
    return {"entry": entry, "ch": ch, "plan": _plan(case, a)}


def run(state):
    entry = state["entry"]
    if entry == "plan":
        return state["plan"].run(state["ch"])
    if entry == "plan_cf":
        images = state["plan"].run(state["ch"])
        image, cf = ops.coherence_factor(images, int(Dimension.transmit))
        return {"images": images, "image": image, "cf": cf}
    if entry == "go":
        return state["das"].go().data
    if entry == "matrix":
        return ops.das(state["ch"], state["fs"], 0.0, state["tx_apo"], state["rx_apo"], state["tx_delay"],
                       state["rx_delay"], state["fd"], state["dim"], interp=state["interp"])
    if entry == "batch":
        state["batch"].launch()
        return state["outs"]
    if entry == "hilbert":
        return ops.hilbert(state["rf"])
    return ops.demodulate(state["rf"], state["fs"], 0.0, state["f0"], state["b"], state["down"], state["mode"])


# ---------------------------------------------------------------------------
# work
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: the samples, the caller's matrices and the outputs once each (a plan's own tables are the present
    code's choice). Flops: the terms whose weights are not zero, each with its index and fraction once for all
    frames (5 operations; Keys' weights 14 more), and per frame the interpolation and the weighted complex sum (14
    linear, 22 cubic; real weights of RF data 4 fewer); transforms at 5 L log2 L; 4 operations per filter tap and
    output."""
    if case["entry"] == "hilbert":
        n = case["F"] * case["W"] * case["N"]
        return {"bytes": 12 * n * case["L"], "flops": n * 2 * 2.5 * case["L"] * math.log2(case["L"])}
    if case["entry"] == "demodulate":
        n, Lo = case["F"] * case["W"] * case["N"], -(-case["L"] // case["down"])
        taps = len(_taps(case)[2])
        taps = 2 * taps - 1 if case["zero_phase"] else taps
        return {"bytes": n * (4 * case["L"] + 8 * Lo), "flops": n * (6 * case["L"] + 4 * taps * Lo)}
    total = {"bytes": 0, "flops": 0}
    for member in _members(case):
        a = _acquisition(member)
        P = member["nx"] * member["ny"] * member["nz"]
        some = slice(None, None, max(1, P // 4000))
        _, ta, _, ra = _matrices(member, a, some, "cpu")
        terms = float(((ta != 0).sum(0) * (ra != 0).sum(0)).double().mean()) * P
        per = (22 if member["cubic"] else 14) - (4 if member["rf"] else 0)
        samples = member["F"] * member["W"] * member["N"] * member["L"]
        out = _out_values(dict(member, count=1))
        total["flops"] += terms * ((19 if member["cubic"] else 5) + per * member["F"])
        total["bytes"] += 8 * samples + 8 * out
        if member["entry"] == "go" and member["rf"]:
            total["bytes"] -= 4 * samples
        if member["entry"] == "matrix":
            total["bytes"] += 8 * (member["W"] + member["N"]) * P
        if member["entry"] == "plan_cf":
            total["flops"] += 6 * out
            total["bytes"] += 12 * member["F"] * P
    return total


# ---------------------------------------------------------------------------
# exact: the definitions in 64 bits
# ---------------------------------------------------------------------------
def _tukey25(r):
    roll = 0.25
    th = 0.5 * (1.0 - roll)
    taper = 0.5 * (1.0 + torch.cos((2.0 * math.pi / roll) * (r - roll / 2.0 - 0.5)))
    return torch.where(r <= th, torch.ones_like(r), torch.where(r < 0.5, taper, torch.zeros_like(r)))


def _pixels(case, a, pick, device):
    """x, y, z and the depth coordinate of the scan's pixels (depth fastest, then x or azimuth, then y)."""
    first, second, depth = (torch.as_tensor(v, dtype=torch.float64, device=device) for v in a["axes"])
    s, q, z = torch.meshgrid(second, first, depth, indexing="ij")
    z, q, s = z.reshape(-1)[pick], q.reshape(-1)[pick], s.reshape(-1)[pick]
    if case["setup"] == "phased":
        return z * torch.sin(q), torch.zeros_like(z), z * torch.cos(q), z
    return q, s, z, z


def _single(t):
    return t.to(torch.float32).to(torch.float64)


def _matrices(case, a, pick, device="cuda"):
    """Transmit and receive delays and weights ([W, P], [N, P]) rounded to single, in FP64: das.m's matrices."""
    x, y, z, depth = _pixels(case, a, pick, device)
    ex, ey = (torch.as_tensor(v, dtype=torch.float64, device=device)[:, None] for v in (a["probe"].x, a["probe"].y))
    N, W, P = ex.shape[0], case["W"], x.numel()
    rd = torch.sqrt((ex - x) ** 2 + (ey - y) ** 2 + z ** 2) / C
    ra = torch.ones((N, P), dtype=torch.float64, device=device)
    if a["rx"]:
        # linear scans centre the aperture on the pixel, sector scans on the probe's centre
        dx, dy = (ex.expand(N, P), ey.expand(N, P)) if case["setup"] == "phased" else (x - ex, y - ey)
        reach = torch.clamp(depth, min=1e-3 * F_NUMBER)
        ra = _tukey25(torch.abs(F_NUMBER * (dx / reach))) * _tukey25(torch.abs(F_NUMBER * (dy / reach)))
    td = torch.empty((W, P), dtype=torch.float64, device=device)
    ta = torch.ones((W, P), dtype=torch.float64, device=device)
    for w in range(W):
        if a["sources"] is None:
            t = float(a["angles"][w])
            td[w] = (z * math.cos(t) + x * math.sin(t)) / C
            if a["tx"]:
                ta[w] = _tukey25(torch.full((), abs(F_NUMBER * math.tan(t)), dtype=torch.float64))
        else:
            sx, sy, sz = a["sources"][w]
            r0 = math.sqrt(sx * sx + sy * sy + sz * sz)
            td[w] = (torch.sqrt((sx - x) ** 2 + (sy - y) ** 2 + (sz - z) ** 2) - r0) / C
    return _single(td), _single(ta), _single(rd), _single(ra)


def _exact_das(case, a, ch):
    """sum over the case's dimension of ta * ra * exp(i wd (td + rd)) * x((td + rd) fs), das_c's window 1 <= d < L - 1
    (cubic: L - 2); ch complex128 (F, W, N, L)."""
    F, W, N, L = ch.shape
    P = case["nx"] * case["ny"] * case["nz"]
    dim = case["dim"]
    out = torch.zeros((F, W if dim in ("none", "receive") else 1, N if dim in ("none", "transmit") else 1, P),
                      dtype=torch.complex128, device=ch.device)
    wd = float(np.float32(2.0) * np.float32(math.pi) * np.float32(a["fd"]))
    step = max(1, (1 << 23) // W)
    for p0 in range(0, P, step):
        pick = slice(p0, min(P, p0 + step))
        td, ta, rd, ra = _matrices(case, a, pick, ch.device)
        for n in range(N):
            if not bool((ra[n] != 0).any()):
                continue
            delay = td + rd[n]
            d = delay * a["fs"]
            on = (d >= 1.0) & (d < L - (2 if case["cubic"] else 1)) & (ta != 0) & (ra[n] != 0)
            d = torch.where(on, d, torch.ones_like(d))
            i = torch.floor(d)
            b, i = d - i, i.to(torch.int64)
            weight = torch.where(on, ta * ra[n], torch.zeros_like(d))
            weight = torch.polar(weight, wd * delay) if wd else weight
            for f in range(F):
                x = ch[f, :, n, :]
                if case["cubic"]:
                    v = (x.gather(1, i - 1) * (-0.5 * b ** 3 + b ** 2 - 0.5 * b)
                         + x.gather(1, i) * (1.5 * b ** 3 - 2.5 * b ** 2 + 1.0)
                         + x.gather(1, i + 1) * (-1.5 * b ** 3 + 2.0 * b ** 2 + 0.5 * b)
                         + x.gather(1, i + 2) * (0.5 * b ** 3 - 0.5 * b ** 2))
                else:
                    v = x.gather(1, i) * (1.0 - b) + x.gather(1, i + 1) * b
                v = v * weight
                if dim == "none":
                    out[f, :, n, pick] = v
                elif dim == "receive":
                    out[f, :, 0, pick] += v
                else:
                    out[f, 0, n if dim == "transmit" else 0, pick] += v.sum(0)
    return out


def _exact_demodulate(case, rf):
    fs, f0, b = _taps(case)
    L, down = case["L"], case["down"]
    x = rf.reshape(-1, L).to(torch.float64)
    mixed = x * torch.polar(torch.ones(L, dtype=torch.float64, device=x.device),
                            -2.0 * math.pi * f0 / fs * torch.arange(L, dtype=torch.float64, device=x.device))
    b = torch.as_tensor(np.asarray(b), dtype=torch.float64, device=x.device)
    K = b.numel()

    def causal(v):
        n = v.shape[-1] + K - 1
        return torch.fft.ifft(torch.fft.fft(v, n) * torch.fft.fft(b, n))[:, :v.shape[-1]]

    def zero_phase(v):
        # filtfilt: odd extension by 3 K, the filter forward and backward from the state of a constant first sample
        pad = 3 * K
        v = torch.cat([2 * v[:, :1] - v[:, 1:pad + 1].flip(-1), v, 2 * v[:, -1:] - v[:, -pad - 1:-1].flip(-1)], -1)
        for _ in range(2):
            v = causal(torch.cat([v[:, :1].expand(-1, K - 1), v], -1))[:, K - 1:].flip(-1)
        return v[:, pad:-pad]

    out = torch.empty((x.shape[0], -(-L // down)), dtype=torch.complex128, device=x.device)
    for i in range(0, x.shape[0], 2048):
        out[i:i + 2048] = (zero_phase if case["zero_phase"] else causal)(mixed[i:i + 2048])[:, ::down]
    return out.reshape(rf.shape[:-1] + (-1,))


def exact(case, seed):
    if case["entry"] == "hilbert":
        return _analytic(_front_end_rf(case, seed))
    if case["entry"] == "demodulate":
        return _exact_demodulate(case, _front_end_rf(case, seed))
    if case["entry"] == "batch":
        members, kept = _members(case), []
        outs = []
        for i, member in enumerate(members):
            a = _acquisition(member)
            if i < 4:
                kept.append(_echoes(member, a, seed * 1000 + i).to(torch.complex128))
            outs.append(_exact_das(member, a, kept[i % 4]))
        return outs
    a = _acquisition(case)
    x = _echoes(case, a, seed)
    if not case["rf"]:
        ch = x.to(torch.complex128)
    elif case["entry"] == "go":
        ch = _analytic(x)
    else:
        ch = _analytic(x).to(torch.complex64).to(torch.complex128)
    out = _exact_das(case, a, ch)
    if case["entry"] == "go":
        if not case["rf"]:
            # the reference phase of IQ images
            w0 = float(np.float32(2.0) * np.float32(math.pi) * np.float32(a["fd"]))
            r = _pixels(case, a, slice(None), out.device)[3]
            out = out * torch.polar(torch.ones_like(r), -2.0 * w0 / C * r)
        return out.permute(3, 2, 1, 0)
    if case["entry"] == "plan_cf":
        total = out.sum(1, keepdim=True)
        energy = (out.abs() ** 2).sum(1, keepdim=True)
        cf = torch.nan_to_num(total.abs() ** 2 / energy / case["W"])
        return {"images": out, "image": cf * total, "cf": cf}
    return out
