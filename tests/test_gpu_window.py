"""Dimension receive and none on patch tiles with staged sample windows: scans
whose axes leave part tiles, every wave count around a step, traces that end
inside the image (terms out of the window), partly weighted tiles and coarse
grids (long rows), against the FP64 beamformer on the plan's own matrices; RF
data against das_c's arithmetic bit for bit."""
from __future__ import annotations

import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from ustb_amd import ops
from ustb_amd.enums import Window
from ustb_amd.geometry import make_plan
from ustb_amd.uff import Apodization, LinearArray, LinearScan, MatrixArray, SectorScan, Wave

pytestmark = pytest.mark.gpu
C = 1540.0


def _setup(kind, W, nx, nz, zmax=25e-3, N=21):
    if kind == "sector":
        prb = LinearArray(N, 0.2e-3)
        ang = np.deg2rad(np.linspace(-30, 30, W)) if W > 1 else np.zeros(1)
        src = [(-10e-3 * math.sin(a), 0.0, -10e-3 * math.cos(a)) for a in ang]
        seq = [Wave.spherical(*s, sound_speed=C, origin=s) for s in src]
        return prb, SectorScan(np.deg2rad(np.linspace(-40, 40, nx)), np.linspace(2e-3, zmax, nz)), seq
    if kind == "volume":
        seq = [Wave.spherical(x, 0.0, -8e-3, sound_speed=C, origin=(x, 0.0, -8e-3)) for x in np.linspace(-2e-3, 2e-3, W)]
        return (MatrixArray(5, 4, 0.3e-3), LinearScan(np.linspace(-3e-3, 3e-3, nx), np.linspace(4e-3, zmax, nz),
                                                       np.linspace(-2e-3, 2e-3, 7)), seq)
    seq = [Wave.plane(a, sound_speed=C) for a in (np.deg2rad(np.linspace(-16, 16, W)) if W > 1 else np.zeros(1))]
    return LinearArray(N, 0.3e-3), LinearScan(np.linspace(-8e-3, 8e-3, nx), np.linspace(4e-3, zmax, nz)), seq


def _run(cuda, kind, dim, W, nx, nz, F, rf, cubic, phase, L, rx, zmax=25e-3, tx=Apodization()):
    prb, scan, seq = _setup(kind, W, nx, nz, zmax)
    fs, fd = (20.8e6, 0.0) if rf else (10.4e6, 5.2e6)
    plan = make_plan(prb, scan, seq, n_samples=L, n_frames=F, sampling_frequency=fs, initial_time=0.0,
                     modulation_frequency=fd, sound_speed=C, receive_apodization=rx, transmit_apodization=tx,
                     dimension=dim, interpolation=int(cubic), separable_phase=phase == "separable")
    rng = np.random.default_rng(W * 100 + nz)
    ch = (rng.standard_normal((F, W, prb.N_elements, L)) +
          1j * rng.standard_normal((F, W, prb.N_elements, L))).astype(np.complex64)
    dch = torch.from_numpy(ch).to(cuda)
    got = plan.run(dch)
    ta, ra, td, rd = plan.materialize()
    plan.close()
    return got, dch, (ta, ra, td, rd), fs, fd


TUKEY = Apodization(Window.tukey25, f_number=1.7)
BOX = Apodization(Window.boxcar, f_number=2.5)
CASES = [
    # kind, W, nx, nz, F, cubic, phase, L, rx, zmax
    ("linear", 1, 37, 61, 1, False, "separable", 512, TUKEY, 25e-3),
    ("linear", 4, 16, 16, 1, False, "separable", 512, Apodization(), 25e-3),
    ("linear", 5, 33, 65, 2, False, "dasc", 512, BOX, 25e-3),
    ("linear", 8, 17, 130, 1, True, "separable", 300, TUKEY, 25e-3),   # traces end inside the image
    ("linear", 9, 40, 31, 3, True, "dasc", 260, BOX, 25e-3),
    ("linear", 3, 35, 24, 2, False, "separable", 512, TUKEY, 40e-3),   # coarse depths: rows of 128 samples
    ("sector", 7, 29, 50, 1, False, "dasc", 512, BOX, 25e-3),
    ("sector", 13, 18, 33, 5, False, "separable", 310, TUKEY, 25e-3),
    ("volume", 5, 9, 35, 1, False, "separable", 400, Apodization(Window.tukey25, f_number=(1.2, 1.2)), 12e-3),
    ("volume", 2, 6, 18, 2, True, "dasc", 400, Apodization(), 12e-3),
]


@pytest.mark.parametrize("dim", [0, 1])
@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c[:7]))
def test_iq_against_fp64(cuda, case, dim):
    kind, W, nx, nz, F, cubic, phase, L, rx, zmax = case
    print(f"case window {case[:8]} dim={dim}", flush=True)
    got, ch, (ta, ra, td, rd), fs, fd = _run(cuda, kind, dim, W, nx, nz, F, False, cubic, phase, L, rx, zmax)
    ref = O.beamform_fp64(ch.cpu().numpy(), fs, 0.0, ta.cpu().numpy(), ra.cpu().numpy(), td.cpu().numpy(),
                          rd.cpu().numpy(), fd, dim, interp="cubic" if cubic else "linear", w0=O.dasc_wd(fd),
                          index="fp32")
    # FP32 products and sums of at most 21 terms and the FP32 phase argument
    # of das_c (wd * delay up to 1700 rad at 6e-8 relative: 1e-4 per term)
    tol = 2e-4 if phase == "dasc" else 1e-5
    assert np.max(np.abs(got.cpu().numpy() - ref)) <= tol * np.max(np.abs(ref))


@pytest.mark.parametrize("dim", [0, 1])
@pytest.mark.parametrize("kind,W,nx,nz,F,L", [("linear", 1, 37, 61, 1, 900), ("linear", 6, 20, 45, 1, 500),
                                               ("sector", 5, 31, 33, 3, 500), ("volume", 3, 9, 20, 2, 500)])
def test_rf_is_das_c(cuda, kind, W, nx, nz, F, L, dim):
    print(f"case window rf {kind} W={W} dim={dim}", flush=True)
    got, ch, (ta, ra, td, rd), fs, fd = _run(cuda, kind, dim, W, nx, nz, F, True, False, "separable", L, BOX, 12e-3)
    ref = ops.das(ch, fs, 0.0, ta, ra, td, rd, fd, dim, dasc_order=True)
    assert torch.equal(got, ref)


@pytest.mark.parametrize("dim", [0, 1])
def test_samples_outside_the_weights_stay_out(cuda, dim):
    """Non-finite samples reach no term that das_c skips (zero receive weight)."""
    prb, scan, seq = _setup("linear", 3, 40, 64)
    plan = make_plan(prb, scan, seq, n_samples=512, n_frames=1, sampling_frequency=10.4e6, initial_time=0.0,
                     modulation_frequency=5.2e6, sound_speed=C, receive_apodization=BOX, transmit_apodization=Apodization(),
                     dimension=dim, interpolation=0)
    rng = np.random.default_rng(3)
    ch = (rng.standard_normal((1, 3, 21, 512)) + 1j * rng.standard_normal((1, 3, 21, 512))).astype(np.complex64)
    ch[0, :, 4, 100:140] = np.nan
    got = plan.run(torch.from_numpy(ch).to(cuda)).cpu().numpy()
    ta, ra, td, rd = (t.cpu().numpy() for t in plan.materialize())
    plan.close()
    ref = O.beamform_fp64(ch, 10.4e6, 0.0, ta, ra, td, rd, 5.2e6, dim, w0=O.dasc_wd(5.2e6), index="fp32")
    assert np.array_equal(np.isnan(got), np.isnan(ref)) and np.isnan(ref).any()


BOTH = [
    # kind, W, nx, nz, F, rf, cubic, L: work of at least 640, 512 or 400 of the
    # largest tiles (x 2 frames), with tiles of half of it
    ("linear", 9, 540, 900, 1, False, False, 512),
    ("linear", 13, 251, 333, 7, True, False, 500),    # traces end inside the image
    ("linear", 33, 401, 700, 1, False, False, 420),
    ("sector", 17, 401, 401, 5, False, True, 512),
    ("volume", 26, 110, 170, 3, False, False, 400),
]


@pytest.mark.parametrize("rx", [TUKEY, BOX], ids=["tukey", "boxcar"])
@pytest.mark.parametrize("kind,W,nx,nz,F,rf,cubic,L", BOTH)
def test_both_against_set_tiles(cuda, kind, W, nx, nz, F, rf, cubic, L, rx):
    """Dimension both on the library's choice (staged windows) against the
    gathering kernel of a set tile shape, with non-finite samples that only
    zero weights meet somewhere; both sum the same FP32 terms in another order."""
    print(f"case window both {kind} W={W} F={F} cubic={cubic}", flush=True)
    prb, scan, seq = _setup(kind, W, nx, nz, 25e-3 if kind != "volume" else 14e-3)
    fs, fd = (20.8e6, 0.0) if rf else (10.4e6, 5.2e6)
    # plane waves: one weight per wave; sector: tiles partly outside the waves' cones
    tx = {"linear": Apodization(Window.tukey25, f_number=1.5), "sector": Apodization(Window.boxcar, f_number=0.7),
          "volume": Apodization()}[kind]
    plan = make_plan(prb, scan, seq, n_samples=L, n_frames=F, sampling_frequency=fs, initial_time=0.0,
                     modulation_frequency=fd, sound_speed=C, receive_apodization=rx, transmit_apodization=tx,
                     dimension=3, interpolation=int(cubic), reference_phase=not rf)
    assert plan.variant == (2, 0, 0)
    g = torch.Generator(cuda).manual_seed(W)
    ch = torch.randn((F, W, prb.N_elements, L), dtype=torch.complex64, device=cuda, generator=g)
    ch[0, :, 2, 60:70] = float("nan")
    got = plan.run(ch)
    plan.set_tiles(8, 4)
    assert plan.variant == (2, 8, 4)
    ref = plan.run(ch)
    plan.close()
    a, b = torch.view_as_real(got), torch.view_as_real(ref)
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    # sums of at most 33 x 21 FP32 terms in another order: sqrt(700) * 6e-8 of
    # the RMS sum, ten times that of the peak
    assert (torch.nan_to_num(a - b).abs().max() / torch.nan_to_num(b).abs().max()).item() <= 5e-6


def test_both_keeps_small_plans_on_the_gathering_kernel(cuda):
    prb, scan, seq = _setup("linear", 4, 300, 500)
    kw = dict(n_samples=512, n_frames=1, sampling_frequency=10.4e6, initial_time=0.0, modulation_frequency=5.2e6,
              sound_speed=C, receive_apodization=TUKEY, dimension=3)
    few_waves = make_plan(prb, scan, seq, **kw)
    prb, scan, seq = _setup("linear", 12, 40, 64)
    few_tiles = make_plan(prb, scan, seq, **kw)
    assert few_waves.variant[1:] != (0, 0) and few_tiles.variant[1:] != (0, 0)
    few_waves.close()
    few_tiles.close()


def test_both_sums_are_closed_over_many_channels(cuda):
    """Constant data: every term is the same number, so one running sum over
    the 576 channels drifts (7.4e-6 of the sum at this value). Each of the 6
    waves of a group, the 32 channels of a block, the 18 blocks and the two
    groups add at most half an ulp: 58 * 2^-24 = 3.5e-6."""
    print("case window both constant data", flush=True)
    W, F, L = 12, 2, 700
    prb = MatrixArray(24, 24, 0.3e-3)
    seq = [Wave.spherical(x, 0.0, -8e-3, sound_speed=C, origin=(x, 0.0, -8e-3)) for x in np.linspace(-2e-3, 2e-3, W)]
    scan = LinearScan(np.linspace(-3e-3, 3e-3, 64), np.linspace(4e-3, 12e-3, 48), np.linspace(-2e-3, 2e-3, 64))
    plan = make_plan(prb, scan, seq, n_samples=L, n_frames=F, sampling_frequency=20.8e6, initial_time=0.0,
                     modulation_frequency=0.0, sound_speed=C, receive_apodization=Apodization(),
                     transmit_apodization=Apodization(), dimension=3, interpolation=0)
    assert plan.variant == (2, 0, 0)
    c = float(np.float32(1.8018805787183079))
    got = torch.view_as_real(plan.run(torch.full((F, W, prb.N_elements, L), complex(c, c), dtype=torch.complex64,
                                                 device=cuda))).double()
    plan.close()
    assert (got / (prb.N_elements * W * c) - 1.0).abs().max().item() <= 58 * 2.0 ** -24


def test_more_frames_than_one_grid(cuda):
    """A grid holds fewer than 2^32 threads: 8200 frames of 528 x 1040 pixels, 36
    GB of image, against plans of the first and last frames."""
    print("case window both 8200 frames", flush=True)
    W, F, L, Q = 9, 8200, 64, 3
    prb = LinearArray(4, 0.3e-3)
    seq = [Wave.plane(a, sound_speed=C) for a in np.deg2rad(np.linspace(-8, 8, W))]
    scan = LinearScan(np.linspace(-2e-3, 2e-3, 528), np.linspace(1e-3, 4e-3, 1040))
    kw = dict(n_samples=L, sampling_frequency=10.4e6, initial_time=0.0, modulation_frequency=5.2e6, sound_speed=C,
              receive_apodization=Apodization(), transmit_apodization=Apodization(), dimension=3, interpolation=0)
    g = torch.Generator(cuda).manual_seed(8)
    ch = torch.randn((F, W, prb.N_elements, L), dtype=torch.complex64, device=cuda, generator=g)
    plan = make_plan(prb, scan, seq, n_frames=F, **kw)
    few = make_plan(prb, scan, seq, n_frames=Q, **kw)
    assert plan.variant == few.variant == (2, 0, 0)
    got = plan.run(ch)
    for f in (0, 4000, F - Q):
        assert torch.equal(got[f:f + Q], few.run(ch[f:f + Q].contiguous())), f
    plan.close()
    few.close()


@pytest.mark.parametrize("kind,W,nx,nz,F,dim,phase,shape", [
    ("linear", 9, 540, 900, 1, 3, "separable", (2, 8, 4)), ("volume", 26, 110, 170, 3, 3, "separable", (2, 16, 4)),
    ("sector", 6, 31, 70, 2, 1, "separable", (0, 16, 1)), ("linear", 5, 33, 65, 1, 0, "separable", (0, 8, 1)),
    ("linear", 5, 33, 65, 1, 1, "dasc", (0, 8, 1))])
def test_tile_shapes_select_and_restore(cuda, kind, W, nx, nz, F, dim, phase, shape):
    """A set tile shape runs and is reported; the reported one restores the staged windows."""
    print(f"case window shapes {kind} W={W} dim={dim} {phase}", flush=True)
    prb, scan, seq = _setup(kind, W, nx, nz, 25e-3 if kind != "volume" else 14e-3)
    plan = make_plan(prb, scan, seq, n_samples=512, n_frames=F, sampling_frequency=10.4e6, initial_time=0.0,
                     modulation_frequency=5.2e6, sound_speed=C, receive_apodization=TUKEY,
                     transmit_apodization=Apodization(), dimension=dim, interpolation=0,
                     separable_phase=phase == "separable")
    g = torch.Generator(cuda).manual_seed(W)
    ch = torch.randn((F, W, prb.N_elements, 512), dtype=torch.complex64, device=cuda, generator=g)
    v = plan.variant
    assert v == (shape[0], 0, 0)
    staged = plan.run(ch)
    plan.set_tiles(*shape[1:])
    assert plan.variant == shape and plan.has_variant(0) and plan.variant == shape
    own = plan.run(ch)
    # the same FP32 terms in another order (das_c's phase: the same order)
    assert (own - staged).abs().max().item() <= (0.0 if phase == "dasc" else 5e-6) * staged.abs().max().item()
    plan.set_tiles(0, shape[2])
    assert plan.variant == shape
    plan.set_tiles(*v[1:])
    assert plan.variant == v and torch.equal(plan.run(ch), staged)
    if dim == 3:
        plan.set_variant(0)
        plan.set_variant(2)
        assert plan.variant == v and torch.equal(plan.run(ch), staged)
    plan.close()


def test_receive_table_is_bounded(cuda):
    """A receive plan whose table would take more than a 32nd of the device memory keeps none."""
    total = torch.cuda.get_device_properties(cuda).total_memory
    N = 128
    nx = int(math.sqrt(total / 32 / 16 / N) * 1.02)
    print(f"case window table bound {nx} x {nx}", flush=True)
    seq = [Wave.plane(0.0, sound_speed=C)]
    kw = dict(n_samples=256, n_frames=1, sampling_frequency=10.4e6, initial_time=0.0, modulation_frequency=5.2e6,
              sound_speed=C, receive_apodization=TUKEY, dimension=1, interpolation=0)
    scans = [LinearScan(np.linspace(-8e-3, 8e-3, n), np.linspace(4e-3, 15e-3, nx)) for n in (nx, 64)]
    large, small = (make_plan(LinearArray(N, 0.3e-3), s, seq, **kw) for s in scans)
    assert small.variant == (0, 0, 0) and large.variant[1:] != (0, 0) and large.device_bytes < total // 64
    ch = torch.randn((1, 1, N, 256), dtype=torch.complex64, device=cuda)
    assert torch.isfinite(torch.view_as_real(large.run(ch))).all()
    large.close()
    small.close()


@pytest.mark.parametrize("N,nx,nz", [(12, 70, 90), (64, 300, 420)], ids=["one launch", "shape by shape"])
@pytest.mark.parametrize("dim", [0, 1])
def test_lists_of_wide_windows(cuda, N, nx, nz, dim):
    """Coarse depths, where the first tile shape does not fit a short row: the
    lists of all shapes from one launch (tables up to 96 MB) or shape by shape,
    against the per-lane kernel."""
    print(f"case window lists N={N} {nx} x {nz} dim={dim}", flush=True)
    zmax, W = 4e-3 + nz * 0.75e-3, 3
    L = int(2 * zmax / C * 10.4e6) + 200
    prb, _, seq = _setup("linear", W, nx, nz, zmax, N)
    scan = LinearScan(np.linspace(-8e-3, 8e-3, nx), np.linspace(4e-3, zmax, nz))
    plan = make_plan(prb, scan, seq, n_samples=L, n_frames=1, sampling_frequency=10.4e6, initial_time=0.0,
                     modulation_frequency=5.2e6, sound_speed=C, receive_apodization=TUKEY,
                     transmit_apodization=Apodization(), dimension=dim, interpolation=0)
    assert plan.variant == (0, 0, 0)
    g = torch.Generator(cuda).manual_seed(N)
    ch = torch.randn((1, W, N, L), dtype=torch.complex64, device=cuda, generator=g)
    got = plan.run(ch)
    plan.set_tiles(8, 1)
    ref = plan.run(ch)
    plan.close()
    # the same FP32 terms, products and (receive) sums of 64 in another order
    assert (got - ref).abs().max().item() <= 5e-6 * ref.abs().max().item()


SHAPES = [
    # W, N, nx, nz, zmax, F, rf, cubic: the groups of 6, 8, 13 and 16 waves, more
    # than 64 channels (no whole number of 32), rows of 128 samples (depths of
    # 0.4 mm at 20.8 MHz, 0.8 mm at 10.4) for every data type
    (9, 65, 640, 560, 25e-3, 1, False, False),
    (15, 70, 420, 470, 25e-3, 1, False, False),
    (26, 67, 360, 400, 25e-3, 1, True, False),
    (31, 65, 360, 400, 25e-3, 1, False, False),
    (16, 66, 200, 300, 25e-3, 5, False, False),
    (11, 20, 1100, 256, 106e-3, 1, True, False),
    (14, 20, 1100, 256, 208e-3, 1, False, False),
    (26, 20, 1000, 256, 106e-3, 1, True, False),
    (30, 20, 1000, 256, 208e-3, 1, False, False),
    (12, 20, 600, 256, 106e-3, 4, True, False),
    (15, 20, 600, 256, 208e-3, 3, False, False),
    (11, 20, 600, 256, 106e-3, 3, True, True),
    (15, 20, 600, 256, 208e-3, 4, False, True),
]


@pytest.mark.parametrize("W,N,nx,nz,zmax,F,rf,cubic", SHAPES)
def test_both_every_shape(cuda, W, N, nx, nz, zmax, F, rf, cubic):
    """Every shape that the dispatch of dimension both picks, against the gathering kernel."""
    print(f"case window both shape W={W} N={N} {nx} x {nz} F={F} rf={rf} cubic={cubic}", flush=True)
    fs, fd = (20.8e6, 0.0) if rf else (10.4e6, 5.2e6)
    L = int(2.1 * zmax / C * fs)
    prb, _, seq = _setup("linear", W, nx, nz, zmax, N)
    scan = LinearScan(np.linspace(-8e-3, 8e-3, nx), np.linspace(4e-3, zmax, nz))
    plan = make_plan(prb, scan, seq, n_samples=L, n_frames=F, sampling_frequency=fs, initial_time=0.0,
                     modulation_frequency=fd, sound_speed=C, receive_apodization=Apodization(),
                     transmit_apodization=Apodization(), dimension=3, interpolation=int(cubic), reference_phase=not rf)
    assert plan.variant == (2, 0, 0)
    g = torch.Generator(cuda).manual_seed(W)
    ch = torch.randn((F, W, N, L), dtype=torch.complex64, device=cuda, generator=g)
    ch[0, :, 2, 60:70] = float("nan")
    got = plan.run(ch)
    plan.set_tiles(8, 4)
    ref = plan.run(ch)
    plan.close()
    a, b = torch.view_as_real(got), torch.view_as_real(ref)
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    # as test_both_against_set_tiles: sums of at most 31 x 65 terms
    assert (torch.nan_to_num(a - b).abs().max() / torch.nan_to_num(b).abs().max()).item() <= 5e-6


@pytest.mark.parametrize("dim", [0, 1])
@pytest.mark.parametrize("kind,W,nx,nz,F,cubic", [("linear", 5, 33, 65, 2, False), ("sector", 9, 29, 50, 1, False),
                                                  ("volume", 3, 9, 20, 1, False), ("linear", 1, 37, 61, 1, False)])
def test_iq_in_das_c_order_is_das_c(cuda, kind, W, nx, nz, F, cubic, dim):
    """das_c's phase: every term as das_c forms it, the channels in its order."""
    print(f"case window das_c {kind} W={W} dim={dim}", flush=True)
    prb, scan, seq = _setup(kind, W, nx, nz, 12e-3)
    plan = make_plan(prb, scan, seq, n_samples=400, n_frames=F, sampling_frequency=10.4e6, initial_time=0.0,
                     modulation_frequency=5.2e6, sound_speed=C, receive_apodization=BOX,
                     transmit_apodization=Apodization(), dimension=dim, interpolation=int(cubic), separable_phase=False)
    assert plan.variant == (0, 0, 0)
    g = torch.Generator(cuda).manual_seed(W)
    ch = torch.randn((F, W, prb.N_elements, 400), dtype=torch.complex64, device=cuda, generator=g)
    ta, ra, td, rd = plan.materialize()
    assert torch.equal(plan.run(ch), ops.das(ch, 10.4e6, 0.0, ta, ra, td, rd, 5.2e6, dim, dasc_order=True))
    plan.close()
