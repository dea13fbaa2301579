"""Plans whose tiles hold one or two waves (several channels at a time) against
the same plan with four wave slots per split (one channel at a time, the
oracle-checked kernel): channel counts around a step of four, tiles with fewer
waves than slots, partly weighted tiles, more tiles than whole groups, frames,
and terms out of every window."""
from __future__ import annotations

import math

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from ustb_amd import ops
from ustb_amd.batch import Batch
from ustb_amd.enums import Window
from ustb_amd.geometry import make_plan
from ustb_amd.uff import Apodization, LinearArray, LinearScan, SectorScan, Wave

pytestmark = pytest.mark.gpu
C = 1540.0


def _plan(W, N, rf, cubic, F, L, rx, tx=Apodization(), sector=False):
    prb = LinearArray(N, 0.3e-3)
    if sector:
        seq = [Wave.spherical(x, 0.0, -10e-3, sound_speed=C, origin=(x, 0.0, -10e-3)) for x in np.linspace(-4e-3, 4e-3, W)]
        scan = SectorScan(np.deg2rad(np.linspace(-40, 40, 21)), np.linspace(0.0, 25e-3, 31))  # a pixel at the apex
    else:
        seq = [Wave.plane(a, sound_speed=C) for a in (np.deg2rad(np.linspace(-12, 12, W)) if W > 1 else np.zeros(1))]
        scan = LinearScan(np.linspace(-8e-3, 8e-3, 33), np.linspace(2e-3, 25e-3, 70))
    fs, fd = (20.8e6, 0.0) if rf else (10.4e6, 5.2e6)
    return make_plan(prb, scan, seq, n_samples=L, n_frames=F, sampling_frequency=fs, initial_time=0.0,
                     modulation_frequency=fd, sound_speed=C, receive_apodization=rx, transmit_apodization=tx,
                     interpolation=int(cubic), separable_phase=True)


TUKEY = Apodization(Window.tukey25, f_number=1.7)
CASES = [
    # W, N, rf, cubic, F, L, rx, sector
    (1, 33, True, False, 1, 900, TUKEY, False),
    (1, 7, False, False, 2, 500, Apodization(), False),
    (1, 34, False, True, 1, 220, TUKEY, False),       # traces end inside the image
    (2, 35, True, True, 1, 900, TUKEY, False),
    (2, 32, False, False, 3, 220, TUKEY, False),
    (2, 5, False, True, 1, 500, Apodization(), True),
    (1, 21, False, False, 1, 500, TUKEY, True),
    (2, 21, True, False, 1, 900, TUKEY, True),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: "-".join(str(v) for v in c[:6]))
def test_against_one_channel_at_a_time(cuda, case):
    W, N, rf, cubic, F, L, rx, sector = case
    print("case few", case[:6], flush=True)
    plan = _plan(W, N, rf, cubic, F, L, rx, sector=sector)
    rng = np.random.default_rng(N)
    ch = torch.from_numpy((rng.standard_normal((F, W, N, L)) + 1j * rng.standard_normal((F, W, N, L)))
                          .astype(np.complex64)).to(cuda)
    v = plan.variant
    assert tuple(v) == (2, 4, 8)
    got = plan.run(ch).clone()
    # one batch item of the same shape: the same terms in the same order
    b = Batch([plan])
    (out,) = b.set_io([ch])
    b.set_tiles(4, 8)
    b.launch()
    torch.cuda.synchronize()
    assert torch.equal(got.view(torch.float32).nan_to_num(7.0), out.view(torch.float32).nan_to_num(7.0))
    # six wave slots: FP32 regrouping of at most W * N terms at most
    plan.set_tiles(6, 8)
    ref = plan.run(ch)
    fin = torch.isfinite(torch.view_as_real(ref)).all(-1)
    assert torch.equal(fin, torch.isfinite(torch.view_as_real(got)).all(-1))
    peak = float(ref[fin].abs().max())
    assert peak > 0
    assert float((got - ref)[fin].abs().max()) <= 2.0 * W * N * 2.0 ** -24 * peak * 4
    plan.close()


def test_default_shape_follows_the_receive_state(cuda):
    """The kernel that computes the receive state keeps the shapes it was
    measured with, a shape that was set stays."""
    plan = _plan(5, 33, False, False, 1, 500, TUKEY)
    assert plan.variant == (2, 6, 8)
    plan.set_variant(4)
    assert plan.variant == (4, 4, 8)
    assert plan.has_variant(2) and plan.variant == (4, 4, 8)
    plan.set_variant(2)
    assert plan.variant == (2, 6, 8)
    assert plan.has_variant(4) and plan.variant == (2, 6, 8)
    plan.set_tiles(12, 8)
    plan.set_variant(4)
    assert plan.variant == (4, 12, 8)
    plan.close()


def test_a_refused_variant_leaves_the_plan_as_it_was(cuda):
    """The on-the-fly receive state does not take a tilted aperture; asking for it keeps the receive table."""
    plan = _plan(5, 33, False, False, 1, 500, Apodization(Window.tukey25, f_number=1.7, tilt=(0.1, 0.0)))
    ch = torch.randn((1, 5, 33, 500), dtype=torch.complex64, device=cuda)
    v, ref = plan.variant, plan.run(ch)
    assert v[0] == 2 and not plan.has_variant(4)
    assert plan.variant == v
    print("case refused variant", flush=True)
    assert torch.equal(plan.run(ch), ref)
    plan.close()


@pytest.mark.parametrize("kind,W,nx,nz,F,cubic,shape", [
    ("volume", 4, 30, 70, 1, False, (4, 8)),    # 2297 blocks: images of 3 and 4 waves take 4 splits there
    ("linear", 4, 400, 330, 1, False, (4, 4)),  # 2063
    ("sector", 5, 150, 154, 2, True, (5, 8)),   # 722
    ("sector", 9, 150, 164, 1, True, (5, 4)),   # 385
    ("sector", 20, 150, 147, 1, False, (16, 4)),  # 345
    ("sector", 20, 100, 147, 1, False, (16, 8)),  # 230
])
def test_default_shapes(cuda, kind, W, nx, nz, F, cubic, shape):
    """Where a shape for few blocks, few splits or many registers was slower than the one before it."""
    print(f"case default shape {kind} W={W} {nx} x {nz}", flush=True)
    seq = [Wave.spherical(x, 0.0, -10e-3, sound_speed=C, origin=(x, 0.0, -10e-3)) for x in np.linspace(-4e-3, 4e-3, W)]
    x, z = np.linspace(-8e-3, 8e-3, nx), np.linspace(2e-3, 25e-3, nz)
    scan = (SectorScan(np.deg2rad(np.linspace(-40, 40, nx)), z) if kind == "sector" else
            LinearScan(x, z, np.linspace(-8e-3, 8e-3, 70) if kind == "volume" else (0.0,)))
    plan = make_plan(LinearArray(33, 0.3e-3), scan, seq, n_samples=500, n_frames=F, sampling_frequency=10.4e6,
                     initial_time=0.0, modulation_frequency=5.2e6, sound_speed=C, receive_apodization=TUKEY,
                     interpolation=int(cubic), separable_phase=True)
    assert plan.variant == (2, *shape)
    plan.close()


@pytest.mark.parametrize("W,N,F,sector", [(1, 33, 1, False), (2, 21, 2, True)])
def test_coefficient_variant(cuda, W, N, F, sector):
    """Variant 3 (cubic coefficients) with one and two waves against variant 2's shapes of six slots."""
    print("case few coefficients", W, N, F, flush=True)
    plan = _plan(W, N, False, True, F, 500, TUKEY, sector=sector)
    ch = torch.randn((F, W, N, 500), dtype=torch.complex64, device=cuda, generator=torch.Generator(cuda).manual_seed(N))
    plan.set_tiles(6, 8)
    ref = plan.run(ch)
    plan.set_tiles(4, 8)
    plan.set_variant(3)
    assert plan.variant == (3, 4, 8)
    got = plan.run(ch)
    fin = torch.isfinite(torch.view_as_real(ref)).all(-1)
    assert torch.equal(fin, torch.isfinite(torch.view_as_real(got)).all(-1))
    # the same cubic by its polynomial's coefficients (FP32, magnitudes up to 10 samples), W * N terms
    assert float((got - ref)[fin].abs().max()) <= 40 * W * N * 2.0 ** -24 * float(ref[fin].abs().max())
    plan.close()
