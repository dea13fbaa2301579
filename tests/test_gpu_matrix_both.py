"""Dimension both of the matrix contract in the library's own summation order,
at the wave counts, frame counts and pixel counts where its blocks change,
against das_c's order (split 1) on the same matrices."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from tests.cases import matrix_problem
from ustb_amd import ops

pytestmark = pytest.mark.gpu


def _images(cuda, q, fd, **kw):
    t = {k: torch.from_numpy(q[k]).to(cuda) for k in ("ch", "tx_apo", "rx_apo", "tx_delay", "rx_delay")}
    args = (t["ch"], q["fs"], q["t0"], t["tx_apo"], t["rx_apo"], t["tx_delay"], t["rx_delay"], fd, 3)
    return ops.das(*args, **kw), ops.das(*args, dasc_order=True, **kw)


def _close(got, ref, terms):
    a, b = torch.view_as_real(got), torch.view_as_real(ref)
    assert torch.equal(torch.isnan(a), torch.isnan(b))
    err = torch.nan_to_num(a - b).abs().max() / torch.nan_to_num(b).abs().max()
    # the same terms (FP32, the same rounded phase) added in another order
    assert err.item() <= 6e-8 * (4 + terms ** 0.5)


@pytest.mark.parametrize("fd", [0.0, 0.11, -3.7])
@pytest.mark.parametrize("P,N,W,F", [(63, 5, 2, 1), (64, 1, 3, 4), (65, 7, 8, 5), (1, 3, 9, 1), (130, 12, 33, 1),
                                     (200, 9, 70, 6)])
@pytest.mark.parametrize("interp,edge", [(0, 0), (0, 1), (1, 0)])
def test_against_dasc_order(cuda, P, N, W, F, fd, interp, edge):
    print(f"case matrix both P={P} N={N} W={W} F={F} fd={fd} interp={interp} edge={edge}", flush=True)
    q = matrix_problem(seed=P + W, P=P, N=N, W=W, F=F)
    got, ref = _images(cuda, q, fd, interp=interp, edge=edge)
    _close(got, ref, N * W)


def test_physical_delays(cuda):
    """Phases of thousands of radians, an initial time, unlisted waves."""
    rng = np.random.default_rng(9)
    P, N, W, L = 300, 11, 12, 900
    q = dict(ch=(rng.standard_normal((2, W, N, L)) + 1j * rng.standard_normal((2, W, N, L))).astype(np.complex64),
             fs=20.8e6, t0=3.1e-6, tx_apo=rng.uniform(0.1, 1.0, (W, P)).astype(np.float32),
             rx_apo=rng.uniform(-0.5, 1.0, (N, P)).astype(np.float32),
             tx_delay=rng.uniform(-1e-6, 2.4e-5, (W, P)).astype(np.float32),
             rx_delay=rng.uniform(2e-6, 2.4e-5, (N, P)).astype(np.float32))
    q["tx_apo"][3:7] = 0.0
    q["tx_apo"][8, :128] = 0.0
    for fd in (5.2e6, 2.0e7):
        _close(*_images(cuda, q, fd), N * W)


def test_non_finite_weights_delays_and_samples(cuda):
    """What das_c skips stays out of the sums, what it multiplies reaches them."""
    q = matrix_problem(seed=5, P=200, N=9, W=6, F=2, L=80)
    q["rx_apo"][2, 30:90] = np.nan
    q["tx_apo"][1, 80:100] = np.nan
    q["rx_delay"][4, 10:20] = np.nan
    q["tx_delay"][0, 150:160] = np.inf
    q["ch"][0, 3, 5, 20:24] = np.nan
    q["ch"][1, 2, 1, 40] = np.inf
    got, ref = _images(cuda, q, 0.13)
    assert torch.equal(torch.isfinite(torch.view_as_real(got)), torch.isfinite(torch.view_as_real(ref)))
    fine = torch.isfinite(ref.real) & torch.isfinite(ref.imag)
    assert fine.any() and not fine.all()
    assert (got[fine] - ref[fine]).abs().max() <= 1e-6 * ref[fine].abs().max()


@pytest.mark.parametrize("interp,F", [(0, 1), (0, 3), (1, 1)])
@pytest.mark.parametrize("t0", [0.9e-3, 3.2e-3, 3.2e-2])
def test_large_phases(cuda, t0, interp, F):
    """Delays of any size: around 3e4, 1e5 and 1e6 rad, the first on both sides of where the rotation changes form."""
    print(f"case matrix both phases t0={t0} interp={interp} F={F}", flush=True)
    rng = np.random.default_rng(11)
    P, N, W, L, fd = 300, 9, 11, 400, 5.2e6
    q = dict(ch=(rng.standard_normal((F, W, N, L)) + 1j * rng.standard_normal((F, W, N, L))).astype(np.complex64),
             fs=2.6e6, t0=t0, tx_apo=rng.uniform(0.1, 1.0, (W, P)).astype(np.float32),
             rx_apo=rng.uniform(0.1, 1.0, (N, P)).astype(np.float32),
             tx_delay=(0.4 * t0 + np.linspace(0.0, 1.4e-4, P) * rng.uniform(0.5, 1.0, (W, 1))).astype(np.float32),
             rx_delay=(0.6 * t0 + rng.uniform(0.0, 1e-5, (N, P))).astype(np.float32))
    if t0 == 0.9e-3:
        p = 2 * np.pi * fd * (q["tx_delay"][:, None] + q["rx_delay"][None])
        assert (p < 32768).any() and (p > 32768).any()
    _close(*_images(cuda, q, fd, interp=interp), N * W)


@pytest.mark.parametrize("interp", [0, 1])
@pytest.mark.parametrize("fd", [0.0, 0.13])
def test_infinities_stay_infinities(cuda, fd, interp):
    """Infinite samples and weights, and weights whose product is moderate, give das_c's infinities and NaN."""
    print(f"case matrix both infinities fd={fd} interp={interp}", flush=True)
    q = matrix_problem(seed=6, P=260, N=9, W=6, F=5, L=80)
    q["ch"].imag[0, 3, 5, 20] = np.inf
    q["ch"].real[0, 2, 1, 40] = -np.inf
    q["ch"].real[1, 2, 1, 41:43] = np.inf
    q["rx_apo"][2, 230:240] = np.inf
    q["tx_apo"][1, 235:250] = -np.inf
    q["tx_apo"][:, 120:128] = 3e37       # with samples of 20: beyond FP32 before the receive weight
    q["rx_apo"][:, 120:128] = 1e-37
    q["ch"][2] *= 20.0
    got, ref = _images(cuda, q, fd, interp=interp)
    a, b = torch.view_as_real(got), torch.view_as_real(ref)
    fine = torch.isfinite(b)
    assert torch.isinf(b).any() and torch.isnan(b).any() and fine[2, 120:128].all()
    assert torch.equal(torch.where(fine, 0.0, a).nan_to_num(7.0), torch.where(fine, 0.0, b).nan_to_num(7.0))
    if fd == 0.0:  # no phase: FP64 is the better reference (das_c's order is 7e-7 from it at the moderate products)
        ex = O.beamform_fp64(q["ch"], q["fs"], q["t0"], q["tx_apo"], q["rx_apo"], q["tx_delay"], q["rx_delay"], fd, 3,
                             interp="cubic" if interp else "linear", w0=0.0, index="fp32")
        b = torch.view_as_real(torch.from_numpy(np.ascontiguousarray(ex.reshape(got.shape))).to(cuda))
    for f in range(5):
        err = (a[f] - b[f])[fine[f]].abs().max() / b[f][fine[f]].abs().max()
        assert err.item() <= 6e-8 * (4 + 54 ** 0.5)
