"""Down-mixing and filtering at the edges of the kernel's forms: decimations
with a form of their own (1, 2) and without, tap counts around the lanes' blocks
of 4 and 8, trace lengths that leave part blocks and odd output rows (stores
of two outputs at the alignment of one), and a NaN sample, which only the
outputs whose taps reach it may show."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from ustb_amd import _lib as L
from ustb_amd import ops

pytestmark = pytest.mark.gpu
FS, T0, F0 = 20e6, 1.25e-6, 4.7e6


def _reference(x, b, down, mode):
    """FP64 sums of the FP32 mixed samples and FP32 taps, and the sums of magnitudes."""
    n = x.shape[-1]
    t = T0 + np.arange(n) / FS
    e = np.exp(-2j * np.pi * F0 * t).astype(np.complex64)
    v = (x * e.real).astype(np.float32) + 1j * (x * e.imag).astype(np.float32).astype(np.complex64)
    K = b.size
    if mode == L.FIR_CAUSAL:
        taps = b.astype(np.float32).astype(np.float64)
        ext = np.concatenate([np.zeros(v.shape[:-1] + (K - 1,)), v], -1)
    else:
        taps = np.correlate(b, b, "full").astype(np.float32).astype(np.float64)
        pre = (2 * v[..., :1] - v[..., K - 1:0:-1]).astype(np.complex64)
        post = (2 * v[..., -1:] - v[..., -2:-K - 1:-1]).astype(np.complex64)
        ext = np.concatenate([pre, v, post], -1)
    idx = (np.arange(0, n, down)[:, None] + np.arange(taps.size)[None, :])
    win = ext[..., idx].astype(np.complex128)
    w = taps[::-1] if mode == L.FIR_CAUSAL else taps
    return (win * w).sum(-1), (np.abs(win) * np.abs(w)).sum(-1)


@pytest.mark.parametrize("mode", [L.FIR_CAUSAL, L.FIR_ZERO_PHASE], ids=["causal", "zero_phase"])
@pytest.mark.parametrize("down", [1, 2, 3, 7])
@pytest.mark.parametrize("K,n", [(1, 5), (4, 64), (7, 257), (8, 1023), (9, 2049), (31, 4099), (97, 700)])
def test_edges_against_fp64(cuda, K, n, down, mode):
    print(f"case demodulate K={K} n={n} down={down} mode={mode}", flush=True)
    rng = np.random.default_rng(K * 10 + down)
    x = rng.standard_normal((3, n)).astype(np.float32)
    b = rng.standard_normal(K) / K
    ref, mag = _reference(x, b, down, mode)
    got = ops.demodulate(torch.from_numpy(x).to(cuda), FS, T0, F0, b, down, mode).cpu().numpy()
    assert got.shape == ref.shape
    # FP32 sums of up to 2K - 1 terms, and the edge samples' own rounding
    assert (np.abs(got - ref) <= (2 * K + 8) * 2.0 ** -24 * mag + 1e-30).all()
    x[1, n // 2] = np.nan
    bad, _ = _reference(x, b, down, mode)
    got = ops.demodulate(torch.from_numpy(x).to(cuda), FS, T0, F0, b, down, mode).cpu().numpy()
    assert np.array_equal(np.isnan(got.real), np.isnan(bad.real))
    ok = ~np.isnan(bad.real)
    assert (np.abs(got - bad)[ok] <= (2 * K + 8) * 2.0 ** -24 * mag[ok] + 1e-30).all()


@pytest.mark.parametrize("mode,K", [(L.FIR_CAUSAL, 63), (L.FIR_CAUSAL, 64), (L.FIR_CAUSAL, 65), (L.FIR_CAUSAL, 767),
                                    (L.FIR_ZERO_PHASE, 32), (L.FIR_ZERO_PHASE, 33), (L.FIR_ZERO_PHASE, 129),
                                    (L.FIR_ZERO_PHASE, 384)])
@pytest.mark.parametrize("n", [1156, 2311])
def test_long_filters_without_decimation(cuda, mode, K, n):
    """Taps in LDS from 64 on (zero phase: of the autocorrelation), up to the longest filters."""
    test_edges_against_fp64(cuda, K, n, 1, mode)
