"""Two traces share one transform: a trace's error is relative to its own norm
whatever its neighbour's amplitude, and nothing of a neighbour's range reaches
it."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from ustb_amd.ops import hilbert

pytestmark = pytest.mark.gpu


def _imag_error(cuda, x):
    """RMS error of each trace's imaginary part over its RMS."""
    got = hilbert(torch.from_numpy(x).to(cuda)).cpu().numpy()
    ref = O.hilbert(x.astype(np.float64), axis=-1)
    assert np.array_equal(got.real, x)
    d = np.sqrt(np.mean((got.imag.astype(np.float64) - ref.imag) ** 2, axis=-1))
    return d / np.sqrt(np.mean(x.astype(np.float64) ** 2, axis=-1))


# two FP32 transforms of up to 2^14 points: RMS error 0.6 * sqrt(log2 N) * 6e-8
# each, and a pair whose norms differ by up to 2: 4e-7
TOL = 5e-7


@pytest.mark.parametrize("L", [3, 301, 1021, 1527, 2049, 5003])
@pytest.mark.parametrize("db", [40, 80, 160, 300])
def test_unequal_amplitudes(cuda, L, db):
    print(f"case hilbert pair L={L} {db} dB", flush=True)
    rng = np.random.default_rng(L + db)
    x = rng.standard_normal((6, L))
    x[[0, 3, 4]] *= 10.0 ** (-db / 20)
    assert np.max(_imag_error(cuda, x.astype(np.float32))) <= TOL


@pytest.mark.parametrize("L", [301, 1527])
def test_unequal_crest_factors(cuda, L):
    print(f"case hilbert crest L={L}", flush=True)
    rng = np.random.default_rng(L)
    x = rng.standard_normal((4, L)).astype(np.float32)
    x[1] = 0.0
    x[1, L // 3] = 1.0
    x[2] = 0.0
    x[2, 5] = -3e-4
    assert np.max(_imag_error(cuda, x)) <= TOL


@pytest.mark.parametrize("L", [301, 1527, 5003])
def test_range_of_fp32(cuda, L):
    """Finite samples whose transform or squares leave FP32's range, subnormal
    samples and zero traces."""
    print(f"case hilbert range L={L}", flush=True)
    rng = np.random.default_rng(L)
    x = rng.uniform(-1.0, 1.0, (9, L))
    x[0] *= 1e37
    x[3] *= 3e38
    x[4] *= 1e-25
    x = x.astype(np.float32)
    x[5] = 0.0
    x[7] *= np.float32(1e-36)
    x[8] = 0.0
    with np.errstate(over="ignore"):
        got = hilbert(torch.from_numpy(x).to(cuda)).cpu().numpy()
    assert not got[[5, 8]].imag.any() and np.array_equal(got.real, x)
    ref = O.hilbert(x.astype(np.float64), axis=-1).imag
    for k in (0, 1, 2, 4, 6, 7):
        d = np.sqrt(np.mean((got[k].imag.astype(np.float64) - ref[k]) ** 2))
        assert d <= TOL * 4 * np.sqrt(np.mean(x[k].astype(np.float64) ** 2)), k  # scaled by the peak: norms up to sqrt(3) apart
    fits = np.abs(ref[3]) < 3.4e38  # beyond: infinite
    assert np.max(np.abs(got[3].imag[fits] - ref[3][fits])) <= 2e-6 * 3e38
    small = O.hilbert(x[7:8].astype(np.float64), axis=-1).imag[0]
    assert np.max(np.abs(got[7].imag - small)) <= 2e-6 * 1e-36 + 2.0 ** -149
