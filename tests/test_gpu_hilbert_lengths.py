"""The analytic signal at the lengths where its LDS convolution changes
(edges of the power-of-two transforms, primes, the shortest and longest
trace), and its isolation of traces with samples that are not finite."""
from __future__ import annotations

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from oracle import oracle as O
from ustb_amd.ops import hilbert

pytestmark = pytest.mark.gpu
# FP32 FFTs of up to 2^14 points, two of them: the usual bound log2(N) * eps
# per transform is 2 * 14 * 6e-8 = 1.7e-6 of the RMS; of the peak, 1e-6 is the
# tenth of the module's contract 1e-5
TOL = 2e-6


@pytest.mark.parametrize("L", [1, 2, 3, 4, 5, 255, 256, 257, 511, 513, 1023, 1025, 1531, 1600, 2047, 2049, 2176, 4095,
                               4097, 6144, 8191, 8192, 8193])
@pytest.mark.parametrize("traces", [1, 5])
def test_every_length(cuda, L, traces):
    print(f"case hilbert L={L} traces={traces}", flush=True)
    x = np.random.default_rng(L).standard_normal((traces, L)).astype(np.float32)
    got = hilbert(torch.from_numpy(x).to(cuda)).cpu().numpy()
    ref = O.hilbert(x.astype(np.float64), axis=-1)
    assert np.max(np.abs(got - ref)) <= TOL * max(1.0, float(np.max(np.abs(ref))))


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
@pytest.mark.parametrize("L", [301, 1527, 5003])
def test_non_finite_trace_stays_alone(cuda, L, bad):
    print(f"case hilbert non-finite L={L} {bad}", flush=True)
    x = np.random.default_rng(L).standard_normal((5, L)).astype(np.float32)
    x[1, L - 2] = bad
    x[4, 0] = bad
    got = hilbert(torch.from_numpy(x).to(cuda)).cpu().numpy()
    assert np.isnan(got[[1, 4]].real).all() and np.isnan(got[[1, 4]].imag).all()
    ref = O.hilbert(x[[0, 2, 3]].astype(np.float64), axis=-1)
    assert np.max(np.abs(got[[0, 2, 3]] - ref)) <= TOL * float(np.max(np.abs(ref)))


def test_more_traces_than_one_grid(cuda):
    """A grid holds fewer than 2^32 threads: 2^27 traces of the shortest transform."""
    L, traces = 5, (1 << 27) + 12345
    print(f"case hilbert L={L} traces={traces}", flush=True)
    x = torch.randn((traces, L), device=cuda, generator=torch.Generator(cuda).manual_seed(5))
    z = hilbert(x)
    for at in (0, (1 << 27) - 200, traces - 200):  # even: the same pairs
        at -= at % 2
        assert torch.equal(z[at:at + 200], hilbert(x[at:at + 200].contiguous()))
