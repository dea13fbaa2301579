"""The facade's plan key follows every array a plan is built from."""
from __future__ import annotations

import numpy as np
import pytest

from ustb_amd.das import DAS
from ustb_amd.uff import ChannelData, LinearArray, LinearScan, SectorScan, Wave, XYZScan

X, Z, Y = np.linspace(-5e-3, 5e-3, 6), np.linspace(5e-3, 20e-3, 9), np.linspace(-1e-3, 1e-3, 3)
A = np.deg2rad(X * 1e3)


def _key(scan, samples=256, frames=1):
    das = DAS()
    das.channel_data = ChannelData(probe=LinearArray(8, 0.3e-3), sequence=[Wave.plane(0.0)], sampling_frequency=2e7,
                                   initial_time=0.0, sound_speed=1540.0, modulation_frequency=0.0)
    das.scan = scan
    return das._plan_key(samples, frames)


@pytest.mark.parametrize("make", [lambda: LinearScan(X, Z, Y), lambda: SectorScan(A, Z, A[:2], (0.0, 0.0, -1e-3)),
                                  lambda: XYZScan(X, X, X + 1e-2)])
def test_equal_scans_share_a_key(make):
    assert _key(make()) == _key(make())
    assert _key(make()) != _key(make(), frames=2)


def test_every_scan_array_counts():
    bump = lambda a: np.where(np.arange(a.size) == a.size // 2, a + 1e-9, a)
    scans = [LinearScan(X, Z, Y), LinearScan(bump(X), Z, Y), LinearScan(X, bump(Z), Y), LinearScan(X, Z, bump(Y)),
             LinearScan(X, Z), LinearScan(Z, X), SectorScan(A, Z), SectorScan(bump(A), Z), SectorScan(A, bump(Z)),
             SectorScan(A, Z, A[:2]), SectorScan(A, Z, bump(A[:2])), SectorScan(A, Z, origin=(0.0, 0.0, 1e-9)),
             LinearScan(A, Z), XYZScan(X, X, X), XYZScan(X, bump(X), X),
             # the same values split over the axes elsewhere
             LinearScan(np.r_[X, Y[:1]], Z, Y[1:]), LinearScan(X, np.r_[Z, X[:1]], Y)]
    keys = [_key(s) for s in scans]
    assert len(set(keys)) == len(keys)
