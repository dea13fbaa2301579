"""A captured graph with a Hilbert call keeps what it reads: its length's table
stays while more other lengths pass through than the table pool holds."""
from __future__ import annotations

import pytest

torch = pytest.importorskip("torch")

from ustb_amd.ops import hilbert

pytestmark = pytest.mark.gpu


def test_replays_outlive_the_table_pool(cuda):
    lengths = (270, 1500, 1527)
    g = torch.Generator(cuda).manual_seed(1)
    x = {L: torch.randn((5, L), device=cuda, generator=g) for L in lengths}
    z = {L: torch.empty((5, L), dtype=torch.complex64, device=cuda) for L in lengths}
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        for L in lengths:  # builds the tables
            hilbert(x[L], out=z[L])
    side.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        for L in lengths:
            hilbert(x[L], out=z[L])
    for k in range(3):
        for L in range(300 + 70 * k, 370 + 70 * k):  # a pool holds 64 tables
            hilbert(torch.ones((1, L), device=cuda))
        torch.cuda.synchronize()
        for L in lengths:
            x[L].copy_(torch.randn((5, L), device=cuda, generator=g))
            z[L].zero_()
        print(f"case hilbert graph replay {k}", flush=True)
        graph.replay()
        torch.cuda.synchronize()
        for L in lengths:
            assert torch.equal(z[L], hilbert(x[L])), (k, L)
