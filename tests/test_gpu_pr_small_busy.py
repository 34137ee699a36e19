"""The one-launch-per-iteration PageRank beside work that holds compute units.

A launch's late blocks can start after its block 0 has set the stop flag: a
block must then return as a whole or not at all.  Every solve gives the same
bits, whatever runs beside it.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_same_ranks_beside_a_busy_stream(gpu):
    gb = gpu
    import torch
    rng = np.random.default_rng(17)
    V, E = 60000, 900000
    h = gb.HostCSR.from_edges(V, rng.integers(0, V, E), rng.integers(0, V, E))
    g = gb.Graph.from_host(h)
    ref, r0 = gb.pagerank(g)
    assert (r0["items_per_thread"], r0["row_block"], r0["binned"]) == (0, 0, 0)
    a = torch.rand(1 << 26, device="cuda")
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for _ in range(20):
        with torch.cuda.stream(side):
            for _ in range(8):
                a.mul_(1.000001)
        for _ in range(5):
            x, r = gb.pagerank(g)
            assert torch.equal(x, ref) and r == r0
    side.synchronize()
