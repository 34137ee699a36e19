"""Batched SSSP with a distance array of 4 GiB or more (64-bit offsets) and one
below, near the last vertices, against Dijkstra on the same edges over the
vertices that have any: distances are whole numbers, equal to the bit."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [(1 << 24) - 1, (1 << 24) + 5])  # x 64 sources x 4 bytes
@pytest.mark.parametrize("scan", ["0", "1"])
def test_wide_offsets(gpu, monkeypatch, V, scan):
    gb = gpu
    monkeypatch.setenv("GB_MSSSP_SCAN", scan)
    rng = np.random.default_rng(V)
    n = 3000  # vertices with edges: the first and the last ones
    ids = np.concatenate([np.arange(n // 2), np.arange(V - n // 2, V)])
    src, dst = rng.integers(0, n, 20000), rng.integers(0, n, 20000)
    w = rng.integers(1, 1 << 20, 20000).astype(np.uint32)
    small = gb.HostCSR.from_edges(n, src, dst, w)
    g = gb.Graph.from_host(gb.HostCSR.from_edges(V, ids[src], ids[dst], w), need_reverse=False)
    pick = rng.integers(0, n, 40)
    pick[0], pick[1] = n - 1, 0
    d = gb.u32(gb.sssp(g, ids[pick].astype(np.int32)))
    rest = np.setdiff1d(rng.integers(0, V, 2000), ids)
    for i, s in enumerate(pick):
        assert np.array_equal(d[i][ids], oracle.dijkstra(small.row_ptr, small.col, small.w, int(s)))
        assert (d[i][rest] == oracle.UINF).all()
