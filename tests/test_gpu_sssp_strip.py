"""Merged buckets on a graph of high diameter: a long strip of a grid, where
every phase is small.  Ranges that widened as long as phases were small made the
solve relax each edge hundreds of times."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsrc", [1, 8, 40])
def test_strip_relaxes_few_edges_again(gpu, nsrc):
    gb = gpu
    n, m = 30, 4000
    i = np.arange(n * m).reshape(n, m)
    a = np.concatenate([i[:, :-1].ravel(), i[:-1, :].ravel()])
    b = np.concatenate([i[:, 1:].ravel(), i[1:, :].ravel()])
    rng = np.random.default_rng(3)
    w = rng.integers(1, 256, 2 * len(a)).astype(np.uint32)
    h = gb.HostCSR.from_edges(n * m, np.concatenate([a, b]), np.concatenate([b, a]), w)
    g = gb.Graph.from_host(h, need_reverse=False)
    srcs = rng.integers(0, n * m, nsrc).astype(np.int32)
    d, st = gb.sssp(g, srcs, stats=True)
    for k in (0, nsrc - 1):
        assert np.array_equal(gb.u32(d)[k], oracle.dijkstra(h.row_ptr, h.col, h.w, int(srcs[k])))
    # 2 to 5 with ranges of at most about SPAN_MOST phases, 20 and more without
    assert st["relax_edges"] <= 10 * st["traversed"]
