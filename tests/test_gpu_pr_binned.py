"""The binned PageRank's shared values: a source's edges into one bin read one
value, whose index each edge counts from bits in the batch.  Against the
oracle's FP64 iteration, row by row: every term is positive, and an iteration
rounds a term at most six times to FP32 (rank, 1 / out-degree, their product,
the sum, the damped sum, the new rank), so three iterations stay within
18 * 2^-24 = 1.1e-6 of a row; the fixed-point sums add less than 1e-9."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _edges(kind, rng):
    V = 45001  # no multiple of a bin or chunk: a short last one of each
    if kind == "runs":  # 1 to 9 edges of a source in one bin, across batches
        src = np.repeat(np.arange(V), 1 + np.arange(V) % 9)
        return V, src, (src // 3 + 7 * np.arange(len(src)) % 4096) % V
    if kind == "long":  # one source's run over many batches and pieces
        src = np.concatenate([np.full(20011, 30000), np.full(9000, 5), rng.integers(0, V, 3000)])
        return V, src, rng.integers(0, 8192, len(src))
    if kind == "hub":  # only hub sources; most bins' other segments are empty
        return V, rng.integers(0, 8192, 60000), rng.integers(0, V, 60000)
    if kind == "nohub":  # no hub source, bins without edges
        return V, rng.integers(20480, V, 60000), rng.integers(0, V, 60000) // 8192 * 8192 % 24576
    if kind == "even":  # bins of one size, left whole
        return 150001, rng.integers(0, 150001, 700000), rng.integers(0, 150001, 700000)
    if kind == "skew":  # a few bins with most edges
        return 150001, rng.integers(0, 150001, 400000), rng.integers(0, 387, 400000) ** 2
    if kind == "sparse":  # segments of 0 to 5 values
        return V, rng.integers(0, V, 70), rng.integers(0, V, 70)
    src = rng.integers(0, V, 65536)  # "batch": bins near whole batches of 256
    return V, src, src * 13 % V


@pytest.mark.parametrize("kind", ["runs", "long", "hub", "nohub", "even", "skew", "sparse", "batch"])
@pytest.mark.parametrize("piece", ["4096", None])
def test_shared_values(gpu, monkeypatch, kind, piece):
    gb = gpu
    if piece:
        monkeypatch.setenv("GB_PR_PB_PIECE", piece)
    V, src, dst = _edges(kind, np.random.default_rng(len(kind)))
    h = gb.HostCSR.from_edges(V, src, dst)
    r = h.transpose()
    g = gb.Graph.from_host(h, reverse=r)
    ref, _, _ = oracle.pagerank_cfg(r.row_ptr, r.col, h.outdeg(), 0.85, 0.0, 3)
    for shape in range(1, 7):
        for relabel in (-1, 1):
            x, res = gb.pagerank(g, binned=shape, relabel=relabel, max_iter=3, tol=0.0)
            assert res["binned"] == shape and res["iterations"] == 3
            err = np.abs(x.cpu().numpy().astype(np.float64) - ref) / ref
            assert err.max() <= 1.2e-6, (shape, relabel)
