"""Rows of many edges in the one-launch-per-iteration PageRank: at the length
from which a row is summed in pieces, at the pieces' edges, rows side by side,
first and last; against the oracle's FP64 iteration (L1 1e-6, the bar of every
FP32 form) and, for the time, against the general form."""
import time

import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu

# (V, in-degrees of rows [at, at + n), other edges)
CASES = [
    (5000, 0, [2047, 2048, 2049], 3000),
    (5000, 4996, [4096, 4097, 0, 6145], 3000),
    (300, 100, [2049] * 9, 100),
    (70000, 69999, [70001], 0),
    (3, 1, [1000000], 0),  # tiles of one size at most, one row over all of them
    (900000, 7, [200000, 1, 0, 500000, 3000], 100000),
]


def _graph(gb, case):
    V, at, rows, extra = case
    rng = np.random.default_rng(V + extra)
    dst = np.repeat(np.arange(at, at + len(rows)), rows)
    src = rng.integers(0, V, len(dst) + extra)
    h = gb.HostCSR.from_edges(V, src, np.concatenate([dst, rng.integers(0, V, extra)]))
    r = h.transpose()
    return h, r, gb.Graph.from_host(h, reverse=r)


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"V{c[0]}")
def test_long_rows(gpu, case):
    gb = gpu
    import torch
    h, r, g = _graph(gb, case)
    x, res = gb.pagerank(g)
    assert (res["items_per_thread"], res["row_block"], res["binned"]) == (0, 0, 0)
    ref, it, _ = oracle.pagerank_cfg(r.row_ptr, r.col, h.outdeg(), 0.85, 1e-7, 100)
    assert np.abs(x.cpu().numpy().astype(np.float64) - ref).sum() <= 1e-6
    assert abs(res["iterations"] - it) <= 1
    # another form splits the handle's tiles anew in between
    gb.pagerank(g, items_per_thread=8)
    again, r2 = gb.pagerank(g)
    assert torch.equal(x, again) and r2 == res


def test_long_row_is_spread(gpu, monkeypatch):
    """A row of half the edges: one block over all of it took 25 times the
    general form's time."""
    gb = gpu
    import torch

    def best():
        t = []
        for _ in range(5):
            t0 = time.perf_counter()
            gb.pagerank(g, max_iter=20, tol=0.0)
            t.append(time.perf_counter() - t0)
        return min(t)

    _, _, g = _graph(gb, (16000, 7, [1 << 19], 20000))
    gb.pagerank(g)
    small = best()
    monkeypatch.setenv("GB_PR_SMALL", "0")
    gb.pagerank(g)
    assert small < 3 * best()
