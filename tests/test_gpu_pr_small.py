"""The one-launch-per-iteration PageRank at the edges of its tiles, chunks and
limits, against the oracle's FP64 iteration: L1 1e-6, the bar of every FP32
form (V * 2^-24 relative rounding of ranks summing to 1 stays under 1e-7)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _case(kind, rng):
    if kind == "one":
        return 1, [0], [0]
    if kind == "noedge":
        return 700, [], []
    if kind == "tile":  # V + E = one tile of 1024 exactly
        return 24, rng.integers(0, 24, 1000), rng.integers(0, 24, 1000)
    if kind == "hub":  # one row of many chunks, between empty rows
        return 3000, rng.integers(0, 3000, 50000), np.full(50000, 1500)
    if kind == "hubs":  # rows that begin and end inside chunks
        return 50, rng.integers(0, 50, 30011), rng.integers(20, 27, 30011)
    if kind == "empty":  # far more rows than edges
        return 300000, rng.integers(0, 300000, 2000), rng.integers(0, 300000, 2000)
    if kind == "ragged":
        return 20011, rng.integers(0, 20011, 160000), rng.integers(0, 20011, 160000) // 3
    # past 1024 blocks of 1024 items
    return 1000003, rng.integers(0, 1000003, 1000000), rng.integers(0, 1000003, 1000000)


@pytest.mark.parametrize("kind", ["one", "noedge", "tile", "hub", "hubs", "empty", "ragged", "most"])
def test_matches_oracle(gpu, monkeypatch, kind):
    gb = gpu
    import torch
    rng = np.random.default_rng(len(kind))
    V, src, dst = _case(kind, rng)
    h = gb.HostCSR.from_edges(V, src, dst)
    r = h.transpose()
    g = gb.Graph.from_host(h, reverse=r)
    x, res = gb.pagerank(g)
    assert (res["items_per_thread"], res["row_block"], res["binned"]) == (0, 0, 0)
    ref, it, _ = oracle.pagerank_cfg(r.row_ptr, r.col, h.outdeg(), 0.85, 1e-7, 100)
    assert np.abs(x.cpu().numpy().astype(np.float64) - ref).sum() <= 1e-6
    assert abs(res["iterations"] - it) <= 1
    again, r2 = gb.pagerank(g, use_graph=False)
    assert torch.equal(x, again) and r2 == res
    # a start of its own, in the output array, and a cap on the iterations
    y = torch.rand(V, device="cuda") + 0.1
    y /= y.sum()
    y0 = y.clone()
    z, rz = gb.pagerank(g, x0=y, out=y, max_iter=3, tol=0.0)
    monkeypatch.setenv("GB_PR_SMALL", "0")
    zo, ro = gb.pagerank(g, x0=y0, max_iter=3, tol=0.0)
    assert (rz["iterations"], ro["iterations"]) == (3, 3)
    assert float((z.double() - zo.double()).abs().sum()) <= 1e-6
    assert abs(rz["residual"] - ro["residual"]) <= 1e-6
    assert abs(rz["dangling"] - ro["dangling"]) <= 1e-6
    monkeypatch.delenv("GB_PR_SMALL")
    _, r0 = gb.pagerank(g, max_iter=0)
    assert r0["iterations"] == 0 and r0["converged"] == 0
