"""Weighted Brandes with infinite weights (edges that lead nowhere): the
one-workgroup form takes what the engine takes and gives its scores."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [60, 5000])
def test_infinite_weights(gpu, monkeypatch, V):
    gb = gpu
    import torch
    rng = np.random.default_rng(V)
    # the last tenth is reached over infinite weights only
    lim = V - V // 10
    E = 6 * V
    src, dst = rng.integers(0, lim, E), rng.integers(0, lim, E)
    w = rng.integers(1, 64, E).astype(np.float64) / 8.0
    far = rng.integers(0, lim, V // 20)
    src = np.concatenate([src, far, rng.integers(lim, V, V // 10)])
    dst = np.concatenate([dst, rng.integers(lim, V, V // 20), rng.integers(lim, V, V // 10)])
    w = np.concatenate([w, np.full(V // 20, np.inf), np.full(V // 10, 2.0)])

    def csr(key, val):
        o = np.argsort(key, kind="stable")
        rp = np.concatenate([[0], np.cumsum(np.bincount(key, minlength=V))]).astype(np.int32)
        return [torch.from_numpy(a).cuda() for a in (rp, val[o].astype(np.int32), w[o])]

    rp, col, w64 = csr(src, dst)
    rrp, rcol, rw64 = csr(dst, src)
    g = gb.Graph(V, len(w), rp, col, None, rrp, rcol, None, w64, rw64)
    srcs = rng.integers(0, lim, 5).astype(np.int32)
    a = gb.bc(g, srcs, weighted=True)
    monkeypatch.setenv("GB_SSSP_SMALL", "0")
    b = gb.bc(g, srcs, weighted=True)
    assert bool(torch.isinf(b).any())  # a vertex before an infinite edge
    # sums of n terms in another order: a few n * 2^-53
    assert torch.allclose(a, b, rtol=1e-11, atol=0.0, equal_nan=True)
