"""Weighted Brandes from one source of the largest graph of the one-workgroup
form, under an allocation cap that a solve by the engine fits (145 bytes a
vertex and 128 KB): level offsets are allocated for the sources there are."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_one_source_under_a_cap(gpu):
    gb = gpu
    import torch
    V, E = 16384, 65536
    rng = np.random.default_rng(8)
    src, dst = rng.integers(0, V, E), rng.integers(0, V, E)
    w = rng.integers(1, 64, E).astype(np.float64) / 8.0

    def csr(key, val):
        o = np.argsort(key, kind="stable")
        rp = np.concatenate([[0], np.cumsum(np.bincount(key, minlength=V))]).astype(np.int32)
        return [torch.from_numpy(a).cuda() for a in (rp, val[o].astype(np.int32), w[o])]

    rp, col, w64 = csr(src, dst)
    rrp, rcol, rw64 = csr(dst, src)
    g = gb.Graph(V, E, rp, col, None, rrp, rcol, None, w64, rw64)
    ref = gb.bc(g, [int(src[0])], weighted=True)
    gb.lib().gb_release_workspaces()
    gb.lib().gb_set_mem_cap(145 * V + (128 << 10))
    try:
        out = gb.bc(g, [int(src[0])], weighted=True)
    finally:
        gb.lib().gb_set_mem_cap(0)
    assert torch.equal(out, ref)
