"""CSR builds one after another under an allocation cap that each fits alone:
what an earlier build left (weights, row ids) makes room."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_builds_make_room(gpu):
    gb = gpu
    import torch
    rng = np.random.default_rng(2)
    V, E, E2 = 65536, 1 << 20, 1200000
    d = lambda a: torch.from_numpy(a).cuda()
    src, dst = rng.integers(0, V, E2).astype(np.int32), rng.integers(0, V, E2).astype(np.int32)
    w = rng.random(E)
    L = gb.lib()
    L.gb_release_workspaces()
    L.gb_set_mem_cap(25500000)
    try:
        # 25.3 MB: row ids, two key arrays, values and 8-byte weights
        rp, col, wo = gb.csr_from_edges(V, d(src[:E]), d(dst[:E]), d(w))
        trp, tcol, tw = gb.csr_transpose(rp, col, wo)
        # 15 MB without weights, beside 12.6 MB of row ids and weights
        rp2, col2, _ = gb.csr_from_edges(V, d(src), d(dst))
        # 20 MB: row ids that must grow first
        trp2, tcol2, _ = gb.csr_transpose(rp2, col2)
    finally:
        L.gb_set_mem_cap(0)
    o = np.argsort(src[:E], kind="stable")
    t = np.argsort(dst[:E][o], kind="stable")
    assert np.array_equal(tcol.cpu().numpy(), src[:E][o][t])
    assert np.array_equal(tw.cpu().numpy(), w[o][t])
    o = np.argsort(src, kind="stable")
    t = np.argsort(dst[o], kind="stable")
    assert np.array_equal(col2.cpu().numpy(), dst[o])
    assert np.array_equal(tcol2.cpu().numpy(), src[o][t])
    assert np.array_equal(trp2.cpu().numpy(),
                          np.concatenate([[0], np.cumsum(np.bincount(dst, minlength=V))]))
