"""Brandes and BFS where vertices are summed by chunks: degrees around whole
chunks, hubs whose chunk counts share a factor with the waves, distinct in- and
out-hubs; rows that some sources of a group never reach; 3000 levels.  Against the oracle:
1e-12 relative (FP64 sums of positive terms in another order: n * 2^-53 with n
below 2000 terms per level and 4 levels stays under 1e-12)."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _graph(gb, kind, rng):
    V = 16001  # past the one-workgroup form
    if kind == "edges":  # degree chunk - 1 .. 3 chunks + 1
        degs = [255, 256, 257, 511, 512, 513, 767, 768, 769]
        src = np.repeat(np.arange(len(degs)), degs)
        dst = rng.integers(20, V, len(src))
    elif kind == "share":  # one hub of 64 chunks, many of two
        src = np.concatenate([np.zeros(15900, np.int64), np.repeat(np.arange(1, 60), 300)])
        dst = np.concatenate([np.arange(100, 16000), rng.integers(100, 16000, 59 * 300)])
    elif kind == "deep":  # more levels than the first level table and pool hold
        src, dst = np.arange(3000), np.arange(1, 3001)
    else:  # two components
        src = np.concatenate([rng.integers(0, 40, 30000), rng.integers(8000, V, 30000)])
        dst = np.concatenate([rng.integers(0, 7900, 30000), rng.integers(8000, V, 30000)])
    m = src != dst
    key = np.unique(src[m] * np.int64(V) + dst[m])
    return V, key // V, key % V


@pytest.mark.parametrize("kind", ["edges", "share", "deep", "parts"])
@pytest.mark.parametrize("directed", [False, True])
def test_hub_chunks(gpu, kind, directed):
    gb = gpu
    rng = np.random.default_rng(len(kind))
    V, src, dst = _graph(gb, kind, rng)
    if not directed:
        src, dst = np.concatenate([src, dst]), np.concatenate([dst, src])
        key = np.unique(src * np.int64(V) + dst)
        src, dst = key // V, key % V
    h = gb.HostCSR.from_edges(V, src, dst)
    r = h.transpose()
    g = gb.Graph.from_host(h, reverse=r) if directed else gb.Graph.from_host(h, need_reverse=False)
    srcs = np.concatenate([np.arange(0, 9), rng.integers(0, 3000 if kind == "deep" else V, 80),
                           [V - 1, 0]]).astype(np.int32)
    ref = oracle.brandes_bfs(h.row_ptr, h.col, srcs, r.row_ptr, r.col)
    both = [gb.bc(g, srcs, batch=batch).cpu().numpy() for batch in (0, 64)]
    for bc in both:
        np.testing.assert_allclose(bc, ref, rtol=1e-12, atol=1e-12)
    # sources are grouped by their reach over the whole call, not by batch
    assert np.array_equal(*both)
    mixed = gb.bc(g, rng.permutation(srcs)).cpu().numpy()
    np.testing.assert_allclose(mixed, ref, rtol=1e-12, atol=1e-12)
    lv = gb.bfs(g, srcs[:12]).cpu().numpy()
    for i, s in enumerate(srcs[:12]):
        assert np.array_equal(lv[i], oracle.bfs_levels(h.row_ptr, h.col, int(s)))
