"""SSSP and weighted Brandes in one workgroup per source, at the edges of the
form's LDS sizes, queue and launches, against the oracle."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _graph(gb, kind, V, rng, wmax=255):
    if kind == "star":  # a hub, and every leaf back to it and to the next one
        leaf = np.arange(1, V)
        src = np.concatenate([np.zeros(V - 1, np.int64), leaf, leaf])
        dst = np.concatenate([leaf, np.zeros(V - 1, np.int64), leaf % (V - 1) + 1])
    elif kind == "path":
        src, dst = np.arange(V - 1), np.arange(1, V)
    else:  # half of the vertices have no edges; parallel edges and self-loops stay
        E = max(1, V * 6)
        src, dst = rng.integers(0, max(1, V // 2), E), rng.integers(0, V, E)
    w = rng.integers(0, wmax + 1, len(src)).astype(np.uint32)
    return gb.HostCSR.from_edges(V, src, dst, w)


# 8192 / 32768 vertices are the two LDS sizes; queue of 8192, batches of 1024
CASES = [("random", 1), ("random", 2), ("random", 63), ("random", 65), ("random", 8192),
         ("random", 8193), ("random", 32768), ("random", 32769), ("star", 30000), ("path", 3000)]


@pytest.mark.parametrize("kind,V", CASES)
@pytest.mark.parametrize("delta", [0, 1, 1 << 20])
def test_sssp_u32(gpu, kind, V, delta):
    gb = gpu
    h = _graph(gb, kind, V, np.random.default_rng(V))
    g = gb.Graph.from_host(h, need_reverse=False)
    srcs = [0, V // 2, V - 1]
    d, st = gb.sssp(g, srcs, delta=delta, stats=True)
    reached = trav = 0
    for i, s in enumerate(srcs):
        ref = oracle.dijkstra(h.row_ptr, h.col, h.w, s)
        assert np.array_equal(gb.u32(d)[i], ref)
        ok = ref != oracle.UINF
        reached += int(ok.sum())
        trav += int(h.outdeg()[ok].sum())
    assert (st["reached"], st["traversed"]) == (reached, trav)
    assert st["relax_edges"] >= trav


def test_sssp_more_sources_than_a_launch(gpu, monkeypatch):
    gb = gpu
    h = _graph(gb, "random", 700, np.random.default_rng(5))
    g = gb.Graph.from_host(h, need_reverse=False)
    srcs = np.arange(600) % 350
    d = gb.u32(gb.sssp(g, srcs))
    monkeypatch.setenv("GB_SSSP_SMALL", "0")
    assert np.array_equal(d, gb.u32(gb.sssp(g, srcs)))  # the batched engine


@pytest.mark.parametrize("nsrc", [1, 3])
def test_sssp_overflow_verdict_is_the_engines(gpu, monkeypatch, nsrc):
    """A sum past 2^32 - 2 is left to the engine: a vertex first reached over a
    heavy edge and then over light ones is fine, a far one is refused."""
    gb = gpu
    big = 4_000_000_000
    src, dst = [0, 0, 1, 2], [1, 2, 2, 3]
    for last, fails in ((10, False), (big, True)):
        w = np.array([5, big, 5, last], np.uint32)
        h = gb.HostCSR.from_edges(4, src, dst, w)
        if fails:
            h = gb.HostCSR.from_edges(5, src + [3], dst + [4], np.append(w, np.uint32(big)))
        g = gb.Graph.from_host(h, need_reverse=False)
        seen = []
        for small in ("1", "0"):
            monkeypatch.setenv("GB_SSSP_SMALL", small)
            try:
                seen.append(gb.u32(gb.sssp(g, [0] * nsrc, delta=16)).tolist())
            except gb.GBError as e:
                seen.append(e.status)
        assert seen[0] == seen[1]
        assert (seen[0] == 4) == fails


# 4096 / 16384 vertices are the two LDS sizes of FP64 distances
@pytest.mark.parametrize("kind,V", [("random", 1), ("random", 64), ("random", 4096),
                                    ("random", 4097), ("random", 16384), ("star", 16000),
                                    ("path", 2000)])
def test_sssp_f64(gpu, kind, V):
    gb = gpu
    h = _graph(gb, kind, V, np.random.default_rng(V + 1))
    w64 = h.w.astype(np.float64) / 7.0
    g = gb.Graph.from_host(h, need_reverse=False, w64=w64)
    for delta in (0.1, 1e9):
        d = gb.sssp_f64(g, [0, V - 1], delta).cpu().numpy()
        for i, s in enumerate((0, V - 1)):
            assert np.array_equal(d[i], oracle.dijkstra(h.row_ptr, h.col, w64, s))


@pytest.mark.parametrize("kind,V,nsrc,batch", [("random", 3, 2, 0), ("random", 4096, 5, 2),
                                               ("random", 4097, 4, 0), ("random", 16384, 3, 0),
                                               ("star", 9000, 2, 0), ("path", 700, 3, 0),
                                               ("random", 150, 300, 0)])
def test_bc_weighted(gpu, kind, V, nsrc, batch):
    """Hubs past 128 out-edges, levels wider than a queue, one level per vertex,
    more sources than a launch.  Sums of at most V * nsrc dependencies, each a
    few ulps off the oracle's: 1e-12 relative, as the engine's form is held to
    1e-9."""
    gb = gpu
    rng = np.random.default_rng(V + 2)
    h = _graph(gb, kind, V, rng)
    h.w[:] = np.maximum(h.w, 1)
    r = h.transpose()
    w64, rw64 = h.w.astype(np.float64) / 8.0, r.w.astype(np.float64) / 8.0
    g = gb.Graph.from_host(h, reverse=r, w64=w64, rw64=rw64)
    srcs = [int(x) for x in rng.integers(0, V, nsrc)]
    bc = gb.bc(g, srcs, batch=batch, weighted=True).cpu().numpy()
    ref = oracle.brandes_weighted(h.row_ptr, h.col, w64, r.row_ptr, r.col, rw64, srcs)
    np.testing.assert_allclose(bc, ref, rtol=1e-12, atol=1e-9 * max(1.0, np.abs(ref).max()) * 1e-3)


# 4096 / 14336 vertices are the two LDS sizes; past them the batched engine
@pytest.mark.parametrize("kind,V,nsrc,batch", [("random", 1, 1, 0), ("random", 64, 9, 0),
                                               ("random", 4096, 70, 64), ("random", 4097, 6, 0),
                                               ("random", 14336, 3, 0), ("random", 14337, 3, 0),
                                               ("star", 14000, 2, 0), ("path", 900, 3, 0),
                                               ("random", 150, 300, 0)])
def test_bc_unweighted(gpu, kind, V, nsrc, batch):
    """Directed graphs with parallel edges, self-loops and unreached vertices:
    hubs past 128 out-edges, levels wider than a batch of the edge spreading,
    one level per vertex, more sources than a launch."""
    gb = gpu
    rng = np.random.default_rng(V + 3)
    h = _graph(gb, kind, V, rng)
    h = gb.HostCSR(h.row_ptr, h.col)
    r = h.transpose()
    g = gb.Graph.from_host(h, reverse=r)
    srcs = [int(x) for x in rng.integers(0, V, nsrc)]
    bc, st = gb.bc(g, srcs, batch=batch, stats=True)
    ref = oracle.brandes_bfs(h.row_ptr, h.col, srcs, r.row_ptr, r.col)
    np.testing.assert_allclose(bc.cpu().numpy(), ref, rtol=1e-12, atol=1e-12)
    depth = max(int(oracle.bfs_levels(h.row_ptr, h.col, s).max()) for s in srcs)
    assert st["max_depth"] == depth
