"""Solves under allocation caps that they fitted with two queues and without
lists of their own for one direction: batched SSSP, BFS."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _capped(gb, cap, f):
    gb.lib().gb_release_workspaces()
    gb.lib().gb_set_mem_cap(cap)
    try:
        return f()
    finally:
        gb.lib().gb_set_mem_cap(0)


@pytest.mark.parametrize("tune", ["0", "1"])
def test_batched_sssp(gpu, monkeypatch, tune):
    """65536 vertices, 1 M edges, 8 sources: 11.6 MB."""
    gb = gpu
    monkeypatch.setenv("GB_MSSSP_TUNE", tune)
    h = gb.gen_rmat(16, 16, seed=3, weights="uniform", wlo=1, whi=255)
    srcs = gb.pick_sources(h, 8, 1)
    g = gb.Graph.from_host(h, need_reverse=False)
    for _ in range(2):
        d = gb.u32(_capped(gb, 11600000, lambda: gb.sssp(g, srcs, delta=100)))
        for i in (0, 7):
            assert np.array_equal(d[i], oracle.dijkstra(h.row_ptr, h.col, h.w, int(srcs[i])))
    # and the form of the rule again once there is room
    assert np.array_equal(gb.u32(gb.sssp(g, srcs, delta=100)), d)


def test_bfs(gpu):
    """32768 vertices, 1 M edges: 3.16 MB."""
    gb = gpu
    h = gb.gen_rmat(15, 16, seed=3, weights="none", symmetric=True)
    srcs = gb.pick_sources(h, 3, 1)
    g = gb.Graph.from_host(h, need_reverse=False)
    lv = _capped(gb, 3160000, lambda: gb.bfs(g, srcs)).cpu().numpy()
    for i in range(3):
        assert np.array_equal(lv[i], oracle.bfs_levels(h.row_ptr, h.col, int(srcs[i])))
