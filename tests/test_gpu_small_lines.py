"""Calls on both sides of the lines between one workgroup per source and the
engines: wide widths, many sources, FP64 weights of any scale."""
import numpy as np
import pytest

import oracle

pytestmark = pytest.mark.gpu


def _graph(gb, V, E, seed):
    rng = np.random.default_rng(seed)
    return gb.HostCSR.from_edges(V, rng.integers(0, V, E), rng.integers(0, V, E),
                                 rng.integers(0, 500, E).astype(np.uint32))


# past 2^17 edges one source, past 2^19 less than 64 sources with a wide width
@pytest.mark.parametrize("E,nsrc", [((1 << 17) + 3, 1), ((1 << 19) + 3, 32), ((1 << 19) + 3, 64)])
@pytest.mark.parametrize("delta", [1, 8, 1 << 31])
def test_sssp_widths(gpu, E, nsrc, delta):
    gb = gpu
    h = _graph(gb, 3000, E, nsrc)
    g = gb.Graph.from_host(h, need_reverse=False)
    srcs = np.random.default_rng(1).integers(0, 3000, nsrc).astype(np.int32)
    d, st = gb.sssp(g, srcs, delta=delta, stats=True)
    for i in (0, nsrc - 1):
        assert np.array_equal(gb.u32(d)[i], oracle.dijkstra(h.row_ptr, h.col, h.w, int(srcs[i])))
    if delta == 1 << 31:  # every distance lies in the first bucket
        assert st["improved_far"] == 0 and st["improved_near"] > 0


@pytest.mark.parametrize("scale", [1e-12, 1.0, 1e12])
@pytest.mark.parametrize("E,nsrc", [(0, 1), (700, 1), (50000, 3), ((1 << 19) + 3, 32),
                                    ((1 << 19) + 3, 64)])
def test_sssp_f64_scales(gpu, scale, E, nsrc):
    gb = gpu
    h = _graph(gb, 1000, E, nsrc + E)
    w64 = h.w.astype(np.float64) * scale
    g = gb.Graph.from_host(h, need_reverse=False, w64=w64)
    srcs = np.random.default_rng(1).integers(0, 1000, nsrc).astype(np.int32)
    for delta in (scale, 1e9):
        d = gb.sssp_f64(g, srcs, delta).cpu().numpy()
        for i in (0, nsrc - 1):
            assert np.array_equal(d[i], oracle.dijkstra(h.row_ptr, h.col, w64, int(srcs[i])))


# 257 sources are two launches: from 2^18 edges on the engine's
@pytest.mark.parametrize("E", [1 << 18, (1 << 18) + 1])
@pytest.mark.parametrize("nsrc,batch", [(256, 0), (257, 0), (257, 64)])
def test_bc_launches(gpu, monkeypatch, E, nsrc, batch):
    gb = gpu
    import torch
    h = _graph(gb, 600, E, 3)
    g = gb.Graph.from_host(gb.HostCSR(h.row_ptr, h.col))
    srcs = np.random.default_rng(2).integers(0, 600, nsrc).astype(np.int32)
    a = gb.bc(g, srcs, batch=batch)
    # a form for the whole call: the batches change no bit
    assert torch.equal(a, gb.bc(g, srcs))
    monkeypatch.setenv("GB_BC_SMALL", "0")
    # sums of nsrc * 600 terms at most, in another order
    assert torch.allclose(a, gb.bc(g, srcs), rtol=1e-10, atol=1e-10)
