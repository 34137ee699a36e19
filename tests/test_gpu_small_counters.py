"""Relaxation outcomes of the one-workgroup SSSP, pinned on out-trees: a
vertex's one in-edge is relaxed once, and the improvement is near iff it stays in
the bucket of the caller's width, whatever ranges the solve steps over.  The two
LDS sizes of each distance type, one source and several."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [3000, 16384])
@pytest.mark.parametrize("nsrc", [1, 5])
@pytest.mark.parametrize("wide", [False, True])
def test_counters_on_a_tree(gpu, V, nsrc, wide):
    gb = gpu
    rng = np.random.default_rng(V + nsrc)
    parent = np.array([rng.integers(0, i) for i in range(1, V)])
    w = rng.integers(1, 301, V - 1).astype(np.uint32)
    h = gb.HostCSR.from_edges(V, parent, np.arange(1, V), w)
    srcs = np.concatenate([[0], rng.integers(1, V, nsrc - 1)]).astype(np.int32)
    if wide:  # FP64: eighths, exact in every sum
        w64 = h.w.astype(np.float64) / 8.0
        g = gb.Graph.from_host(h, need_reverse=False, w64=w64)
    else:
        g = gb.Graph.from_host(h, need_reverse=False)
    at = np.repeat(np.arange(V), np.diff(h.row_ptr))
    for delta in (1, 3, 50, 200, 1 << 20):
        if wide:
            d, st = gb.sssp_f64(g, srcs, float(delta) / 8.0, stats=True)
            d = d.cpu().numpy()
            d = np.where(np.isinf(d), -1, d * 8).astype(np.int64)
        else:
            d, st = gb.sssp(g, srcs, delta=delta, stats=True)
            d = gb.u32(d).astype(np.int64)
            d = np.where(d == 0xFFFFFFFF, -1, d)
        near = far = 0
        for i in range(nsrc):
            du = d[i][at]
            ok = du >= 0
            stays = (du[ok] + h.w[ok]) // delta == du[ok] // delta
            near += int(stays.sum())
            far += int((~stays).sum())
        assert st["relax_edges"] == near + far == st["traversed"]
        assert (st["improved_near"], st["improved_far"]) == (near, far), delta
