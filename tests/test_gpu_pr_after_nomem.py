"""PageRank on a handle after another form's tables found no memory: the tables
of the form used before were given up for them and are built again."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

COARSE = [dict(items_per_thread=16), dict(row_block=4096)]
FINE = {"small": dict(), "merge": dict(items_per_thread=4), "rows": dict(row_block=1024)}


@pytest.mark.parametrize("fine", FINE)
@pytest.mark.parametrize("coarse", COARSE, ids=["merge", "rows"])
def test_form_after_a_failed_one(gpu, coarse, fine):
    gb = gpu
    import torch
    rng = np.random.default_rng(1)
    V, E = 30000, 400000
    h = gb.HostCSR.from_edges(V, rng.integers(0, V, E), rng.integers(0, V, E))
    g = gb.Graph.from_host(h)
    ref, _ = gb.pagerank(g, **coarse)
    gb.lib().gb_set_mem_cap(1)
    try:
        with pytest.raises(gb.GBError):
            gb.pagerank(g, **FINE[fine])
    finally:
        gb.lib().gb_set_mem_cap(0)
    x, _ = gb.pagerank(g, **coarse)
    assert torch.equal(x, ref)
    y, _ = gb.pagerank(g, **FINE[fine])
    assert float((y.double() - ref.double()).abs().sum()) <= 1e-6
