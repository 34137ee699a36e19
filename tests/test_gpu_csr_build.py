"""The radix build of CSRs at the edges of its tiles, digits and scan groups,
against numpy's stable sort."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (V, E, rows drawn from): one digit (V <= 2048), two, three; tiles of 8192
# edges, scan groups of 64 tiles; one row only; almost only empty rows
SIZES = [(1, 1, 1), (2048, 8192, 2048), (2049, 8193, 2049), (70000, 64 * 8192 + 1, 70000),
         ((1 << 22) + 1, 100003, (1 << 22) + 1), (5000, 40000, 1), (3000000, 50, 3000000)]


@pytest.mark.parametrize("V,E,span", SIZES)
@pytest.mark.parametrize("wb", [0, 4, 8])
def test_build_and_transpose(gpu, V, E, span, wb):
    gb = gpu
    import torch
    rng = np.random.default_rng(V + E + wb)
    src = (rng.integers(0, span, E) if span > 1 else np.full(E, V // 2)).astype(np.int32)
    dst = rng.integers(0, V, E).astype(np.int32)
    w = None if wb == 0 else rng.integers(0, 1 << 30, E).astype(np.int32)
    w = w.astype(np.float64) if wb == 8 else w
    d = lambda a: None if a is None else torch.from_numpy(a).cuda()

    def ref(key, val, x):
        o = np.argsort(key, kind="stable")
        rp = np.concatenate([[0], np.cumsum(np.bincount(key, minlength=V))]).astype(np.int32)
        return rp, val[o], None if x is None else x[o], key[o]

    rp, col, wo = gb.csr_from_edges(V, d(src), d(dst), d(w))
    rrp, rcol, rw, rrow = ref(src, dst, w)
    assert np.array_equal(rp.cpu().numpy(), rrp)
    assert np.array_equal(col.cpu().numpy(), rcol)
    assert w is None or np.array_equal(wo.cpu().numpy(), rw)
    trp, tcol, tw = gb.csr_transpose(rp, col, wo)
    trrp, trcol, trw, _ = ref(rcol, rrow, rw)
    assert np.array_equal(trp.cpu().numpy(), trrp)
    assert np.array_equal(tcol.cpu().numpy(), trcol)
    assert w is None or np.array_equal(tw.cpu().numpy(), trw)


@pytest.mark.parametrize("passes_V", [100, 1 << 20, 1 << 23])
def test_bad_endpoint_leaves_outputs(gpu, passes_V):
    """An endpoint outside [0, V) is refused and nothing is written."""
    gb = gpu
    import ctypes as C
    import torch
    E = 20000
    src = torch.arange(E, dtype=torch.int32, device="cuda") % passes_V
    dst = src.clone()
    dst[E - 1] = -1
    rp = torch.full((passes_V + 1,), -7, dtype=torch.int32, device="cuda")
    col = torch.full((E,), -7, dtype=torch.int32, device="cuda")
    st = gb.lib().gb_csr_from_edges(passes_V, E, src.data_ptr(), dst.data_ptr(), None, 0,
                                    rp.data_ptr(), col.data_ptr(), None, None)
    assert st == 1
    assert bool((rp == -7).all()) and bool((col == -7).all())
