"""CSR builds whose outputs take the place of their keys, at one, two and three
digit passes, against numpy's stable sort."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

V_OF = {1: 2048, 2: 70000, 3: (1 << 22) + 1}


def _ref(key, val, w, V):
    o = np.argsort(key, kind="stable")
    return np.concatenate([[0], np.cumsum(np.bincount(key, minlength=V))]), val[o], w[o], key[o]


def _same(t, a):
    return np.array_equal(t.cpu().numpy(), a)


@pytest.mark.parametrize("passes", [1, 2, 3])
@pytest.mark.parametrize("E", [5000, 300007])
def test_outputs_over_keys(gpu, passes, E):
    gb = gpu
    import torch
    V = V_OF[passes]
    rng = np.random.default_rng(passes + E)
    src = rng.integers(0, V, E).astype(np.int32)
    dst = rng.integers(0, V, E).astype(np.int32)
    w = rng.integers(0, 1 << 30, E).astype(np.int32)
    d = lambda a: torch.from_numpy(a.copy()).cuda()
    p = lambda t: C.c_void_p(t.data_ptr())
    rp_ref, col_ref, w_ref, row_ref = _ref(src, dst, w, V)
    L = gb.lib()
    rp = torch.empty(V + 1, dtype=torch.int32, device="cuda")
    # columns over the sources, then weights over the sources
    a, b, x, out = d(src), d(dst), d(w), torch.empty(E, dtype=torch.int32, device="cuda")
    assert L.gb_csr_from_edges(V, E, p(a), p(b), p(x), 4, p(rp), p(a), p(out), gb._stream()) == 0
    assert _same(rp, rp_ref) and _same(a, col_ref) and _same(out, w_ref)
    a = d(src)
    assert L.gb_csr_from_edges(V, E, p(a), p(b), p(x), 4, p(rp), p(out), p(a), gb._stream()) == 0
    assert _same(rp, rp_ref) and _same(out, col_ref) and _same(a, w_ref)
    # a transpose in place: columns and offsets over the input's
    t_rp, t_col, t_w, _ = _ref(col_ref, row_ref, w_ref, V)
    col, ww = d(col_ref), d(w_ref)
    assert L.gb_csr_transpose(V, E, p(rp), p(col), p(ww), 4, p(rp), p(col), p(out),
                              gb._stream()) == 0
    assert _same(rp, t_rp) and _same(col, t_col) and _same(out, t_w)
