"""Merged buckets: the host model of both engines' loops (CPU), and the engines
against Dijkstra and against single buckets (GPU)."""
import os
import shutil
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "graphbench_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def test_span_model_matches_dijkstra(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    exe = tmp_path / "spans"
    src = os.path.join(HERE, "models", "spans_ctl_model.hip")
    subprocess.run([HIPCC, "-O2", "-std=c++17", "--offload-arch=gfx950", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops", "-I", CSRC, "-o", str(exe),
                    src], check=True, capture_output=True)
    r = subprocess.run([str(exe), "400"], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("nsrc,scan", [(1, "0"), (3, "0"), (3, "1"), (40, "0"), (40, "1")])
@pytest.mark.parametrize("shape", ["path", "random", "hub"])
def test_engines_over_ranges(gpu, monkeypatch, shape, nsrc, scan):
    """Narrow buckets that merge (a path: one vertex each; a random graph; a hub
    whose chunks fill a phase), every engine form; counters by the caller's
    width on the path, a tree."""
    import oracle
    gb = gpu
    monkeypatch.setenv("GB_MSSSP_SCAN", scan)  # also keeps the one-workgroup form out
    rng = np.random.default_rng(nsrc)
    V = 4000 if shape == "path" else 20000
    if shape == "path":
        src, dst = np.arange(V - 1), np.arange(1, V)
    elif shape == "random":
        src, dst = rng.integers(0, V, 5 * V), rng.integers(0, V, 5 * V)
    else:
        src = np.concatenate([np.zeros(V - 1, np.int64), np.arange(1, V)])
        dst = np.concatenate([np.arange(1, V), np.arange(1, V) % (V - 1) + 1])
    w = rng.integers(1, 256, len(src)).astype(np.uint32)
    h = gb.HostCSR.from_edges(V, src, dst, w)
    g = gb.Graph.from_host(h, need_reverse=False)
    srcs = rng.integers(0, V, nsrc).astype(np.int32)
    srcs[0] = 0
    for delta in (1, 7):
        d, st = gb.sssp(g, srcs, delta=delta, stats=True)
        d = gb.u32(d)
        for i in (0, nsrc // 2, nsrc - 1):
            assert np.array_equal(d[i], oracle.dijkstra(h.row_ptr, h.col, h.w, int(srcs[i])))
        monkeypatch.setenv("GB_SSSP_SPANS", "0")
        d1, st1 = gb.sssp(g, srcs, delta=delta, stats=True)
        monkeypatch.delenv("GB_SSSP_SPANS")
        assert np.array_equal(d, gb.u32(d1))
        assert st["phases"] < st1["phases"]
        assert (st["reached"], st["traversed"]) == (st1["reached"], st1["traversed"])
        if shape == "path":
            for k in ("relax_edges", "improved_near", "improved_far"):
                assert st[k] == st1[k], k
