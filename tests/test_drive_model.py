"""The loop that launches phases ahead of the device, against a host model of
the device: records behind, level with and ahead of the host, phases reported
one by one or every third, a device that reports nothing."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.join(HERE, "..")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def test_drive_loop(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not available")
    exe = tmp_path / "drive"
    subprocess.run([HIPCC, "-O2", "-std=c++17", "--offload-arch=gfx950", "-Xclang",
                    "-target-feature", "-Xclang", "-packed-fp32-ops",
                    "-I", os.path.join(ROOT, "graphbench_amd", "csrc"),
                    "-I", os.path.join(ROOT, "include"), "-o", str(exe),
                    os.path.join(HERE, "models", "drive_model.hip")],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.startswith("ok"), r.stdout + r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("nsrc", [2, 40])
def test_scan_form_with_waiting_launches(gpu, nsrc):
    """The scan form from sources with and without out-edges, in a process whose
    launches wait for their kernels: its first state advance has run before the
    first phase is launched."""
    import subprocess as sp
    import sys
    code = (
        "import numpy as np, graphbench_amd as gb, oracle\n"
        "gb.init(0)\n"
        "h = gb.gen_rmat(12, 8, seed=5, weights='uniform', wlo=1, whi=255)\n"
        "g = gb.Graph.from_host(h, need_reverse=False)\n"
        "od = np.diff(h.row_ptr)\n"
        f"s = np.concatenate([np.argsort(od)[:1], np.argsort(od)[-{nsrc - 1}:]]).astype(np.int32)\n"
        "d = gb.u32(gb.sssp(g, s, delta=100))\n"
        "for i in range(len(s)):\n"
        "    assert np.array_equal(d[i], oracle.dijkstra(h.row_ptr, h.col, h.w, int(s[i])))\n"
        "d = gb.u32(gb.sssp(g, [int(s[0])] * 2, delta=100))\n"
        "assert (d[0] == oracle.dijkstra(h.row_ptr, h.col, h.w, int(s[0]))).all()\n"
        "print('same')\n")
    env = dict(os.environ, HIP_LAUNCH_BLOCKING="1", GB_MSSSP_SCAN="1", GB_MSSSP_TUNE="0")
    r = sp.run([sys.executable, "-c", code], capture_output=True, text=True, timeout=100,
               cwd=ROOT, env=env)
    assert r.returncode == 0 and "same" in r.stdout, r.stdout + r.stderr
