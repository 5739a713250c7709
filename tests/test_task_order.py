"""CPU test of the order of a tile's block tasks in the host tile builder
(tests/cpp/task_order_check.cpp; the device builder's tiles are its bytes)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "finetools.jl_amd", "csrc")


def test_task_order(tmp_path):
    hipcc = shutil.which("hipcc") or ("/opt/rocm/bin/hipcc" if os.path.exists("/opt/rocm/bin/hipcc") else None)
    if hipcc is None:
        pytest.skip("no hipcc")
    exe = str(tmp_path / "task_order_check")
    srcs = [os.path.join(ROOT, "tests", "cpp", "task_order_check.cpp")] + \
        [os.path.join(CSRC, f) for f in ("tiles.cpp", "meshgen.cpp", "pool.cpp")]
    subprocess.check_call([hipcc, "-O2", "-std=c++17", "-I", CSRC, "-I", os.path.join(ROOT, "include")] + srcs +
                          ["-o", exe, "-lpthread"], cwd=str(tmp_path))
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stderr[-4000:]
    assert out.stdout.strip().splitlines()[-1] == "ok"
