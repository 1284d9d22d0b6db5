"""The host's pass over an MSM's reduction rows (runtime_impl.h msm_combine) never waits for a
helper thread that has not begun: with a pool that starts none in time, refuses every task, or
runs them all, the sum is the same point and the call returns. Built host-only with hipcc."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
pytestmark = pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not installed")


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = tmp_path_factory.mktemp("combine") / "msm_combine"
    subprocess.run([HIPCC, "-O1", "-std=c++17", "--cuda-host-only", "-x", "hip",
                    os.path.join(HERE, "host", "msm_combine.cpp"), "-o", str(out), "-lpthread"],
                   check=True, capture_output=True, timeout=600)
    return str(out)


@pytest.mark.parametrize("pool", ["run", "late", "throw"])
def test_combine(exe, pool):
    r = subprocess.run([exe, pool], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
