"""The library's Makefile: the flags that the kernels are written for reach every HIP compile line
whatever HIPFLAGS the caller sets, a change of the Makefile rebuilds every object, and
msm_quad.cuh does not compile for the device without them."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "..", "snarkrs_amd", "csrc")
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


def _dry_run(obj, *args):
    r = subprocess.run(["make", "-n", "-C", CSRC, f"OBJ={obj}", f"OUT={obj}", *args],
                       capture_output=True, text=True, check=True, timeout=60)
    return [line for line in r.stdout.splitlines() if " -c " in line]


def _sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp")))


def test_flags_survive_the_caller(tmp_path):
    lines = [x for x in _dry_run(tmp_path, "HIPFLAGS=-O2") if ".hip" in x]
    assert len(lines) == sum(f.endswith(".hip") for f in _sources())
    for line in lines:
        assert "-amdgpu-dpp-combine=0" in line and "-packed-fp32-ops" in line, line
        assert "--offload-arch=gfx950" in line and " -O2 " in line, line


def test_changed_flags_rebuild(tmp_path):
    for f in _sources():
        (tmp_path / (os.path.splitext(f)[0] + ".o")).touch()
    assert _dry_run(tmp_path) == []
    assert len(_dry_run(tmp_path, "-W", "Makefile")) == len(_sources())


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc is not installed")
def test_quad_needs_the_define(tmp_path):
    src = tmp_path / "quad.hip"
    src.write_text(f'#include "{CSRC}/msm_quad.cuh"\n')
    cmd = [HIPCC, "--offload-arch=gfx950", "-std=c++17", "-fsyntax-only", str(src)]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode != 0 and "amdgpu-dpp-combine=0" in r.stderr
    subprocess.run(cmd + ["-DG16_NO_DPP_COMBINE"], check=True, capture_output=True, timeout=300)
