"""The tiles of a run of steps agree on whether it is kept (sem2dpack_amd/csrc/sem2d_commit.hpp):
every order of the accesses of up to four tiles, on the CPU (tests/native/run_commit_check.cpp)."""
import os
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "sem2dpack_amd", "csrc")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_tiles_decide_alike():
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "run_commit_check")
        subprocess.run([HIPCC, "-O2", "-std=c++17", "--offload-arch=gfx950", "-I", CSRC, "-o", exe,
                        os.path.join(HERE, "native", "run_commit_check.cpp")], check=True, cwd=tmp)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    states, wrong = (int(x) for x in r.stdout.split())
    assert states > 10_000
    assert wrong == 0 and r.returncode == 0
