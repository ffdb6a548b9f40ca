"""Event location on a step's cubic interpolant (FP64 and FP32 symplectic) in a host build against bisection of the same interpolant
(cpp/event_locate_check.cpp states the cases and the bar)."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"),
                    reason="needs g++ and the HIP headers")
def test_event_locate(tmp_path):
    exe = str(tmp_path / "event_locate_check")
    b = subprocess.run(["g++", "-std=c++17", "-O2", "-I/opt/rocm/include", "-D__HIP_PLATFORM_AMD__",
                        os.path.join(HERE, "cpp", "event_locate_check.cpp"), "-o", exe], capture_output=True, text=True,
                       timeout=300)
    assert b.returncode == 0, b.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout
