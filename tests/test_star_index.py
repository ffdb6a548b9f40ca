"""The celestial spheres' star index on the host, through the library's own function
(cpp/star_index_check.cpp states the cases): no star whose cut reaches a direction is missing from that
direction's cell, lists are in catalogue order, and catalogues whose lists would be long have none."""
import os
import shutil
import subprocess

import pytest

from sirius_amd import accelerator

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.dirname(accelerator.LIB_PATH)


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.exists(accelerator.LIB_PATH),
                    reason="needs g++ and the built library")
def test_star_index(tmp_path):
    exe = str(tmp_path / "star_index_check")
    b = subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", os.path.join(HERE, "cpp", "star_index_check.cpp"),
                        "-L", LIB, "-lsirius_hip", "-Wl,-rpath," + LIB, "-L/opt/rocm/lib", "-Wl,-rpath-link,/opt/rocm/lib",
                        "-Wl,-rpath,/opt/rocm/lib", "-o", exe], capture_output=True, text=True, timeout=300)
    assert b.returncode == 0, b.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), (r.returncode, r.stdout)
    print(r.stdout)
