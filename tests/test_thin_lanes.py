"""The rule for the lanes per wave of small FP32 batches in a host build (cpp/thin_lanes_check.cpp), and on
the GPU that the grid a caller chooses changes no ray of a small batch."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from oracle import oracle_py as O
from sirius_amd import abi

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"),
                    reason="needs g++ and the HIP headers")
def test_rule(tmp_path):
    exe = str(tmp_path / "thin_lanes_check")
    b = subprocess.run(["g++", "-std=c++17", "-O2", "-I/opt/rocm/include", "-D__HIP_PLATFORM_AMD__",
                        os.path.join(HERE, "cpp", "thin_lanes_check.cpp"), "-o", exe], capture_output=True, text=True,
                       timeout=300)
    assert b.returncode == 0, b.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("scene", ["disk", "wormhole"])
@pytest.mark.parametrize("block,blocks", [(64, 1), (64, 3), (256, 1), (256, 2)])
def test_grids(acc, scene, block, blocks):
    m, r, emission = ((abi.metric_ks(1.0, 0.7), 40.0, abi.EMISSION_THIN_DISK) if scene == "disk" else
                      (abi.metric_mt(1.0), 10.0, abi.EMISSION_NONE))
    o = O.default_opts(abi.PRECISION_FP32_ESCALATE)
    o.emission, o.n_bins = emission, 4
    cam = abi.camera(r, 70.0, 40.0, 131, 61, disk=(0.0, 20.0), phi_deg=33.0, yaw=0.1)
    print(f"[case] thin lanes {scene} {block}/{blocks}", flush=True)
    own, _ = acc.trace_batch([cam], [m], o)
    o.block_size, o.blocks_per_cu = block, blocks
    got, _ = acc.trace_batch([cam], [m], o)
    for k in ("cls", "flags", "theta", "phi", "lam", "disk_r", "redshift", "steps", "intensity"):
        assert np.array_equal(getattr(got, k), getattr(own, k)), k
