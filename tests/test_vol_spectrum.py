"""The volumetric spectrum of the FP32 path: its exponentials in a host build against FP64
(cpp/exp_parts_check.cpp states the bars), and intensities with one bin, with as many as accumulate in
registers, and with one more, over narrow and wide frequency ranges, against the FP64 oracle for rays
outside the shadow at the FP32 path's tolerance of 2e-3 of a ray's brightest bin."""
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
def test_exponentials(tmp_path):
    exe = str(tmp_path / "exp_parts_check")
    b = subprocess.run(["g++", "-std=c++17", "-O2", "-I/opt/rocm/include", "-D__HIP_PLATFORM_AMD__",
                        os.path.join(HERE, "cpp", "exp_parts_check.cpp"), "-o", exe], capture_output=True, text=True,
                       timeout=300)
    assert b.returncode == 0, b.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    print(r.stdout)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("x_min,x_max", [(0.1, 10.0), (1e-4, 300.0)])
@pytest.mark.parametrize("n_bins", [1, 8, 9])
def test_bins(acc, n_bins, x_min, x_max):
    w, h = 13, 9
    m, cam = abi.metric_ks(1.0, 0.6), abi.camera(30.0, 75.0, 45.0, w, h, disk=(0.0, 20.0), phi_deg=20.0)
    print(f"[case] volumetric spectrum {n_bins} bins {x_min}..{x_max}", flush=True)
    o, r = O.default_opts(abi.PRECISION_FP32_ESCALATE), O.default_opts(abi.PRECISION_FP64)
    for q in (o, r):
        q.emission, q.n_bins, q.x_min, q.x_max = abi.EMISSION_VOLUMETRIC, n_bins, x_min, x_max
    got, _ = acc.trace_batch([cam], [m], o)
    ref, _ = O.trace([cam], [m], r)
    a, b = np.asarray(got.intensity, np.float64), np.asarray(ref.intensity, np.float64)
    assert np.all(np.isfinite(a)) and np.all(a >= 0)
    out = np.array([O.critical_distance(cam, m, i % w, i // w) > 0.5 for i in range(w * h)])
    sel = out & (b.max(0) > 0)
    assert sel.sum() > 20
    top = b[:, sel].max(0)
    assert np.all(np.abs(a - b)[:, sel].max(0) <= 2e-3 * np.maximum(top, 1e-2 * np.median(top)))
