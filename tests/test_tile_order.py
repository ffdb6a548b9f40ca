"""The order in which whole batches are traced: the position-to-pixel map in a host build
(cpp/tile_order_check.cpp), and on the GPU that the order changes no ray. Batches above 65,536 FP64
Kerr-Schild rays trace the rays near the critical curve first, from lists: a camera's rays in such a
batch hold the bits they have in a smaller one, which is traced without lists. Ragged sides."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from oracle import oracle_py as O
from sirius_amd import abi

HERE = os.path.dirname(os.path.abspath(__file__))
FIELDS = ("cls", "flags", "theta", "phi", "lam", "disk_r", "redshift", "steps", "intensity")


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"),
                    reason="needs g++ and the HIP headers")
def test_position_to_pixel(tmp_path):
    exe = str(tmp_path / "tile_order_check")
    b = subprocess.run(["g++", "-std=c++17", "-O2", "-I/opt/rocm/include", "-D__HIP_PLATFORM_AMD__",
                        os.path.join(HERE, "cpp", "tile_order_check.cpp"), "-o", exe], capture_output=True, text=True,
                       timeout=300)
    assert b.returncode == 0, b.stderr[-4000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.strip().endswith("OK"), r.stdout


@pytest.mark.gpu
@pytest.mark.parametrize("emission", [abi.EMISSION_THIN_DISK, abi.EMISSION_NONE, abi.EMISSION_VOLUMETRIC])
def test_lists_change_no_ray(acc, emission):
    w, h = 211, 163  # 34,393 rays: two cameras are above the line, one with a single pixel is below it
    m = abi.metric_ks(1.0, 0.7)
    cam, other, tiny = (abi.camera(40.0, 70.0, 40.0, a, b, disk=(0.0, 20.0), phi_deg=p) for a, b, p in
                        ((w, h, 10.0), (w, h, 75.0), (1, 1, 75.0)))
    o = O.default_opts(abi.PRECISION_FP64)
    o.emission, o.n_bins, o.rtol, o.atol = emission, 4, 1e-6, 1e-8
    n = w * h
    print(f"[case] fp64 lists {w}x{h} emission {emission}", flush=True)
    small, _ = acc.trace_batch([cam, tiny], [m], o)
    for schedule in (abi.SCHEDULE_GRID, abi.SCHEDULE_PERSISTENT):
        o.schedule = schedule
        large, _ = acc.trace_batch([cam, other], [m], o)
        for k in FIELDS:
            assert np.array_equal(getattr(large, k)[..., :n], getattr(small, k)[..., :n]), (k, schedule)
    last, _ = acc.trace_batch([tiny, other], [m], o)
    for k in FIELDS:
        assert np.array_equal(getattr(large, k)[..., n:], getattr(last, k)[..., 1:]), k


@pytest.mark.gpu
def test_lists_change_no_bundle(acc):
    w, h = 181, 173  # 31,313 bundles: one camera is below the line of 32,768, two are above it
    m = abi.metric_ks(1.0, 0.7)
    cams = [abi.camera(40.0, 70.0, 40.0, w, h, disk=(0.0, 20.0), phi_deg=p) for p in (10.0, 75.0)]
    o = O.default_opts(abi.PRECISION_FP64)
    o.rtol, o.atol = 1e-6, 1e-8
    print(f"[case] bundle lists {w}x{h}", flush=True)
    both, n = acc.trace_bundle(cams, [m], o), w * h
    for i, cam in enumerate(cams):
        one = acc.trace_bundle([cam], [m], o)
        for k in ("cls", "flags", "jac", "beam"):
            assert np.array_equal(both[k][..., i * n:(i + 1) * n], one[k]), (k, i)
