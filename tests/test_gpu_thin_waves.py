"""FP32 batches of fewer rays than the chip has lanes run with some of each wave's lanes: a camera's rays in a
small batch hold the bits they have in a batch large enough for whole waves. One ray, a few, odd counts,
the last sizes below and above the line of 65,536 rays; Kerr disk and sky, wormhole and warp bubble; and
with a caller's block size and blocks per CU."""
import numpy as np
import pytest

from oracle import oracle_py as O
from sirius_amd import abi

pytestmark = pytest.mark.gpu
FIELDS = ("cls", "flags", "theta", "phi", "lam", "disk_r", "redshift", "steps", "intensity")
SCENES = {
    "disk": (abi.metric_ks(1.0, 0.7), 40.0, abi.EMISSION_THIN_DISK),
    "sky": (abi.metric_ks(1.0, 0.7), 40.0, abi.EMISSION_NONE),
    "wormhole": (abi.metric_mt(1.0), 10.0, abi.EMISSION_NONE),
    "warp": (abi.metric_warp(0.5, 1.0, 8.0), 10.0, abi.EMISSION_NONE),
}


def _cam(w, h, r, phi=33.0):
    return abi.camera(r, 70.0, 40.0, w, h, disk=(0.0, 20.0), phi_deg=phi, yaw=0.1)


@pytest.mark.parametrize("scene", SCENES)
@pytest.mark.parametrize("w,h", [(1, 1), (5, 3), (63, 1), (65, 17), (131, 90), (251, 260)])
def test_thin_waves(acc, w, h, scene):
    m, r, emission = SCENES[scene]
    o = O.default_opts(abi.PRECISION_FP32_ESCALATE)
    o.emission, o.n_bins = emission, 4
    cam, tiny, big = _cam(w, h, r), _cam(1, 1, r, 80.0), _cam(300, 240, r, 80.0)
    n = w * h
    print(f"[case] thin waves {scene} {w}x{h}", flush=True)
    # two cameras either way, so that both batches run the same kernel
    thin, _ = acc.trace_batch([cam, tiny], [m], o)
    whole, _ = acc.trace_batch([cam, big], [m], o)
    for k in FIELDS:
        assert np.array_equal(getattr(thin, k)[..., :n], getattr(whole, k)[..., :n]), k
    o.block_size, o.blocks_per_cu, o.refill_min = 64, 2, 3
    other, _ = acc.trace_batch([cam, tiny], [m], o)
    for k in FIELDS:
        assert np.array_equal(getattr(thin, k), getattr(other, k)), k
