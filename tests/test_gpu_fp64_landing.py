"""FP64 landings: a wave lands its ended rays together before it takes new ones. Batches of one ray, one
lane short of a wave, a whole wave, one more and several waves, under the static grid and under
persistent queues that refill a lane, a quarter wave or a whole wave at a time, against the oracle
(both integrate at rtol 1e-8; away from the critical curve their directions, radii and intensities
agree to 1e-6) and bit for bit against each other (schedules never change results)."""
import numpy as np
import pytest

from oracle import oracle_py as O
from sirius_amd import abi

pytestmark = pytest.mark.gpu

FIELDS = ("cls", "flags", "theta", "phi", "lam", "disk_r", "redshift", "steps", "intensity")


@pytest.mark.parametrize("emission", [abi.EMISSION_THIN_DISK, abi.EMISSION_NONE])
@pytest.mark.parametrize("w,h", [(1, 1), (9, 7), (8, 8), (13, 5), (50, 3)])
def test_landings_under_every_schedule(acc, w, h, emission):
    m = abi.metric_ks(1.0, 0.7)
    cam = abi.camera(40.0, 70.0, 40.0, w, h, disk=(0.0, 20.0), phi_deg=33.0, yaw=0.1)
    o = O.default_opts(abi.PRECISION_FP64)
    o.emission, o.n_bins = emission, 4
    print(f"[case] fp64 landing {w}x{h} emission {emission}", flush=True)
    grid, st = acc.trace_batch([cam], [m], o)
    ref, _ = O.trace([cam], [m], o)
    band = np.array([abs(O.critical_distance(cam, m, i % w, i // w)) > 0.5 for i in range(w * h)])
    assert np.array_equal(grid.cls[band], ref.cls[band])
    esc = band & (ref.cls == abi.RAY_ESCAPED)
    assert (np.abs(grid.direction()[esc] - ref.direction()[esc]).max() if esc.any() else 0) < 1e-6
    hit = band & (ref.cls == abi.RAY_DISK)
    for k in ("disk_r", "redshift", "intensity"):
        a, b = getattr(grid, k)[..., hit], getattr(ref, k)[..., hit]
        assert np.all(np.abs(a - b) <= 1e-6 * np.abs(b).max() if b.size else True)
    o.schedule = abi.SCHEDULE_PERSISTENT
    for block, refill in ((64, 1), (256, 16), (128, 64)):
        o.block_size, o.refill_min = block, refill
        other, _ = acc.trace_batch([cam], [m], o)
        for k in FIELDS:
            assert np.array_equal(getattr(grid, k), getattr(other, k)), (k, block, refill)
