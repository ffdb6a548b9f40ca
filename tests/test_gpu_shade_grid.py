"""The shading kernel's block-strided grid: every ray of a frame gets its radiance, for frames of one
ray, of a partial block and of more rays than the grid has lanes (2048 blocks of 256), where the
last rays belong to the second stride. The radiance is compared with the shading restatement
(oracle/oracle_shade.py) at its bar: relative 2e-5 per channel, floored at 1e-6 of the brightest
value (the two sides' exp and pow differ in the last bits)."""
import numpy as np
import pytest

from oracle import oracle_py as O
from oracle import oracle_shade as S
from sirius_amd import abi
from sirius_amd.accelerator import default_opts

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(1, 1), (19, 13), (1024, 513)])
def test_every_ray_is_shaded(acc, w, h):
    m = abi.metric_ks(1.0, 0.9)
    cam = abi.camera(50.0, 75.0, 20.0, w, h, disk=(0.0, 30.0), yaw=0.05)
    o = default_opts(abi.PRECISION_FP32_ESCALATE)
    acc.initialise(w, h)
    print(f"[case] shade {w}x{h}", flush=True)
    acc.launch(cam, m, o)
    fb = acc.getFrameBuffer().reshape(-1, 4)
    rays = acc.fetch_results(with_state=True)
    assert np.all(fb[:, 3] == 1.0)
    assert not fb[rays.cls == abi.RAY_CAPTURED, :3].any()
    dk = np.nonzero(rays.cls == abi.RAY_DISK)[0]
    dk = np.unique(np.concatenate([dk[:8], dk[:: max(1, len(dk) // 64)], dk[-64:]]))
    te = np.array([50000.0 * O.lib().oracle_disk_temperature_ratio(float(rays.disk_r[i]), m.a, O.lib().oracle_isco(0.9), 30.0)
                   for i in dk])
    k = np.array([O.rhs(m, rays.state[i, :4], rays.state[i, 4:])[0] for i in dk]).reshape(-1, 4)
    want = S.disk_radiance(te, rays.redshift[dk], np.abs(k[:, 3]) / np.linalg.norm(k[:, 1:], axis=1), 5.0)
    if not len(dk):  # the one ray of the 1 x 1 frame falls into the hole: black, checked above
        assert rays.cls.tolist() == [abi.RAY_CAPTURED]
        return
    assert want.max() > 0
    err = np.abs(fb[dk, :3] - want) / np.maximum(np.abs(want), 1e-6 * want.max())
    assert err.max() < 2e-5
