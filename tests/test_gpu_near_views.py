"""FP32 Kerr-Schild views narrower than the shadow, which are traced in rows, against the same cameras in a
batch of more than 1.5 M rays, which is traced in squares: every ray keeps its bits. Views wider than the
shadow beside them."""
import numpy as np
import pytest

from oracle import oracle_py as O
from sirius_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lam", [0.0, 1e-5])
@pytest.mark.parametrize("r,fov", [(6.0, 20.0), (10.0, 25.0), (15.0, 38.2), (15.0, 38.6), (15.0, 90.0)])
def test_rows_and_squares(acc, r, fov, lam):
    o = O.default_opts(abi.PRECISION_FP32_ESCALATE)
    o.emission, o.n_bins = abi.EMISSION_NONE, 0
    m, w, h = abi.metric_ks(1.0, 0.9, 0.1, lam), 331, 211  # above the thin waves' 65,536 rays
    cam, tiny, big = (abi.camera(r, 75.0, fov, a, b, phi_deg=p) for a, b, p in ((w, h, 33.0), (1, 1, 80.0), (1500, 1000, 80.0)))
    print(f"[case] near view r {r} fov {fov} lambda {lam}", flush=True)
    small, _ = acc.trace_batch([cam, tiny], [m], o)
    large, _ = acc.trace_batch([cam, big], [m], o)
    for k in ("cls", "flags", "theta", "phi", "lam", "redshift", "steps"):
        assert np.array_equal(getattr(small, k)[:w * h], getattr(large, k)[:w * h]), k
