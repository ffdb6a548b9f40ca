"""The far end of the FP32 path's volumetric spectrum, for frequency ranges up to 1e12 times the disk's: a bin
whose intensity in the FP64 oracle is below 1e-38 of the ray's brightest (e^-x times x^3, x above 100) is
exactly 0, no bin rises again after that, and every bin is within the path's 2e-3 of the brightest
of the oracle's, for rays outside the shadow. With the spectra of up to 8 bins and with more."""
import numpy as np
import pytest

from oracle import oracle_py as O
from sirius_amd import abi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_bins", [4, 8, 9])
@pytest.mark.parametrize("x_max", [1e3, 1e6, 1e10, 1e12])
def test_tail(acc, x_max, n_bins):
    w, h = 13, 9
    m, cam = abi.metric_ks(1.0, 0.6), abi.camera(30.0, 75.0, 45.0, w, h, disk=(0.0, 20.0), phi_deg=20.0)
    print(f"[case] volumetric tail {n_bins} bins to {x_max}", flush=True)
    o, r = O.default_opts(abi.PRECISION_FP32_ESCALATE), O.default_opts(abi.PRECISION_FP64)
    for q in (o, r):
        q.emission, q.n_bins, q.x_min, q.x_max = abi.EMISSION_VOLUMETRIC, n_bins, 0.1, x_max
    got, _ = acc.trace_batch([cam], [m], o)
    ref, _ = O.trace([cam], [m], r)
    a, b = np.asarray(got.intensity, np.float64), np.asarray(ref.intensity, np.float64)
    out = np.array([O.critical_distance(cam, m, i % w, i // w) > 0.5 for i in range(w * h)])
    sel = out & (b.max(0) > 0)
    assert sel.sum() > 20
    a, b = a[:, sel], b[:, sel]
    top = b.max(0)
    assert np.all(np.isfinite(a)) and np.all(a >= 0)
    assert np.all(np.abs(a - b) <= 2e-3 * np.maximum(top, 1e-2 * np.median(top)))
    assert np.all(a[b < 1e-38 * top] == 0)
    assert (b < 1e-38 * top).any()
