"""Ray bundles run on a pair of lanes per ray: batches of one ray, of one pair short of a wave (31), a
whole wave (32), one more, and several cameras. Every ray's class is the trace's under the same
options away from the critical curve, and a sub-batch gives the same bits as the whole. The
Jacobian agrees with differences of FP64 traces through (u +- 1/8, v +- 1/8) of each pixel to 1e-2
of its norm: 4 M or more from the critical curve the lens map's second derivative per pixel is a
few per cent of its first, which central differences over a quarter pixel reduce to under 1e-3."""
import numpy as np
import pytest

from oracle import oracle_py as O
from sirius_amd import abi

pytestmark = pytest.mark.gpu


def _cam(w, h, phi=33.0):
    return abi.camera(40.0, 70.0, 40.0, w, h, disk=(0.0, 20.0), phi_deg=phi, yaw=0.1)


def _opts():
    o = O.default_opts(abi.PRECISION_FP64)
    o.rtol, o.atol = 1e-10, 1e-12
    return o


@pytest.mark.parametrize("w,h", [(1, 1), (31, 1), (8, 4), (11, 3), (40, 9)])
def test_pairs(acc, w, h):
    m, cam, o = abi.metric_ks(1.0, 0.7), _cam(w, h), _opts()
    print(f"[case] bundle pairs {w}x{h}", flush=True)
    out = acc.trace_bundle([cam], [m], o)
    rays, _ = acc.trace_batch([cam], [m], o)
    far = np.array([abs(O.critical_distance(cam, m, i % w, i // w)) > 0.5 for i in range(w * h)])
    assert np.array_equal(out["cls"][far], rays.cls[far])
    assert np.all(out["flags"][rays.cls == abi.RAY_CAPTURED] & 1)
    # several cameras in one batch: each camera's rays are its own batch's, bit for bit
    both = acc.trace_bundle([cam, _cam(w, h, 80.0)], [m], o)
    other = acc.trace_bundle([_cam(w, h, 80.0)], [m], o)
    n = w * h
    for k in ("cls", "flags", "jac", "beam"):
        assert np.array_equal(both[k][..., :n], out[k]) and np.array_equal(both[k][..., n:], other[k]), k


def test_jacobian_by_differences(acc):
    """Columns of the Jacobian: images of the same camera at 4 times the resolution hold the traces
    through (u +- 1/8, v +- 1/8) of each pixel."""
    w, h = 24, 14
    m, o = abi.metric_ks(1.0, 0.7), _opts()
    print("[case] bundle jacobian by differences", flush=True)
    out = acc.trace_bundle([_cam(w, h)], [m], o)
    fine, _ = acc.trace_batch([_cam(4 * w, 4 * h)], [m], o, with_state=True)
    cls = fine.cls.reshape(4 * h, 4 * w)
    d = np.array([abs(O.critical_distance(_cam(w, h), m, i % w, i // w)) for i in range(w * h)]).reshape(h, w)
    X = fine.state[:, 1:3].reshape(4 * h, 4 * w, 2)
    checked = 0
    for y in range(h):
        for x in range(w):
            q = cls[4 * y + 1:4 * y + 3, 4 * x + 1:4 * x + 3]
            if d[y, x] < 4.0 or not (q == abi.RAY_DISK).all() or out["cls"][y * w + x] != abi.RAY_DISK:
                continue
            P = X[4 * y + 1:4 * y + 3, 4 * x + 1:4 * x + 3]
            du = (P[:, 1] - P[:, 0]).mean(0) / 0.25
            dv = (P[1] - P[0]).mean(0) / 0.25
            want = np.array([du[0], dv[0], du[1], dv[1]])
            got = out["jac"][:, y * w + x]
            assert np.linalg.norm(got - want) < 1e-2 * np.linalg.norm(want)
            checked += 1
    assert checked > 20
