"""Kerr-Schild batches whose cameras all have Lambda = 0 run kernels without the Lambda terms; one
camera with Lambda in the batch and every ray runs the general ones. Both evaluate the same equations
in FP64, so 0.5 M or more from the critical curve a ray ends alike in both: rounding (1e-16 a step, some
hundred steps, stretched less than a thousandfold by the lensing there) stays under 1e-9. Batches of one
ray, of a wave less one, and of odd sizes, for the trace, the symplectic integrator and the ray bundles."""
import numpy as np
import pytest

from oracle import oracle_py as O
from sirius_amd import abi

pytestmark = pytest.mark.gpu


def _cam(w, h):
    return abi.camera(40.0, 70.0, 40.0, w, h, disk=(0.0, 20.0), phi_deg=33.0, yaw=0.1)


def _far(cam, m, w, h):
    return np.array([abs(O.critical_distance(cam, m, i % w, i // w)) > 0.5 for i in range(w * h)])


def _close(a, b, tol, what):
    a, b = np.asarray(a, np.float64), np.asarray(b, np.float64)
    assert np.all(np.abs(a - b) <= tol * np.maximum(1.0, np.abs(b))), (what, np.abs(a - b).max())


@pytest.mark.parametrize("emission,symplectic", [(abi.EMISSION_THIN_DISK, False), (abi.EMISSION_NONE, False),
                                                 (abi.EMISSION_VOLUMETRIC, False), (abi.EMISSION_THIN_DISK, True),
                                                 (abi.EMISSION_NONE, True)])
@pytest.mark.parametrize("w,h", [(1, 1), (9, 7), (13, 5)])
@pytest.mark.parametrize("a,q", [(0.0, 0.0), (0.7, 0.4), (0.998, 0.0)])
def test_flat_and_general_trace(acc, w, h, a, q, emission, symplectic):
    m, ml, cam = abi.metric_ks(1.0, a, q), abi.metric_ks(1.0, a, q, 1e-4), _cam(w, h)
    o = O.default_opts(abi.PRECISION_FP64)
    o.emission, o.n_bins = emission, 4
    if symplectic:
        o.integrator = abi.INTEGRATOR_SYMPLECTIC
    print(f"[case] flat {w}x{h} a {a} q {q} emission {emission} symplectic {symplectic}", flush=True)
    flat, _ = acc.trace_batch([cam], [m], o, with_state=True)
    gen, _ = acc.trace_batch([cam, cam], [m, ml], o, with_state=True)
    n, far = w * h, _far(cam, m, w, h)
    assert np.array_equal(flat.cls[far], gen.cls[:n][far])
    same = far & (flat.steps == gen.steps[:n])
    assert same.sum() >= 0.9 * far.sum()  # a rounding can move an accept or reject, seldom
    out = same & (flat.cls != abi.RAY_CAPTURED)  # at the horizon dt/dlambda diverges
    _close(flat.state[out], gen.state[:n][out], 1e-9, "state")


@pytest.mark.parametrize("w,h", [(1, 1), (31, 1), (11, 3)])
@pytest.mark.parametrize("a,q", [(0.0, 0.0), (0.7, 0.4)])
def test_flat_and_general_bundle(acc, w, h, a, q):
    m, ml, cam = abi.metric_ks(1.0, a, q), abi.metric_ks(1.0, a, q, 1e-4), _cam(w, h)
    o = O.default_opts(abi.PRECISION_FP64)
    print(f"[case] flat bundle {w}x{h} a {a} q {q}", flush=True)
    flat = acc.trace_bundle([cam], [m], o)
    gen = acc.trace_bundle([cam, cam], [m, ml], o)
    n, far = w * h, _far(cam, m, w, h)
    assert np.array_equal(flat["cls"][far], gen["cls"][:n][far])
    out = far & (flat["cls"] != abi.RAY_CAPTURED)
    # float32 results: 2^-24 of the largest, and the tangents' rounding
    scale = np.abs(gen["jac"][:, :n]).max(0)[out]
    assert np.all(np.abs(flat["jac"] - gen["jac"][:, :n])[:, out] <= 1e-6 * scale)
