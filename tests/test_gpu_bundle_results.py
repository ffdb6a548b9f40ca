"""Ray bundles delivered to host memory hold the device arrays' bytes, in one block with one wait up to 1 MiB (29
bytes a ray: 36,157 rays and their 16-byte padding) and array by array above: one ray, odd counts, and
counts on both sides of that size. And a caller may ask for some of the arrays only."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle_py as O
from sirius_amd import abi

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 5001, 36151, 36157, 36158, 50021])
def test_bundle_results(acc, n):
    m, cam = abi.metric_ks(1.0, 0.7), abi.camera(40.0, 70.0, 40.0, n, 1, disk=(0.0, 20.0))
    o = O.default_opts(abi.PRECISION_FP64)
    o.rtol, o.atol = 1e-6, 1e-8
    print(f"[case] bundle results of {n} rays", flush=True)
    shape = dict(cls=(n,), flags=(n,), jac=(4, n), beam=(3, n))
    dev = {k: torch.zeros(s, dtype=torch.uint8 if k in ("cls", "flags") else torch.float32, device="cuda") for k, s in shape.items()}
    torch.cuda.synchronize()

    def trace(**ptr):
        bo = abi.BundleOutput(**ptr)
        acc._check(acc._L.sirius_hip_trace_bundle(acc._h, C.byref(cam), 1, C.byref(m), 1, C.byref(o), C.byref(bo)))

    trace(on_device=1, **{k: t.data_ptr() for k, t in dev.items()})
    want = {k: t.cpu().numpy() for k, t in dev.items()}
    assert n == 1 or (want["jac"].any() and want["beam"].any())  # the one ray of n = 1 is captured
    host = acc.trace_bundle([cam], [m], o)
    for k in shape:
        assert np.ascontiguousarray(host[k]).tobytes() == want[k].tobytes(), k
    some = {k: np.zeros_like(want[k]) for k in ("flags", "beam")}
    trace(on_device=0, **{k: a.ctypes.data for k, a in some.items()})
    for k, a in some.items():
        assert a.tobytes() == want[k].tobytes(), k
