"""Results for host memory of up to 1 MiB travel in one block with the statistics, larger ones array by
array: both hold the device arrays' bytes. One ray (every array shorter than a 16-byte word or with a
tail), odd counts, counts whose arrays just fit and just do not (132 bytes per ray with the state and 4
bins), and larger ones; trace, fetch and bundles."""
import numpy as np
import pytest

from oracle import oracle_py as O
from sirius_amd import abi

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 5001, 7900, 9500, 20011])
def test_small_results(acc, n):
    m, cam = abi.metric_ks(1.0, 0.7), abi.camera(40.0, 70.0, 40.0, n, 1, disk=(0.0, 20.0))
    o = O.default_opts(abi.PRECISION_FP32_ESCALATE)
    o.n_bins = 4
    print(f"[case] results of {n} rays", flush=True)
    dt = dict(cls=torch.uint8, flags=torch.uint8, steps=torch.int32, state=torch.float64)
    shape = dict(intensity=(4, n), state=(n, 8))
    names = dict(cls="cls", flags="flags", theta="theta", phi="phi", lam="lambda_", disk_r="disk_r", redshift="redshift",
                 steps="steps", intensity="intensity", state="state")
    dev = {k: torch.zeros(shape.get(k, (n,)), dtype=dt.get(k, torch.float32), device="cuda") for k in names}
    torch.cuda.synchronize()
    ro = abi.RayOutput(on_device=1, **{names[k]: t.data_ptr() for k, t in dev.items()})
    _, sd = acc.trace_batch([cam], [m], o, device_out=ro)
    host, sh = acc.trace_batch([cam], [m], o, with_state=True)
    fetched = acc.fetch_results(with_state=True)
    for k, t in dev.items():
        for got in (getattr(host, k), getattr(fetched, k)):
            assert np.ascontiguousarray(got).tobytes() == t.cpu().numpy().tobytes(), k
    for k in ("rays", "steps_accepted", "steps_rejected", "steps_bulk", "null_drift_max", "null_drift_median"):
        assert sd[k] == sh[k], k
    res = acc.trace_bundle([cam], [m], o)
    assert np.array_equal(res["cls"], acc.trace_bundle([cam], [m], o)["cls"]) and np.isfinite(res["jac"]).all()
