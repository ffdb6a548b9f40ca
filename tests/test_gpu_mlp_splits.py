"""Loss and gradient of the network for batches whose weight gradients are summed in several splits of the
samples (one split per 16 tiles of 32 samples, 32 splits at most): the smallest of two splits with a last
tile of one sample, two equal ones, an odd second one, five with a ragged last, and batches around the
largest number of splits. Against the network oracle with its operands rounded to BF16 where the device
rounds them: every layer's gradient to 2e-2 in relative L2 norm and the loss to 1e-3 (a rounding on the
other side of a tie moves one activation by 2^-8)."""
import numpy as np
import pytest

from devmem import DeviceArray
from oracle import oracle_py as O

pytestmark = pytest.mark.gpu

DIMS = [(256, 5), (256, 256), (256, 256), (256, 256), (6, 256)]


@pytest.mark.parametrize("n", [993, 1024, 1025, 2690, 16385, 17000])
def test_gradient_over_splits(acc, n):
    rng = np.random.default_rng(n)
    p = np.concatenate([v for o, i in DIMS for v in (rng.uniform(-1, 1, o * i) * np.sqrt(6.0 / i), rng.normal(size=o) * 0.1)])
    p = p.astype(np.float32)
    x = rng.uniform(-1, 1, (n, 5)).astype(np.float32)
    cls = rng.integers(0, 3, n).astype(np.int32)
    d = rng.normal(scale=0.2, size=(n, 3)).astype(np.float32)
    acc.mlp_set_params(p)
    print(f"[case] mlp splits n={n}", flush=True)
    xd, cd, dd = DeviceArray(x), DeviceArray(cls), DeviceArray(d)
    gd = DeviceArray(shape=(len(p),), dtype=np.float32)
    loss = acc.mlp_loss_grad(xd.data_ptr(), cd.data_ptr(), dd.data_ptr(), n, gd.data_ptr())
    g = gd.get().astype(np.float64)
    ref_loss, ref = O.mlp_loss_grad(p, x, cls, d, round_bf16=True)
    assert abs(loss - ref_loss) < 1e-3 * abs(ref_loss)
    at = 0
    for k, (o, i) in enumerate(DIMS):
        for name, m in ((f"W{k}", o * i), (f"b{k}", o)):
            err = np.linalg.norm(g[at:at + m] - ref[at:at + m]) / max(np.linalg.norm(ref[at:at + m]), 1e-30)
            assert err < 2e-2, (name, err)
            at += m
