"""Loss and gradient of the network at the edges of the training kernels' tiles (32 samples) and of the
weight gradients' splits (16 tiles each): one row, one short of a tile, a tile, one more, one split
and a ragged second one. Against the network oracle with its operands rounded to BF16 where the
device rounds them: every layer's gradient to 2e-2 in relative L2 norm and the loss to 1e-3 (a
rounding on the other side of a tie moves one activation by 2^-8). The gradient array need not be
aligned to more than a float, and a second call gives the same bits."""
import numpy as np
import pytest

from devmem import DeviceArray
from oracle import oracle_py as O

pytestmark = pytest.mark.gpu

DIMS = [(256, 5), (256, 256), (256, 256), (256, 256), (6, 256)]


@pytest.mark.parametrize("n", [1, 31, 32, 33, 512, 545])
def test_gradient_at_tile_edges(acc, n):
    rng = np.random.default_rng(n)
    p = np.concatenate([v for o, i in DIMS for v in (rng.uniform(-1, 1, o * i) * np.sqrt(6.0 / i), rng.normal(size=o) * 0.1)])
    p = p.astype(np.float32)
    x = rng.uniform(-1, 1, (n, 5)).astype(np.float32)
    cls = rng.integers(0, 3, n).astype(np.int32)
    d = rng.normal(scale=0.2, size=(n, 3)).astype(np.float32)
    acc.mlp_set_params(p)
    print(f"[case] mlp loss_grad n={n}", flush=True)
    xd, cd, dd = DeviceArray(x), DeviceArray(cls), DeviceArray(d)
    gd = DeviceArray(shape=(len(p) + 1,), dtype=np.float32)
    out = []
    for off in (0, 4):
        loss = acc.mlp_loss_grad(xd.data_ptr(), cd.data_ptr(), dd.data_ptr(), n, gd.data_ptr() + off)
        out.append((loss, gd.get()[off // 4:off // 4 + len(p)].copy()))
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
    loss, g = out[0][0], out[0][1].astype(np.float64)
    ref_loss, ref = O.mlp_loss_grad(p, x, cls, d, round_bf16=True)
    assert abs(loss - ref_loss) < 1e-3 * abs(ref_loss)
    at = 0
    for k, (o, i) in enumerate(DIMS):
        for name, m in ((f"W{k}", o * i), (f"b{k}", o)):
            err = np.linalg.norm(g[at:at + m] - ref[at:at + m]) / max(np.linalg.norm(ref[at:at + m]), 1e-30)
            assert err < 2e-2, (name, err)
            at += m
