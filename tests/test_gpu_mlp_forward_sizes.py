"""Inference at the edges of the fused kernel's tiles of 128 rows: one row, one short of a tile, a tile,
one more, several and a remainder. A row's outputs do not depend on the batch around it (the same bits
as in a larger batch), and nothing is written past the last row."""
import pytest

from sirius_amd.accelerator import HipAccelerator

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

ROWS = 1100


@pytest.fixture(scope="module")
def whole():
    acc = HipAccelerator()
    acc.mlp_init(7)
    g = torch.Generator().manual_seed(3)
    x = torch.randn(ROWS, 5, generator=g).cuda()
    y = torch.zeros(ROWS, 6, device="cuda")
    torch.cuda.synchronize()
    acc.mlp_forward(x.data_ptr(), y.data_ptr(), ROWS)
    torch.cuda.synchronize()
    assert torch.isfinite(y).all() and y.std() > 0
    return acc, x, y


@pytest.mark.parametrize("rows", [1, 2, 31, 32, 33, 127, 128, 129, 255, 257, 1024, 1099])
def test_forward_rows(whole, rows):
    acc, x, y = whole
    print(f"[case] forward {rows} rows", flush=True)
    for first in (0, ROWS - rows):  # from the top, and the last rows as a batch of their own
        out = torch.full((rows + 64, 6), 7.5, device="cuda")
        part = x[first:first + rows].contiguous()
        torch.cuda.synchronize()
        acc.mlp_forward(part.data_ptr(), out.data_ptr(), rows)
        torch.cuda.synchronize()
        assert torch.equal(out[:rows], y[first:first + rows])
        assert (out[rows:] == 7.5).all()
