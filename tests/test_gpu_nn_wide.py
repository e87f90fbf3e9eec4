"""A weight gradient on a map whose rows are 4 GB: accepted, and what few
nonzero pixels at its ends and past its 32-bit offsets give."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from simplewinderosion_amd import nn  # noqa: E402
from test_gpu_nn import DEV  # noqa: E402


def test_rows_of_four_gigabytes():
    print("case wgrad 4 GB rows", flush=True)
    W, C = (1 << 28) + 4, 8  # a row: 2^32 + 64 bytes
    assert torch.cuda.mem_get_info()[0] > 12 << 30
    x = torch.zeros((1, 1, W, C), device=DEV, dtype=torch.bfloat16)
    dy = torch.zeros((1, 1, W, C), device=DEV, dtype=torch.bfloat16)
    # pixel, x channel and value: neighbours of the pixels below, over the wrap too
    for p, c, v in ((0, 1, 2.0), (W - 1, 2, 3.0), (W - 2, 3, 5.0), (1, 4, 7.0), ((1 << 27) + 5, 5, 11.0)):
        x[0, 0, p, c] = v
    for p, c, v in ((0, 0, 1.0), (W - 1, 6, 0.5), ((1 << 27) + 4, 7, 4.0)):
        dy[0, 0, p, c] = v
    dw = torch.empty((C, 9, C), device=DEV)
    db = torch.empty((C,), device=DEV)
    nn.wgrad(x, dy, dw, db)
    torch.cuda.synchronize()
    want = torch.zeros((C, 3, C))  # by column shift; each of the three row taps sees the one row
    want[0, 1, 1], want[0, 0, 2], want[0, 2, 4] = 2.0, 3.0, 7.0
    want[6, 1, 2], want[6, 0, 3], want[6, 2, 1] = 1.5, 2.5, 1.0
    want[7, 2, 5] = 44.0
    got = dw.cpu().view(C, 3, 3, C)
    for row in range(3):
        assert torch.equal(got[:, row], want), row
    assert torch.equal(db.cpu(), torch.tensor([1.0, 0, 0, 0, 0, 0, 0.5, 4.0]))
