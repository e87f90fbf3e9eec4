"""k_wgrad_rows and k_wgrad_flat (swe_nn.hip), the weight gradients of small
layers, where they can go wrong: one and several chunks, chunks of a strip cut
short, rows and images crossed within a step, partial channel blocks, one-row
and one-column maps; against float64 with the tolerance of float32 sums over
the pixels, and repeated to the bit."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from simplewinderosion_amd import nn  # noqa: E402
from test_gpu_nn import DEV, rnd  # noqa: E402


@pytest.mark.parametrize("N,H,W,Cin,Cout", [
    # whole strips
    (1, 128, 128, 8, 32), (1, 130, 32, 64, 8), (2, 29, 64, 40, 56), (3, 1, 96, 16, 24), (1, 33, 32, 128, 64),
    # flattened pixels: under 32 of them, 33, a chunk, several, over images and rows
    (1, 1, 1, 8, 8), (1, 3, 11, 8, 72), (8, 4, 4, 192, 256), (8, 2, 2, 40, 264), (2, 9, 7, 24, 8), (3, 300, 1, 72, 16),
    (1, 700, 3, 64, 40),
])
def test_small_wgrad(N, H, W, Cin, Cout):
    print("case wgrad small", N, H, W, Cin, Cout, flush=True)
    whole = -(-Cout // 32) * -(-Cin // 32) * (9 * 32 * 32 + 32)
    assert nn.load().swe_nn_wgrad_work(N, H, W, Cin, Cout) % whole != 0  # one of these kernels
    x = rnd((N, H, W, Cin), seed=51)
    dy = rnd((N, H, W, Cout), seed=52)
    dw = torch.empty((Cout, 9, Cin), device=DEV)
    db = torch.empty((Cout,), device=DEV)
    work = nn.wgrad(x, dy, dw, db)
    again = torch.empty_like(dw)
    nn.wgrad(x, dy, again, None, work)
    torch.cuda.synchronize()
    xd, dd = x.cpu().double(), dy.cpu().double().reshape(-1, Cout)
    taps = [torch.roll(xd, (1 - t // 3, 1 - t % 3), (1, 2)).reshape(-1, Cin) for t in range(9)]
    ref = torch.stack([dd.T @ v for v in taps], 1)
    tol = 1e-5 * (N * H * W) ** 0.5 + 1e-3
    assert torch.allclose(dw.cpu().double(), ref, atol=tol, rtol=1e-4)
    assert torch.allclose(db.cpu().double(), dd.sum(0), atol=tol, rtol=1e-4)
    assert torch.equal(dw.view(torch.int32), again.view(torch.int32))
