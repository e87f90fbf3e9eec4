"""k_conv_tile and k_conv_wide (swe_nn.hip) where they can go wrong: every
workgroup shape (64 PF pixels x 16 CF channels, tiles of 16 or 32 columns),
several tiles a workgroup, one and two weight buffers, channels in several
blocks, the slices of a split reduction, tiles cut by the map's edges, maps
smaller than a patch (rows and columns that wrap more than once), a partial
last 32-channel chunk, channels past the last block, and outputs and masks
that 16-byte accesses cannot take.  Against float64 (CPU) with the tolerance
of float32 accumulation over 9 Cin products."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from simplewinderosion_amd import nn  # noqa: E402
from test_gpu_nn import DEV, ref_conv, rnd  # noqa: E402

CASES = [
    # N, H, W, Cin, Cout
    (16, 128, 160, 8, 8),     # (4, 1), two tiles a workgroup
    (3, 37, 45, 24, 13),      # (4, 1), 16 columns, partial tiles, Cout not a multiple of 8
    (8, 256, 128, 8, 24),     # (4, 2), two tiles a workgroup
    (8, 352, 48, 16, 32),     # (4, 2), 16 columns
    (8, 64, 64, 32, 32),      # (2, 2)
    (8, 128, 48, 8, 192),     # (4, 4), 16 columns
    (8, 64, 64, 16, 136),     # (2, 4), a partial channel block
    (9, 64, 48, 16, 320),     # (2, 4), 16 columns
    # above 32 input channels; `2` is two weight buffers, `k` several blocks of channels
    (1, 9, 21, 264, 24), (1, 9, 16, 72, 24), (2, 19, 21, 72, 24),  # (1, 1): k; 16 columns 2; 2
    (5, 9, 45, 264, 200), (5, 9, 45, 72, 200),      # (1, 2), 16 columns: k, 2
    (8, 9, 21, 72, 200), (8, 9, 21, 40, 200),       # (1, 2): 2
    (5, 17, 45, 136, 200), (5, 17, 45, 72, 200),    # (2, 2), 16 columns: -, 2
    (5, 32, 21, 136, 200), (8, 33, 21, 264, 40),    # (2, 2): -, 2 k
    (5, 33, 45, 104, 200), (5, 17, 45, 264, 200),   # (2, 4), 16 columns: -, 2 k
    (5, 64, 21, 104, 200), (8, 17, 21, 264, 200),   # (2, 4): -, k
    (5, 33, 45, 72, 200), (5, 64, 21, 72, 200),     # (4, 2): 16 columns 2; -
    (5, 32, 21, 192, 200),                          # (4, 2): 2
    (8, 33, 45, 264, 136), (8, 64, 45, 40, 192),    # (4, 4), 16 columns: k, 2
    (8, 33, 21, 264, 200), (8, 128, 128, 40, 64),   # (4, 4): k, 2
    (2, 32, 32, 64, 200), (2, 60, 200, 40, 32),
    (1, 1, 16, 8, 40), (1, 5, 1, 8, 16), (2, 3, 2, 40, 48), (5, 2, 9, 16, 8), (1, 4, 4, 96, 40),  # under a patch
]


@pytest.mark.parametrize("N,H,W,Cin,Cout", CASES)
def test_conv_tile(N, H, W, Cin, Cout):
    print("case conv tile", N, H, W, Cin, Cout, flush=True)
    x = rnd((N, H, W, Cin), seed=31)
    w = rnd((Cout, 9, Cin), seed=32, scale=0.2)
    b = rnd((Cout,), torch.float32, seed=33)
    mask = rnd((N, H, W, Cout), seed=34)
    y32 = torch.empty((N, H, W, Cout), device=DEV)
    y16 = torch.empty((N, H, W, Cout), device=DEV, dtype=torch.bfloat16)
    nn.conv3x3(x, w, b, out16=y16, out32=y32)
    relu = nn.conv3x3(x, w, b, relu=True)
    masked = nn.conv3x3_masked(x, w, mask, torch.empty_like(y16), bias=b)
    # the same through unaligned buffers: two-byte accesses, the same bits
    n = y16.numel()
    off16 = torch.empty(n + 1, device=DEV, dtype=torch.bfloat16)[1:].view(N, H, W, Cout)
    offm = torch.empty(n + 1, device=DEV, dtype=torch.bfloat16)[1:].view(N, H, W, Cout).copy_(mask)
    P = nn._p
    assert nn.load().swe_nn_conv3x3_masked(P(x), N, H, W, Cin, P(w), P(b), Cout, P(offm), P(off16), None) == 0
    torch.cuda.synchronize()
    ref = ref_conv(x, w, b)
    assert torch.allclose(y32, ref, atol=1e-4 * (9 * Cin) ** 0.5, rtol=1e-4)
    assert torch.equal(y16, y32.to(torch.bfloat16))
    assert torch.equal(relu, y32.clamp_min(0).to(torch.bfloat16))
    want = torch.where(mask > 0, y16, torch.zeros_like(y16))
    assert torch.equal(masked, want)
    assert torch.equal(off16, want)
    need = nn.conv_work(N, H, W, Cin, Cout)
    if need:  # the slices of a split reduction, added in order
        work = torch.empty(need, device=DEV)
        nn.conv3x3(x, w, b, relu=True, out16=y16, out32=y32, work=work)
        torch.cuda.synchronize()
        assert torch.allclose(y32, ref.clamp_min(0), atol=1e-4 * (9 * Cin) ** 0.5, rtol=1e-4)
        assert torch.equal(y16, y32.to(torch.bfloat16))


@pytest.mark.parametrize("N,H,W,Cin,Cout", [
    (1, 1, 1, 8, 8),         # one pixel: every tap is it
    (2, 4, 4, 96, 40),       # one chunk: no pass over the partials
    (1, 2, 33, 40, 24), (3, 3, 31, 32, 32), (1, 7, 95, 8, 72),  # 1 .. 7 rows, strips of 1, 31, 32 columns
    (5, 13, 50, 64, 64),     # the last chunk of a strip one row shorter
    (1, 260, 70, 32, 64),    # over 32 chunks
    (3, 9, 70, 512, 520),    # three units a wave, a wave without one
])
def test_wgrad_units(N, H, W, Cin, Cout):
    """k_wgrad's strips, rows and units against float64; columns past a strip's
    end count for nothing even where the map holds infinities there."""
    print("case wgrad units", N, H, W, Cin, Cout, flush=True)
    x = rnd((N, H, W, Cin), seed=41)
    dy = rnd((N, H, W, Cout), seed=42)
    x[0, 0, min(32, W - 1), 3] = float("inf")
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
    assert torch.allclose(dw.cpu().double(), ref, atol=tol, rtol=1e-4, equal_nan=True)
    assert torch.allclose(db.cpu().double(), dd.sum(0), atol=tol, rtol=1e-4)
    assert torch.equal(dw.view(torch.int32), again.view(torch.int32))
