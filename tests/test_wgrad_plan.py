"""Which kernel a weight gradient takes (wgrad_plan in csrc/swe_nn.hip), read
from the workspace it asks for: the faster one of each measured layer (us of
the small layers' kernels / of k_wgrad)."""
import pytest

pytest.importorskip("torch")

from simplewinderosion_amd import nn  # noqa: E402

MEASURED = [
    # N, H, W, Cin, Cout, us small, us k_wgrad (layers whose partials' sizes tell the kernel)
    (1, 128, 128, 8, 32, 9.5, 12.1),
    (1, 256, 256, 8, 32, 11.4, 13.3), (1, 128, 128, 64, 32, 11.5, 12.5),
    (8, 32, 32, 64, 32, 10.4, 11.3), (1, 32, 32, 128, 64, 9.5, 10.7),
    (8, 1, 128, 40, 64, 7.3, 17.6), (8, 4, 4, 192, 256, 11.1, 12.5),
    (8, 2, 2, 256, 256, 9.4, 10.8), (1, 4096, 1, 64, 64, 13.4, 20.4), (3, 8, 4, 32, 8, 7.5, 11.3),
    (8, 128, 128, 64, 64, 26.4, 19.6),
    (8, 64, 64, 128, 128, 30.5, 21.6), (8, 16, 16, 256, 192, 30.6, 16.0),
    (2, 64, 64, 128, 128, 16.8, 13.2), (4, 8, 8, 128, 192, 13.3, 12.4), (4, 4, 4, 256, 256, 10.2, 9.4),
    (1, 8, 8, 256, 192, 9.1, 8.5), (2, 12, 16, 192, 256, 16.0, 10.1), (6, 1, 64, 256, 192, 17.3, 11.1),
    (8, 128, 128, 256, 192, 174.5, 116.7), (4, 256, 256, 192, 8, 49.8, 31.6),
]


@pytest.mark.parametrize("N,H,W,Cin,Cout,small,strips", MEASURED)
def test_the_faster_kernel_is_taken(N, H, W, Cin, Cout, small, strips):
    work = nn.load().swe_nn_wgrad_work(N, H, W, Cin, Cout)
    # floats of a chunk's partials: whole 32 x 32 blocks with their 32 bias sums,
    # or the layer's own weights and biases
    whole, own = -(-Cout // 32) * -(-Cin // 32) * (9 * 32 * 32 + 32), 9 * Cin * Cout + Cout
    assert (work % whole == 0) != (work % own == 0)
    assert (work % whole == 0) == (strips < small)
