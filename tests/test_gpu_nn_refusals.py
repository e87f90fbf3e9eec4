"""Convolutions that are refused stay so: more than 65535 blocks of 32 output
channels on maps of whole 32-pixel strips; one block fewer runs."""
import pytest

torch = pytest.importorskip("torch")

pytestmark = pytest.mark.gpu

from simplewinderosion_amd import nn  # noqa: E402
from test_gpu_nn import DEV  # noqa: E402


@pytest.mark.parametrize("blocks,rc", [(65535, 0), (65536, -1)])
def test_output_channel_blocks(blocks, rc):
    print("case conv refusal", blocks, flush=True)
    cout = 32 * blocks
    x = torch.ones((1, 1, 32, 8), device=DEV, dtype=torch.bfloat16)
    w = torch.zeros((cout, 9, 8), device=DEV, dtype=torch.bfloat16)
    w[-1] = 1.0
    y = torch.empty((1, 1, 32, cout), device=DEV, dtype=torch.bfloat16)
    P = nn._p
    assert nn.load().swe_nn_conv3x3(P(x), 1, 1, 32, 8, P(w), None, cout, 0, P(y), None, None) == rc
    torch.cuda.synchronize()
    if rc == 0:
        assert torch.all(y[..., -1] == 72.0) and torch.all(y[..., :-1] == 0.0)
