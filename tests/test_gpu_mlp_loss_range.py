"""The loss of the three-launch gradients where single squared errors are near
the largest float: their mean is a float, and no sum on the way may overflow."""
import numpy as np
import pytest

from conftest import load_package, gpu_available

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B", [1, 33, 8192])
@pytest.mark.parametrize("dout", [1, 9, 129])
def test_mean_of_large_squares(B, dout):
    if not gpu_available():
        pytest.skip("no GPU")
    import torch
    load_package()
    from ocfd_amd import surrogate
    net = surrogate.MLP([4, 64, dout])
    net.set_params(np.zeros(64 * 4 + 64 + dout * 64 + dout, np.float32))
    x = torch.ones((B, 4), device="cuda")
    y = torch.full((B, dout), 1.7e19, device="cuda")  # squares of 2.9e38, largest float 3.4e38
    loss, g = net.gradients(x, y)
    want = float(np.float32(1.7e19)) ** 2
    assert abs(loss.item() - want) <= 2.0 ** -22 * want
    # the last bias: 2 (0 - y) summed over the batch, over B dout
    gb = g.cpu().numpy()[-dout:]
    assert np.allclose(gb, -2.0 * 1.7e19 / dout, rtol=B * 2.0 ** -23)
