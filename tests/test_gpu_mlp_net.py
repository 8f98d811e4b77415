"""Gradients of networks of at most 256 wide (k_net: a workgroup carries 32
samples through the whole network) and of wider ones (GEMMs layer by layer)
against the oracle with bfloat16 activations: one layer to eight, widths at
and beside the multiples of 64, batches at and beside the multiples of 32.
Tolerances as for the fixed network: a bfloat16 rounding that falls the other
way moves single activations by 2^-9."""
import numpy as np
import pytest

from conftest import load_package, gpu_available
from oracle import mlp_oracle as mo

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def pkg():
    if not gpu_available():
        pytest.skip("no GPU")
    return load_package()


CASES = [((12, 9), 1), ((12, 9), 33), ((3, 64, 5), 31), ((64, 65, 64), 64), ((200, 192, 128, 70), 100),
         ((256, 256, 256), 129), ((1, 7, 1), 257), ((12, 256, 256, 256, 256, 256, 9), 8192),
         ((5, 64, 192, 64, 256, 64, 128, 64, 2), 1000), ((257, 64, 9), 100), ((12, 320, 9), 1000)]


@pytest.mark.parametrize("dims,n", CASES)
def test_gradients(pkg, dims, n):
    import torch
    from ocfd_amd import surrogate
    net = surrogate.MLP(dims, seed=5)
    flat = net.get_params()
    rng = np.random.default_rng(n)
    x = rng.standard_normal((n, dims[0])).astype(np.float32)
    y = rng.standard_normal((n, dims[-1])).astype(np.float32)
    xd, yd = torch.tensor(x).cuda(), torch.tensor(y).cuda()
    for _ in range(2):  # the second call finds its workspace
        loss, g = net.gradients(xd, yd)
    lo, go = mo.gradients(flat.astype(np.float64), dims, x.astype(np.float64), y.astype(np.float64), bf16=True)
    g = g.cpu().numpy()
    assert abs(loss.item() - lo) <= 1e-4 * lo
    k = 0
    for din, dout in zip(dims[:-1], dims[1:]):
        for size in (din * dout, dout):
            a, b = g[k:k + size], go[k:k + size]
            assert np.linalg.norm(a - b) < 2e-2 * np.linalg.norm(b), (din, dout, size)
            k += size


def test_weights_after_training_steps(pkg):
    """Every copy of the weights follows Adam: gradients after train_step
    equal those of a fresh network given the same parameters, bit for bit."""
    import torch
    from ocfd_amd import surrogate
    dims = (12, 100, 256, 9)
    rng = np.random.default_rng(1)
    x = torch.tensor(rng.standard_normal((500, 12)).astype(np.float32)).cuda()
    y = torch.tensor(rng.standard_normal((500, 9)).astype(np.float32)).cuda()
    net = surrogate.MLP(dims, seed=2)
    for _ in range(3):
        net.train_step(x, y, lr=1e-2)
    p = net.get_params()
    la, ga = net.gradients(x, y)
    la, ga = la.item(), ga.cpu().numpy()
    net.set_params(p)
    lb, gb = net.gradients(x, y)
    assert la == lb.item() and np.array_equal(ga, gb.cpu().numpy())
