"""A sample's values in the three-launch gradients (networks of at most 256
wide) and in the chain of matrix products (wider ones), bit for bit.  The wide
network is the narrow one with 64 more units in the first hidden layer, whose
weights and biases are zero: they add exact zeros at the end of each sum.  With
one sample the gradients hold its dZ (biases) and single products (weights), so
nothing but the loss depends on the order of a sum."""
import numpy as np
import pytest

from conftest import load_package, gpu_available

pytestmark = pytest.mark.gpu


def flat(W, b):
    return np.concatenate([np.concatenate([w.ravel(), c]) for w, c in zip(W, b)]).astype(np.float32)


def split(g, dims):
    W, b, o = [], [], 0
    for i, d in zip(dims[:-1], dims[1:]):
        W.append(g[o:o + d * i].reshape(d, i))
        b.append(g[o + d * i:o + d * i + d])
        o += d * i + d
    return W, b


@pytest.mark.parametrize("dims", [(12, 256, 9), (12, 256, 256, 9), (7, 200, 64, 130, 1), (256, 256, 256)])
@pytest.mark.parametrize("seed", [0, 1])
def test_one_sample_equals_the_wide_network(dims, seed):
    if not gpu_available():
        pytest.skip("no GPU")
    import torch
    load_package()
    from ocfd_amd import surrogate
    rng = np.random.default_rng(seed)
    W = [rng.normal(0.0, 1.5 / np.sqrt(i), (d, i)).astype(np.float32) for i, d in zip(dims[:-1], dims[1:])]
    b = [rng.normal(0.0, 0.3, d).astype(np.float32) for d in dims[1:]]
    x, y = rng.normal(size=(1, dims[0])).astype(np.float32), rng.normal(size=(1, dims[-1])).astype(np.float32)
    # the wide one: the first hidden layer up to a multiple of 64, and 64 units more
    h = dims[1]
    wide = (dims[0], (h + 63) // 64 * 64 + 64 * (1 + (256 - (h + 63) // 64 * 64) // 64)) + tuple(dims[2:])
    assert max(dims) <= 256 < wide[1]
    Ww, bw = [w.copy() for w in W], [c.copy() for c in b]
    Ww[0] = np.zeros((wide[1], dims[0]), np.float32)
    Ww[0][:h] = W[0]
    bw[0] = np.zeros(wide[1], np.float32)
    bw[0][:h] = b[0]
    Ww[1] = np.zeros((dims[2], wide[1]), np.float32)
    Ww[1][:, :h] = W[1]
    out = []
    for d, w, c in ((dims, W, b), (wide, Ww, bw)):
        net = surrogate.MLP(list(d))
        net.set_params(flat(w, c))
        X, Y = torch.tensor(x, device="cuda"), torch.tensor(y, device="cuda")
        z = net.forward(X).cpu().numpy()
        loss, g = net.gradients(X, Y)
        out.append((z, loss.cpu().numpy(), split(g.cpu().numpy(), d)))
    (z0, l0, (gw0, gb0)), (z1, l1, (gw1, gb1)) = out
    assert z0.tobytes() == z1.tobytes()
    # the loss is a sum over the outputs as well, whose order differs: at most 256 squares in FP32
    assert abs(float(l0[0]) - float(l1[0])) <= 256 * 2.0 ** -24 * float(l1[0])
    # the last layer's bias gradient is 2 (output - y) / count: the outputs of the gradients' own forward pass
    cnt = np.float32(dims[-1])
    assert gb0[-1].tobytes() == (np.float32(2.0) * (z0[0] - y[0]) / cnt).astype(np.float32).tobytes()
    for k in range(len(dims) - 1):
        a, c = gb1[k], gw1[k]
        if k == 0:
            assert not c[h:].any()
            a, c = a[:h], c[:h]
        if k == 1:
            assert not c[:, h:].any()
            c = c[:, :h]
        assert gb0[k].tobytes() == a.tobytes(), k
        assert gw0[k].tobytes() == np.ascontiguousarray(c).tobytes(), k
