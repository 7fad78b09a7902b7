"""A training step on whole numbers small enough that BF16 and FP32 hold every value and sum exactly:
the prediction, the loss and every gradient are then the float64 ones to the last bit. This runs the
kernels training runs (the ReLU's gradient inside the input-gradient convolution, the one-channel
output, the loss's shares and the folded partial sums), at tile counts where a workgroup of the
weights' gradient walks one item and several.
"""
import numpy as np
import pytest
import torch

from natray_amd import net
from tests.test_net import VOX, from_ncdhw, to_ncdhw, torch_weight


def whole_params(rng):
    """Two weights of +-1 per output channel (16 of the last layer's one), biases of -1..1."""
    p = np.zeros(net.PARAMS, np.float32)
    for cin, cout, _, wo, bo in net.LAYERS:
        W = np.zeros((27 * cin, cout), np.float32)
        for n in range(cout):
            k = 2 if cout > 1 else 16
            W[rng.choice(27 * cin, k, replace=False), n] = rng.choice([-1.0, 1.0], k)
        p[wo:wo + W.size] = W.reshape(-1)
        p[bo:bo + cout] = rng.integers(-1, 2, cout)
    return p


@pytest.mark.gpu
@pytest.mark.parametrize("tiles", [1, 2, 64])
def test_train_step_is_exact_on_whole_numbers(tiles):
    print(f"[net] whole numbers, {tiles} tiles", flush=True)
    rng = np.random.default_rng(tiles)
    n = net.Net(max_tiles=tiles, seed=1)
    p = whole_params(rng)
    n.set_params(p)
    X = rng.integers(-2, 3, (tiles, VOX, 2)).astype(np.float32)

    a = to_ncdhw(torch.from_numpy(X.astype(np.float64)))
    leaves, acts, pres = [], [a], []
    for cin, cout, relu, wo, bo in net.LAYERS:
        W = torch.from_numpy(p[wo:wo + 27 * cin * cout].astype(np.float64).reshape(27, cin, cout)).requires_grad_(True)
        b = torch.from_numpy(p[bo:bo + cout].astype(np.float64)).requires_grad_(True)
        leaves += [W, b]
        pre = torch.nn.functional.conv3d(a, torch_weight(W), b, padding=1)
        pre.retain_grad()
        pres.append(pre)
        a = torch.relu(pre) if relu else pre
        acts.append(a)
    out = from_ncdhw(a)[:, :, 0]
    error = torch.from_numpy(rng.integers(-1, 2, (tiles, VOX)).astype(np.float64))
    target = (out.detach() - error).numpy()
    count = tiles * VOX  # a power of two: dividing by it is exact
    loss = ((out - torch.from_numpy(target)) ** 2).sum() / count
    loss.backward()
    # What makes it exact: BF16 holds whole numbers up to 256, FP32 sums of them up to 2^24. (The
    # gradients are whole numbers of 2 / count.)
    unit = 2.0 / count
    for k in range(4):
        dz, act = pres[k].grad / unit, acts[k].detach()
        assert act.abs().max() <= 256 and dz.abs().max() <= 256
        assert act.abs().max() * dz.abs().sum() <= 1 << 24
        assert 0 < (dz != 0).sum() and 0 < (act == 0).sum() < act.numel()  # (a gate that does something)

    got = n.train_step(X, target.astype(np.float32), np.ones((tiles, VOX), np.float32), lr=0.0)
    grads = n.grads()
    np.testing.assert_array_equal(n.forward(X), out.detach().numpy().astype(np.float32))
    assert got == float(loss.detach())
    want = np.concatenate([t.grad.numpy().ravel() for t in leaves])
    np.testing.assert_array_equal(grads.astype(np.float64), want)
    n.close()
