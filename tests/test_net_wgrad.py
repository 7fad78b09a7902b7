"""The weights' gradient where a workgroup walks several work items (more than 32 tiles) and where
only a few run (1 tile), against torch's CPU conv3d in float64 on the same BF16-rounded tensors."""
import numpy as np
import pytest
import torch

from natray_amd import net
from tests.test_net import VOX, bf16, rel_err, to_ncdhw, torch_weight


@pytest.mark.gpu
@pytest.mark.parametrize("cin,cout,relu,tiles", [(2, 16, True, 1), (2, 16, False, 37), (16, 16, True, 1), (16, 16, False, 37),
                                                 (16, 1, False, 33)])
def test_weight_gradient(cin, cout, relu, tiles):
    rng = np.random.default_rng(cin * 1000 + tiles)
    X = rng.standard_normal((tiles, VOX, cin)).astype(np.float32)
    W = (rng.standard_normal((27, cin, cout)) * np.sqrt(2.0 / (27 * cin))).astype(np.float32)
    b = rng.standard_normal(cout).astype(np.float32) * 0.1
    dY = rng.standard_normal((tiles, VOX, cout)).astype(np.float32)
    Y, _, dW, db = net.layer_check(cin, cout, relu, X, W, b, dY)
    dZ = bf16(np.where(Y > 0, dY, 0.0) if relu else dY)
    w = torch_weight(bf16(W)).requires_grad_(True)
    bias = torch.zeros(cout, dtype=torch.float64, requires_grad=True)
    out = torch.nn.functional.conv3d(to_ncdhw(bf16(X)), w, bias, padding=1)
    (out * to_ncdhw(dZ)).sum().backward()
    ref = w.grad.permute(2, 3, 4, 1, 0).reshape(27, cin, cout)
    # FP32 sums of tiles * 4096 unit-variance products: at most a few sqrt(count) * 2^-24 of the
    # largest partial sum, which is of the size of the largest gradient here.
    assert rel_err(dW, ref) <= 2e-4
    assert rel_err(db, bias.grad) <= 2e-4
