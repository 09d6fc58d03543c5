"""Operands of the extension module's products, weight gradients, replicas and projection tables that do not
fit one another are refused before a kernel could read past them (no GPU needed: the checks come first)."""

import pytest
import torch

from atlas_rnn_amd import _lib
from atlas_rnn_amd import functional as F

BF16 = torch.bfloat16
NT, NN = 0, 1


def _z(*s, dt=BF16):
    return torch.zeros(*s, dtype=dt)


@pytest.mark.parametrize("layout,acts,weights,error", [
    (NT, [_z(4, 16)], [_z(8, 24)], RuntimeError),                  # k of the activation and of the weight differ
    (NN, [_z(4, 16)], [_z(24, 8)], RuntimeError),
    (NT, [_z(4, 16), _z(4, 16)], [_z(8, 16), _z(8, 8)], RuntimeError),
    (NT, [_z(4, 16)], [_z(8, 16)], RuntimeError),                  # fit, but not on a GPU
    (NT, [], [], ValueError),
    (NT, [_z(4, 16), _z(4, 16)], [_z(8, 16)], ValueError),
    (NT, [_z(4, 6, dt=torch.float32)], [_z(8, 7, dt=torch.float32)], RuntimeError),   # torch's product
])
def test_products(layout, acts, weights, error):
    with pytest.raises(error):
        _lib.native().products(layout, acts, weights)


def test_weight_gradients_replicas_and_tables():
    host = _lib.native()
    for dys, xs in (([], []), ([_z(4, 8)], [_z(4, 8), _z(4, 8)])):
        with pytest.raises(ValueError):
            host.wgrads(dys, xs, BF16)
    with pytest.raises(ValueError):
        host.replicate(0, [_z(4)])
    with pytest.raises(ValueError):
        host.replica_sum(0, [_z(4)])
    with pytest.raises(ValueError):
        host.symmetrized(_z(64, 16), 64, BF16)   # [d + d*d, m] is 4160 rows


@pytest.mark.gpu
def test_weights_on_another_device():
    x, w = _z(4, 16).cuda(), _z(8, 16)
    with pytest.raises(RuntimeError, match="do not fit"):
        F.linear(x, w)
    with pytest.raises(RuntimeError, match="do not fit"):
        F.linear(x[:, :8], w.cuda())
