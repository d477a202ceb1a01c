"""The quantized linears as modules (CPU): forward finds its tensors wherever
attribute lookup does -- parameters and buffers, plain attributes as in the
replicas of nn.DataParallel, parametrizations -- as the reference's modules do
(nanovllm/layers/linear_w4a16.py:128-148, linear_w4a4.py:27-35)."""
import pytest
import torch
from torch import nn
from torch.nn.utils import parametrize

from nv4.layers import W4A4Linear, W4A16Linear
from nv4.layers import linear_w4a4, linear_w4a16


@pytest.fixture
def seen(monkeypatch):
    """The tensors that the operators behind forward are called with."""
    calls = []

    def w4a16(x, qweight, qzeros, scales, group_size):
        calls.append((qweight, qzeros, scales))
        return x.new_zeros(x.shape[0], scales.shape[1])

    def w4a4(x, signs, packed, scale, **options):
        calls.append((signs, packed, scale))
        return x.new_zeros(x.shape[0], packed.shape[0])

    monkeypatch.setattr(linear_w4a16, "dequant_matmul_w4a16", w4a16)
    monkeypatch.setattr(linear_w4a4, "w4a4_linear", w4a4)
    return calls


def linears():
    return [(W4A16Linear(256, 64), ("qweight", "qzeros", "scales")),
            (W4A4Linear(4096, 64), ("signs", "packed_weight", "weight_scale"))]


def forward(module, seen, rows=(3,)):
    seen.clear()
    out = module(torch.zeros(*rows, module.in_features, dtype=torch.bfloat16))
    assert out.shape == (*rows, module.out_features)
    return seen[0]


@pytest.mark.parametrize("rows", [(3,), (2, 3)])
def test_plain_attributes(seen, rows):
    for module, names in linears():
        tensors = []
        for name in names:
            t = getattr(module, name).detach().clone()
            delattr(module, name)
            setattr(module, name, t)
            assert name not in module._parameters and name not in module._buffers
            tensors.append(t)
        assert all(a is b for a, b in zip(forward(module, seen, rows), tensors))


def test_data_parallel_replica(seen):
    """What nn.parallel.replicate leaves: no parameters, their copies as plain attributes."""
    for module, names in linears():
        replica = module._replicate_for_data_parallel()
        copies = [getattr(module, name).detach().clone() for name in names]
        for name, t in zip(names, copies):
            setattr(replica, name, t)
        assert all(a is b for a, b in zip(forward(replica, seen), copies))


class _Moved(nn.Module):
    def forward(self, t):
        return t + 1


def test_parametrized(seen):
    module, _ = linears()[0]
    before = module.scales.detach().clone()
    parametrize.register_parametrization(module, "scales", _Moved(), unsafe=True)
    assert torch.equal(forward(module, seen)[2].nan_to_num(), (before + 1).nan_to_num())


def test_registered_tensors(seen):
    for module, names in linears():
        got = forward(module, seen)
        assert all(a is getattr(module, n) for a, n in zip(got, names))
