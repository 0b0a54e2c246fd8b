"""Host side of KSLinear(algo='kernel') without a GPU: which tensors reach the kernels.  The native module is
replaced by the same product in plain tensors, and layers are built on the CPU around the constructor's test of
the device."""
import pytest
import torch
from torch import nn
from torch.nn.utils import parametrize, prune

from ksmm_amd import KSLinear, _lib
from ksmm_amd.layer import from_kernel_format_to_dense

SQUARE = [(1, 4, 4, 2), (2, 4, 4, 1), (1, 4, 4, 2)]  # equally shaped factors: a wrong order fits as well


def cpu_layer(patterns, cls=KSLinear, **kw):
    """A layer whose kernel-format factors live on the CPU."""
    kw = dict(dtype=torch.float32, **kw)
    layer = cls(patterns, algo="kernel", device="cpu:0", **kw)
    return layer


def dense_product(x, factors, patterns, bs_last, bias=None):
    for f, p in zip(factors, patterns):
        k = from_kernel_format_to_dense(f, p)
        x = k @ x if bs_last else x @ k.t()
    return x if bias is None else x + bias


class NativeStub:
    @staticmethod
    def infer(x, factors, patterns, bs_last, scales, fuse, bias, act, quantise):
        return dense_product(x, factors, patterns, bs_last, bias)


@pytest.fixture
def native_stub(monkeypatch):
    monkeypatch.setattr(_lib, "native", lambda: NativeStub)


def pruned(layer, i):
    prune.l1_unstructured(layer.factors, str(i), 0.5)


def pruned_for_good(layer, i):
    pruned(layer, i)
    prune.remove(layer.factors, str(i))


class Halved(nn.Module):
    def forward(self, w):
        return w / 2


def parametrised(layer, i):
    parametrize.register_parametrization(layer.factors, str(i), Halved())


def parametrised_for_good(layer, i):
    parametrised(layer, i)
    parametrize.remove_parametrizations(layer.factors, str(i))


@pytest.mark.parametrize("patterns", [SQUARE, [(2, 3, 5, 2)]])
@pytest.mark.parametrize("change", [pruned, pruned_for_good, parametrised, parametrised_for_good])
def test_factors_of_the_native_call_are_the_layers(native_stub, patterns, change):
    for i in range(len(patterns)):
        for bs_last in (False, True):
            layer = cpu_layer(patterns, bs_last=bs_last)
            x = torch.randn((layer.in_size, 7) if bs_last else (7, layer.in_size))
            before = layer(x)
            change(layer, i)
            want = dense_product(x, list(layer.factors), patterns, bs_last, layer.bias)
            got = layer(x)
            assert torch.equal(got, want), (i, bs_last)
            assert not torch.equal(got, before)


def test_wanted_gradients_are_those_of_the_layers_factors(native_stub):
    layer = cpu_layer(SQUARE)
    pruned(layer, 0)
    with torch.enable_grad():
        prune.l1_unstructured(layer.factors, "1", 0.5)
        for f in layer.factors.parameters():
            f.requires_grad_(False)
        assert layer.factors[1].requires_grad  # the masked tensor keeps its history
        assert layer._infer(torch.randn(3, layer.in_size), None) is None
