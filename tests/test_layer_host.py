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
    return cls(patterns, algo="kernel", device="cpu:0", dtype=torch.float32, **kw)


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


class DenseKernel:
    """What the kernels compute, as dense products."""

    @staticmethod
    def forward(x, factor, bs_last, a, b, c, d, bias=None, **kw):
        with torch.no_grad():
            return dense_product(x, [factor], [(a, b, c, d)], bs_last, bias)

    @staticmethod
    def backward(grad, x, factor, bs_last, a, b, c, d, need_input=True, need_weight=True, **kw):
        with torch.enable_grad():
            xs, fs = x.detach().requires_grad_(), factor.detach().requires_grad_()
            y = dense_product(xs, [fs], [(a, b, c, d)], bs_last)
            return torch.autograd.grad(y, (xs, fs), grad.detach())

    @staticmethod
    def epilogue_backward(grad, z, bs_last, act=None, need_bias=True):
        with torch.no_grad():
            grad = torch.ops.aten.gelu_backward(grad, z) if act else grad
            return grad, grad.sum(1 if bs_last else 0) if need_bias else None


@pytest.fixture
def dense_kernel(monkeypatch):
    from ksmm_amd import kernel

    for name in ("forward", "backward", "epilogue_backward"):
        monkeypatch.setattr(kernel.Kernel, name, staticmethod(getattr(DenseKernel, name)))


def hooked(layer, x):
    """Hooks on a factor, the bias and an input with a history: each runs once a backward pass."""
    x = x * 1.0
    for t in (x, layer.bias, layer.factors[1]):
        if t is not None:
            t.register_hook(lambda g: 2 * g)
    return layer(x)


def tied(layer, x):
    layer.factors[2] = layer.factors[0]
    return layer(x)


def shared(layer, x):
    return layer(layer(x))


@pytest.mark.parametrize("call", [hooked, tied, shared])
@pytest.mark.parametrize("bs_last", [False, True])
@pytest.mark.parametrize("act", [None, "gelu"])
@pytest.mark.parametrize("bias", [False, True])
def test_gradients_with_a_graph(dense_kernel, monkeypatch, call, bs_last, act, bias):
    """create_graph=True: the gradients, and what can be differentiated again, as with a node per factor
    and PyTorch's bias and activation."""
    from ksmm_amd import kernel

    torch.manual_seed(3)
    weights = [torch.randn(p) / 2 for p in SQUARE]
    start, x0, g0 = torch.randn(8, 1) if bs_last else torch.randn(8), torch.randn(8, 8), torch.randn(8, 8)

    def gradients(one_node, create_graph):
        with monkeypatch.context() as m, torch.enable_grad():
            if not one_node:
                m.setattr(kernel.KSLayerFunction, "takes", staticmethod(lambda *a: False))
            layer = cpu_layer(SQUARE, weights=weights, bs_last=bs_last, act=act, bias=bias).double()
            if bias:
                layer.bias.data.copy_(start)
            x, g = x0.double().requires_grad_(), g0.double().requires_grad_()
            y = call(layer, x)
            args = [x] + list(layer.parameters())
            first = torch.autograd.grad(y, args, g, create_graph=create_graph)
            if not create_graph or not bias:
                return first
            assert args[1] is layer.bias and first[1].requires_grad
            again = torch.autograd.grad(first[1].pow(2).sum(), args + [g], allow_unused=True)
            return first + tuple(torch.zeros(1) if t is None else t for t in again)

    plain = gradients(False, False)
    for create_graph in (False, True):
        want, got = gradients(False, create_graph), gradients(True, create_graph)
        assert len(want) == len(got)
        for t, u in zip(got, want):
            torch.testing.assert_close(t, u, rtol=1e-12, atol=1e-12)
        for t, u in zip(got, plain):
            torch.testing.assert_close(t, u, rtol=1e-12, atol=1e-12)


@pytest.mark.parametrize("act", [None, "gelu"])
@pytest.mark.parametrize("create_graph", [False, True])
def test_bias_may_change_before_the_backward_pass(dense_kernel, act, create_graph):
    with torch.enable_grad():
        layer = cpu_layer(SQUARE, act=act).double()
        x, g = torch.randn(5, 8, dtype=torch.float64), torch.randn(5, 8, dtype=torch.float64)
        want = torch.autograd.grad(layer(x), list(layer.parameters()), g)
        y = layer(x)
        with torch.no_grad():
            layer.bias += 1
        for got, t in zip(torch.autograd.grad(y, list(layer.parameters()), g, create_graph=create_graph), want):
            torch.testing.assert_close(got, t, rtol=1e-12, atol=1e-12)


class Doubled(KSLinear):
    def post_process(self, tensor, output):
        return 2 * super().post_process(tensor, output)


class Shifted(KSLinear):
    def pre_process(self, tensor):
        return super().pre_process(tensor) + 1


class Negated(KSLinear):
    def forward_bs_first(self, output, x_scale=None):
        return -super().forward_bs_first(output, x_scale)


@pytest.mark.parametrize("cls,expected", [(Doubled, lambda layer, x: 2 * layer(x)), (Shifted, lambda layer, x: layer(x + 1)),
                                          (Negated, lambda layer, x: -layer(x))])
def test_steps_of_a_subclass_are_kept(native_stub, monkeypatch, cls, expected):
    from ksmm_amd import kernel

    def chain(x, factors, patterns, bs_last, bias=None, **kw):
        return dense_product(x, factors, patterns, bs_last, bias)

    monkeypatch.setattr(kernel.Kernel, "chain_forward", staticmethod(chain))
    plain, layer = cpu_layer(SQUARE), cpu_layer(SQUARE, cls=cls)
    layer.load_state_dict(plain.state_dict())
    x = torch.randn(5, 8)
    torch.testing.assert_close(layer(x), expected(plain, x))
    patched = cpu_layer(SQUARE)
    patched.post_process = lambda tensor, output: output + 3
    patched.load_state_dict(plain.state_dict())
    torch.testing.assert_close(patched(x), plain(x) + 3)


def test_without_the_native_module(monkeypatch):
    """A module that does not load costs a warning and host time, no call."""
    import sys
    import warnings

    import ksmm_amd
    from ksmm_amd import kernel

    monkeypatch.setattr(kernel.Kernel, "chain_forward",
                        staticmethod(lambda x, f, p, last, bias=None, **kw: dense_product(x, f, p, last, bias)))
    monkeypatch.setattr(_lib, "_native", None)
    monkeypatch.delattr(ksmm_amd, "_native", raising=False)
    monkeypatch.setitem(sys.modules, "ksmm_amd._native", None)  # as if it were not there
    layer, x = cpu_layer(SQUARE), torch.randn(5, 8)
    with pytest.warns(RuntimeWarning, match="_native"):
        got = layer(x)
    assert torch.equal(got, dense_product(x, layer.factors, SQUARE, False, layer.bias))
    with warnings.catch_warnings():
        warnings.simplefilter("error")
        layer(x)


def test_build_without_a_host_compiler(monkeypatch, tmp_path):
    from ksmm_amd import build

    for name in ("OBJ", "LIB", "BENCH_LIB", "NATIVE"):
        monkeypatch.setattr(build, name, str(tmp_path / name))
    (tmp_path / "NATIVE").write_text("of an earlier build")
    monkeypatch.setattr(build, "_compile", lambda src: (src, ""))
    run = build.subprocess.run

    def no_gxx(cmd, **kw):
        if cmd[0] == "g++":
            raise FileNotFoundError("g++")
        return run(["true"], **kw)

    monkeypatch.setattr(build.subprocess, "run", no_gxx)
    with pytest.warns(RuntimeWarning, match="g\\+\\+"):
        assert build.build() == build.LIB
    assert not (tmp_path / "NATIVE").exists()
