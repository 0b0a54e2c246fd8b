"""Gradients of a layer's epilogue (ksmm_act_bwd.hip) at the edges of its kernels, and of whole layers
whose epilogue goes through it, against float64.

Tolerance: dz is rounded once to its type (fp32: after a few operations, 2^-21; fp16: 2^-11 = 5e-4),
and a bias gradient is a sum of n <= 5000 of them in fp32, off by about sqrt(n) * 2^-24 < 1e-5 before
the last rounding."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-5, torch.float16: 6e-4}


def rel(got, want):
    return ((got.double() - want).norm() / want.norm()).item()


# features that 16 bytes divide, that a word divides, odd ones; one row, few, several batch ranges; rows of
# lanes that the features fill and not
CASES = [(1, 1), (3, 5), (7, 333), (8, 64), (16, 4197), (66, 130), (384, 31), (385, 515), (520, 1030), (1536, 777), (4, 5000)]


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("bs_last", [False, True])
@pytest.mark.parametrize("act", [None, "gelu"])
@pytest.mark.parametrize("offset", [0, 1])
def test_epilogue_gradient_edges(dt, bs_last, act, offset):
    """``offset``: the operands start one element behind a 16-byte boundary."""
    from ksmm_amd import Kernel

    gen = torch.Generator(device="cuda").manual_seed(7)
    for features, n in CASES:
        shape = (features, n) if bs_last else (n, features)

        def tensor():
            return torch.randn(offset + features * n, generator=gen, device="cuda").to(dt)[offset:].view(shape)

        z, dy = tensor() * 2, tensor()
        if offset:
            z = torch.cat([z.reshape(-1)[:1], z.reshape(-1)])[1:].view(shape)
        gz, gb = Kernel.epilogue_backward(dy, z if act else None, bs_last, act)
        want = dy.double()
        if act:
            x = z.double().requires_grad_(True)
            with torch.enable_grad():
                want = torch.autograd.grad(F.gelu(x), x, want)[0]
            assert rel(gz, want) <= TOL[dt], (features, n)
        else:
            assert gz is dy
        # against the sum of magnitudes' root: sums of random signs cancel
        err = (gb.double() - want.sum(1 if bs_last else 0)).norm() / want.norm()
        assert err.item() <= TOL[dt] * (1 if dt == torch.float32 else 4), (features, n, err.item())


@pytest.mark.parametrize("bs_last", [False, True])
@pytest.mark.parametrize("act", [None, "gelu"])
def test_layer_gradients_equal_those_factor_by_factor(bs_last, act):
    """The layer's one autograd node against a node per factor with PyTorch's bias and activation: all
    combinations of wanted gradients, and second derivatives through the bias."""
    from ksmm_amd import KSLinear
    from ksmm_amd.kernel import layer_by_factors

    patterns = [(2, 24, 16, 3), (3, 20, 16, 3)]
    with torch.enable_grad():
        for wanted in ("xbw", "xw", "w", "bw", "xb"):
            layer = KSLinear(patterns, algo="kernel", dtype=torch.float32, bs_last=bs_last, device="cuda", act=act)
            for f in list(layer.factors)[1:]:
                f.requires_grad_("w" in wanted)
            layer.bias.requires_grad_("b" in wanted)
            x = torch.randn((96, 37) if bs_last else (37, 96), device="cuda", requires_grad="x" in wanted)
            args = ([x] if "x" in wanted else []) + [p for p in layer.parameters() if p.requires_grad]
            y = layer(x)
            ref = layer_by_factors(x, layer.bias, act, bs_last, layer.patterns, layer.factors)
            g = torch.randn_like(y).expand_as(y)
            for got, want in zip(torch.autograd.grad(y, args, g, retain_graph=True),
                                 torch.autograd.grad(ref, args, g, retain_graph=True)):
                assert got.shape == want.shape and got.is_contiguous() and rel(got, want.double()) <= 1e-5
            if act and "b" in wanted:
                second = [torch.autograd.grad(torch.autograd.grad(out, layer.bias, g, create_graph=True)[0].sum(), layer.bias)[0]
                          for out in (y, ref)]
                assert rel(second[0], second[1].double()) <= 1e-5


@pytest.mark.parametrize("bs_last", [False, True])
@pytest.mark.parametrize("act", [None, "gelu"])
@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
def test_gradients_with_a_graph_on_shared_parameters(bs_last, act, dt):
    """create_graph=True through a layer applied twice, with one parameter for two factors and a hook on the bias:
    as without a graph, where the same kernels run (a sum rounds apart)."""
    from ksmm_amd import KSLinear

    patterns = [(1, 16, 16, 4), (4, 16, 16, 1), (1, 16, 16, 4)]
    with torch.enable_grad():
        layer = KSLinear(patterns, algo="kernel", dtype=dt, bs_last=bs_last, device="cuda", act=act)
        layer.factors[2] = layer.factors[0]
        layer.bias.register_hook(lambda g: 2 * g)
        x = torch.randn(64, 64, device="cuda", dtype=dt, requires_grad=True)
        g = torch.randn(64, 64, device="cuda", dtype=dt)
        args = [x] + list(layer.parameters())
        want = torch.autograd.grad(layer(layer(x)), args, g)
        for got, ref in zip(torch.autograd.grad(layer(layer(x)), args, g, create_graph=True), want):
            # fp16: the slope by PyTorch's kernel or the series, rounded to 2^-11 in each of two layers
            assert rel(got, ref.double()) <= (1e-5 if dt == torch.float32 else 2e-3)
