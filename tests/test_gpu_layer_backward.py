"""A layer's backward pass in one call (ksmm_layer_backward) against one call per factor and epilogue, which the
same kernels serve: the same bits.  The shapes are the edges of what the one call adds, the transposes and the sums
of a whole layer in one launch: blocks below, at and above a 64 x 64 square, products a x b x c x d that four does
not divide, few and many partial sums, and every set of wanted gradients."""
import itertools

import pytest
import torch

from ksmm_amd import _lib

pytestmark = pytest.mark.gpu

CASES = [
    ([(1, 7, 5, 3)], 37),  # 105 weights: scalar sums
    ([(2, 64, 64, 1), (1, 65, 128, 1), (5, 63, 13, 1)], 515),
    ([(1, 16, 16, 4), (4, 16, 16, 1)], 9001),  # many partial sums
    ([(3, 130, 1, 2), (1, 1, 260, 3), (1, 129, 1, 3)], 64),
]


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("bs_last", [False, True])
@pytest.mark.parametrize("act", [None, "gelu"])
def test_layer_gradients_equal_those_of_single_calls(dt, bs_last, act, monkeypatch):
    from ksmm_amd import KSLinear

    for patterns, n in CASES:
        layer = KSLinear(patterns, algo="kernel", dtype=dt, bs_last=bs_last, device="cuda", act=act)
        shape = (layer.in_size, n) if bs_last else (n, layer.in_size)
        x = torch.randn(shape, device="cuda").to(dt)
        with torch.enable_grad():
            for wanted in itertools.product((False, True), repeat=2 + len(patterns)):
                if not any(wanted[:1] + wanted[2:]):
                    continue  # the bias alone is a layer without gradients of its factors
                x.requires_grad_(wanted[0])
                layer.bias.requires_grad_(wanted[1])
                for f, w in zip(layer.factors, wanted[2:]):
                    f.requires_grad_(w)
                args = [t for t in (x, *layer.parameters()) if t.requires_grad]
                with monkeypatch.context() as m:
                    m.setattr(_lib, "_native", _lib._NoNative)
                    y = layer(x)
                    g = torch.randn_like(y)
                    want = torch.autograd.grad(y, args, g)
                z = layer(x)
                assert torch.equal(z, y)
                for got, ref in zip(torch.autograd.grad(z, args, g), want):
                    assert got.shape == ref.shape and torch.equal(got, ref), (patterns, wanted)


def test_layer_backward_refuses_what_the_single_calls_refuse():
    lib = _lib.load()
    d = (_lib.KsmmFactorDesc * 2)()
    for i, (a, b, c, dd) in enumerate([(2, 8, 8, 1), (1, 4, 16, 1)]):
        d[i].a, d[i].b, d[i].c, d[i].d, d[i].w_dtype, d[i].scale = a, b, c, dd, _lib.KSMM_F32, 1.0
    assert lib.ksmm_layer_backward_workspace(d, 2, 8, _lib.KSMM_F32, 0, _lib.ACT_NONE) > 0
    assert lib.ksmm_layer_backward_workspace(d, 2, 8, _lib.KSMM_F16, 0, _lib.ACT_NONE) < 0  # weights of another type
    assert lib.ksmm_layer_backward_workspace(d, 2, 0, _lib.KSMM_F32, 0, _lib.ACT_NONE) < 0
    d[1].c = 15
    assert lib.ksmm_layer_backward_workspace(d, 2, 8, _lib.KSMM_F32, 0, _lib.ACT_NONE) < 0  # sizes out of line


@pytest.mark.parametrize("pattern", [(1, 1, 1, 1 << 24), (1 << 24, 1, 1, 1), (1 << 12, 3, 5, 17), (3, 16, 16, 64), (2, 33, 31, 5),
                                     (1, 1, 700, 3), (2, 700, 1, 3), (1, 512, 512, 1), (1, 513, 512, 1), (260, 32, 32, 1),
                                     (5000, 7, 65, 1), (3, 100, 70, 65)])
def test_gradient_through_blocks_of_any_size(pattern):
    """Transposes element by element (few elements, small and thin blocks) and in squares, at both sides of the rule's lines,
    and more blocks than a launch may have workgroups of 256: against the products in float64, one row, whole numbers."""
    from ksmm_amd import Kernel

    a, b, c, d = pattern
    gen = torch.Generator(device="cuda").manual_seed(1)
    w, g = (torch.randint(-1, 2, s, generator=gen, device="cuda").half() for s in ((a * d * c, b), (1, a * b * d)))
    dx, _ = Kernel.backward(g, torch.empty(1, a * c * d, device="cuda").half(), w, False, a, b, c, d, need_weight=False)
    gd = g.view(a, b, d).permute(0, 2, 1).double()
    for k in range(0, c, 99):  # dx[a, c, d] = sum over b of w[a, d, c, b] g[a, b, d], at most 700
        want = (w.view(a, d, c, b)[:, :, k].double() * gd).sum(-1)
        assert torch.equal(dx.view(a, c, d)[:, k].double(), want), (pattern, k)
