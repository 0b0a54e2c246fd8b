"""A layer's backward pass in one call (ksmm_layer_backward) against one call per factor and epilogue, which the
same kernels serve: the same bits; and against float64.  The shapes are the edges of what the one call adds, the transposes and the sums
of a whole layer in one launch: blocks below, at and above a 64 x 64 square, products a x b x c x d that four does
not divide, few and many partial sums, and every set of wanted gradients."""
import ctypes
import itertools
import threading

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


def watched(monkeypatch):
    """The native module with a record of what its training calls returned: None would mean the route of single calls."""
    native, seen = _lib.native(), []
    assert native is not _lib._NoNative

    class Watch:
        infer = staticmethod(native.infer)

        @staticmethod
        def train_forward(*args):
            seen.append(native.train_forward(*args))
            return seen[-1]

        @staticmethod
        def train_backward(*args):
            seen.append(native.train_backward(*args))
            return seen[-1]

    monkeypatch.setattr(_lib, "_native", Watch)
    return seen


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("bs_last", [False, True])
@pytest.mark.parametrize("act", [None, "gelu"])
def test_layer_gradients_equal_those_of_single_calls(dt, bs_last, act, monkeypatch):
    from ksmm_amd import KSLinear

    seen = watched(monkeypatch)
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
                seen.clear()
                z = layer(x)
                assert torch.equal(z, y)
                for got, ref in zip(torch.autograd.grad(z, args, g), want):
                    assert got.shape == ref.shape and torch.equal(got, ref), (patterns, wanted)
                assert len(seen) == 2 and None not in seen, (patterns, wanted)


# Errors of the sums in fp32 (a sum over the batch: up to 1e-6) and of results, intermediates and gradients that are rounded to
# fp16 up to five times on the way (5 x 2^-11)
TOL = {torch.float32: 1e-5, torch.float16: 2.5e-3}


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("bs_last", [False, True])
@pytest.mark.parametrize("act", [None, "gelu"])
def test_layer_gradients_against_float64(dt, bs_last, act, monkeypatch):
    """From two threads on a stream of their own each, with the inputs made there."""
    from ksmm_amd import KSLinear

    seen, errors = watched(monkeypatch), []

    def step(k):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for patterns, n in CASES[k::2]:
                    weights = [(torch.rand(p) * 2 - 1) / p[2] ** 0.5 for p in patterns]
                    layer = KSLinear(patterns, weights=weights, algo="kernel", dtype=dt, bs_last=bs_last, device="cuda", act=act)
                    x = torch.randn((layer.in_size, n) if bs_last else (n, layer.in_size), device="cuda").to(dt).requires_grad_(True)
                    y = layer(x)
                    g = torch.randn_like(y)
                    got = torch.autograd.grad(y, [x, layer.bias, *layer.factors], g)
                    xd = x.detach().double().cpu().requires_grad_(True)
                    bias = layer.bias.detach().double().cpu().requires_grad_(True)
                    fs = [f.detach().double().cpu().requires_grad_(True) for f in layer.factors]
                    h = xd if bs_last else xd.T
                    for f, (a, b, c, d) in zip(fs, patterns):
                        h = torch.einsum("adcb,acdn->abdn", f.view(a, d, c, b), h.reshape(a, c, d, n)).reshape(a * b * d, n)
                    z = h + bias.view(-1, 1)
                    z = torch.nn.functional.gelu(z) if act else z
                    z = z if bs_last else z.T
                    want = torch.autograd.grad(z, [xd, bias, *fs], g.double().cpu())
                    for u, v in zip((y.detach(), *got), (z.detach(), *want)):
                        err = ((u.double().cpu() - v).norm() / v.norm()).item()
                        assert err <= TOL[dt], (patterns, u.shape, err)
        except BaseException as e:
            errors.append(e)

    threads = [threading.Thread(target=step, args=(k,)) for k in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    assert len(seen) == 2 * len(CASES) and None not in seen


@pytest.mark.parametrize("bs_last", [0, 1])
def test_layer_backward_through_the_library(bs_last):
    """The C entry point itself: its status, gradients that are not wanted, and a workspace that is a byte short."""
    from ksmm_amd import Kernel
    from ksmm_amd.kernel import dtype_code

    lib, patterns, n, dt = _lib.load(), [(2, 64, 64, 1), (1, 65, 128, 1)], 515, torch.float32
    made = lambda *shape: torch.randn(shape, device="cuda", dtype=dt)
    ws = [made(a * c * e, b) for a, b, c, e in patterns]
    shape = lambda f: (f, n) if bs_last else (n, f)
    x, dy = made(*shape(128)), made(*shape(65))
    mid = Kernel.forward(x, ws[0], bool(bs_last), *patterns[0])
    d = (_lib.KsmmFactorDesc * 2)()
    for i, (a, b, c, e) in enumerate(patterns):
        d[i].w, d[i].a, d[i].b, d[i].c, d[i].d, d[i].w_dtype, d[i].scale = ws[i].data_ptr(), a, b, c, e, dtype_code(dt), 1.0
    need = lib.ksmm_layer_backward_workspace(d, 2, n, dtype_code(dt), bs_last, _lib.ACT_NONE)
    room = torch.empty(need, dtype=torch.uint8, device="cuda")
    pointers = lambda *ts: (ctypes.c_void_p * 2)(*(t.data_ptr() if t is not None else None for t in ts))
    dx, dw0, dw1, dbias = torch.empty_like(x), torch.empty_like(ws[0]), torch.empty_like(ws[1]), made(65)
    call = lambda to_x, dws, to_bias, size: lib.ksmm_layer_backward(
        d, 2, pointers(x, mid), None, dy.data_ptr(), to_x, dws, to_bias, room.data_ptr(), size, n, dtype_code(dt), bs_last, _lib.ACT_NONE,
        torch.cuda.current_stream().cuda_stream)
    assert call(dx.data_ptr(), pointers(dw0, dw1), dbias.data_ptr(), need - 1) == -9
    assert call(dx.data_ptr(), pointers(dw0, dw1), dbias.data_ptr(), need) == 0
    g1, want1 = Kernel.backward(dy, mid, ws[1], bool(bs_last), *patterns[1])
    g0, want0 = Kernel.backward(g1, x, ws[0], bool(bs_last), *patterns[0])
    assert torch.equal(dx, g0) and torch.equal(dw0, want0) and torch.equal(dw1, want1)
    assert ((dbias - dy.sum(1 if bs_last else 0)).norm() / dbias.norm()).item() <= 1e-5
    for t in (dx, dw0, dw1):
        t.fill_(7.0)
    assert call(None, pointers(dw0, None), None, need) == 0
    assert torch.equal(dw0, want0) and bool((dx == 7).all()) and bool((dw1 == 7).all())


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
