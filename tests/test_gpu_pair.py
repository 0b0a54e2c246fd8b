"""Two factors in one launch (ksmm_pair.hip) against the layer's dense product in float64: the shapes that layers choose by price, and
every shape by itself (batch tiles of 16 and 32, output tiles of 64 and 128 filled in part), strides of one to four and of several
groups, several blocks of the second factor, and whole and ragged rows in either layout.

Tolerances are those of the other chain tests: fp32 1e-5; fp16 2e-3 (each factor rounds to 2^-11); e4m3 5e-3 against the
oracle on the dequantised operands."""
import ctypes
import math

import pytest
import torch

from oracle import ks_oracle as O
from test_gpu_chain16r import FP8, TOL, taken

pytestmark = pytest.mark.gpu

CHAINS = [[(3, 64, 64, 1), (1, 384, 96, 2)], [(4, 48, 32, 1), (1, 80, 192, 1)], [(6, 64, 64, 1), (2, 64, 64, 3)],
          [(8, 16, 32, 1), (1, 64, 32, 4)], [(6, 32, 64, 1), (1, 48, 32, 6)], [(10, 32, 32, 1), (2, 112, 32, 5)]]


@pytest.mark.parametrize("dt", [torch.float32, torch.float16, FP8])
@pytest.mark.parametrize("bs_last", [False, True])
def test_pair_edges(dt, bs_last):
    from ksmm_amd import KSLinear, quantize_fp8

    gen = torch.Generator(device="cuda").manual_seed(7)
    ran = 0
    for k, patterns in enumerate(CHAINS):
        ws = [(torch.rand(p, generator=torch.Generator().manual_seed(k)) * 2 - 1) / math.sqrt(p[2]) for p in patterns]
        layer = KSLinear(patterns, weights=ws, algo="kernel", dtype=dt, bs_last=bs_last, device="cuda", act="gelu" if k % 2 else None)
        dense = layer.get_dense_product(torch.float64).cpu()
        for n in (1, 2, 15, 16, 17, 33, 196, 333):
            x = torch.randn((layer.in_size, n) if bs_last else (n, layer.in_size), generator=gen, device="cuda")
            x, scale = quantize_fp8(x) if dt == FP8 else (x.to(dt), None)
            scale = None if scale is None else float(scale)
            with torch.no_grad():
                y = layer(x, x_scale=scale)
            ran += taken(layer, x, torch.empty_like(y))
            z = dense @ (x.double().cpu() * (scale or 1.0)) if bs_last else (x.double().cpu() * (scale or 1.0)) @ dense.T
            z = z + layer.bias.double().cpu()
            if layer.act:
                z = z * 0.5 * (1 + torch.erf(z / math.sqrt(2)))
            err = O.rel_fro_error(y.double().cpu().numpy(), z.detach().numpy())
            assert err <= TOL[dt], (patterns, n, err)
    assert ran >= 24, ran  # (half of the calls: the others are priced lower on two launches)


# (beside those: planes and partial sums that do not fit the LDS together, which share it)
SHARED = [(32, 64, 32, 1), (1, 64, 512, 4)]


@pytest.mark.parametrize("dt", [torch.float32, torch.float16, FP8])
@pytest.mark.parametrize("bs_last", [False, True])
def test_pair_every_shape(dt, bs_last):
    """Each workgroup shape that the kernel takes a chain with, whatever it is priced at, through the library's own launcher: full and
    ragged batch tiles, odd feature-major rows of which two columns are written twice, bias and GELU, nothing written behind the end."""
    from ksmm_amd import KSLinear, _lib, quantize_fp8
    from ksmm_amd.kernel import dtype_code

    launch = _lib.load()["_ZN4ksmm8pair_runEPK16ksmm_factor_desciPKvPvliiiRKNS_9PairShapeEP12ihipStream_tPK13ksmm_epiloguePKf"]
    vp, i64, i32 = ctypes.c_void_p, ctypes.c_int64, ctypes.c_int
    launch.restype, launch.argtypes = i32, [vp, i32, vp, vp, i64, i32, i32, i32, vp, vp, vp, vp]
    gen = torch.Generator(device="cuda").manual_seed(8)
    seen, shared = set(), 0
    for k, patterns in enumerate(CHAINS + [SHARED]):
        ws = [(torch.rand(p, generator=torch.Generator().manual_seed(k)) * 2 - 1) / math.sqrt(p[2]) for p in patterns]
        layer = KSLinear(patterns, weights=ws, algo="kernel", dtype=dt, bs_last=bs_last, device="cuda", act="gelu" if k % 2 else None)
        dense, bias = layer.get_dense_product(torch.float64), layer.bias.double()
        d = (_lib.KsmmFactorDesc * 2)()
        for i, (f, p) in enumerate(zip(layer.factors, patterns)):
            d[i].w, d[i].w_dtype, d[i].scale = f.data_ptr(), dtype_code(f.dtype), layer.w_scales[i]
            d[i].a, d[i].b, d[i].c, d[i].d = p
        ep = _lib.KsmmEpilogue(layer.bias.data_ptr(), _lib.ACT_GELU if layer.act else _lib.ACT_NONE)
        d1, c1 = patterns[1][3], patterns[1][2]
        dg = d1 if d1 <= 4 else 4 if d1 % 4 == 0 else 3 if d1 % 3 == 0 else 2 if d1 % 2 == 0 else 1
        for n in (1, 2, 15, 31, 32, 33, 65):
            x = torch.randn((layer.in_size, n) if bs_last else (n, layer.in_size), generator=gen, device="cuda")
            x, scale = quantize_fp8(x) if dt == FP8 else (x.to(dt), None)
            xs = scale.float().cuda().reshape(1) if dt == FP8 else None
            x64 = x.float().double() * (float(scale) if dt == FP8 else 1.0)
            want = dense @ x64 + bias if bs_last else x64 @ dense.t() + bias
            if layer.act:
                want = want * 0.5 * (1 + torch.erf(want / math.sqrt(2)))
            for nt in (1, 2):
                for mg in (1, 2):
                    flat = torch.full((want.numel() + 64,), 7.0, device="cuda", dtype=layer.out_dtype)
                    rc = launch(d, 2, x.data_ptr(), flat.data_ptr(), n, dtype_code(x.dtype), dtype_code(flat.dtype), int(bs_last),
                                ctypes.byref((i32 * 2)(nt, mg)), torch.cuda.current_stream().cuda_stream, ctypes.byref(ep),
                                xs.data_ptr() if dt == FP8 else None)
                    if rc == -6:
                        assert (bs_last and n < nt) or patterns is SHARED, (patterns, n, nt, mg)
                        continue
                    assert rc == 0, rc
                    err = ((flat[:want.numel()].view(want.shape).double() - want).norm() / want.norm()).item()
                    assert err <= TOL[dt], (patterns, n, nt, mg, err)
                    assert bool((flat[want.numel():] == 7.0).all()), (patterns, n, nt, mg)
                    if patterns is SHARED:
                        shared += 1
                    else:
                        seen.add((nt, mg, dg))
    assert seen == {(nt, mg, dg) for nt in (1, 2) for mg in (1, 2) for dg in (1, 2, 3, 4)}, seen
    assert shared


def test_pair_takes_any_alignment_and_leaves_the_rest():
    """Tensors one element behind a 16-byte boundary give what aligned ones do; without `fuse` nothing is fused, and chains of
    another form go where they went."""
    from ksmm_amd import KSLinear

    patterns = CHAINS[0]
    for bs_last in (False, True):
        layer = KSLinear(patterns, algo="kernel", dtype=torch.float16, bs_last=bs_last, device="cuda")
        plain = KSLinear(patterns, algo="kernel", dtype=torch.float16, bs_last=bs_last, device="cuda", fuse=False)
        plain.load_state_dict(layer.state_dict())
        flat = torch.randn(layer.in_size * 33 + 1, device="cuda").half()
        x = flat[1:].view((layer.in_size, 33) if bs_last else (33, layer.in_size))
        with torch.no_grad():
            y = layer(x)
            assert taken(layer, x, torch.empty_like(y))
            assert torch.equal(y, layer(x.clone()))
            assert O.rel_fro_error(y.double().cpu().numpy(), plain(x).double().cpu().numpy()) <= TOL[torch.float16]
    for other in ([(1, 64, 64, 3), (3, 64, 64, 1)], [(3, 64, 64, 1), (1, 96, 64, 3), (3, 64, 96, 1)], [(2, 40, 64, 1), (1, 64, 40, 2)]):
        layer = KSLinear(other, algo="kernel", dtype=torch.float16, device="cuda")
        x = torch.randn(33, layer.in_size, device="cuda").half()
        with torch.no_grad():
            assert not taken(layer, x, layer(x))


def test_pair_in_a_graph_goes_by_the_gpus_time():
    """A call of its own may take the one launch to spare the host the other; a graph takes it only where it is priced below two, and
    its replays give what float64 gives, whichever it is."""
    from ksmm_amd import KSLinear

    up = [(6, 64, 64, 1), (1, 768, 192, 2)]
    for dt, bs_last, n, in_graph in ((torch.float32, True, 32, False), (torch.float16, False, 196, True), (torch.float16, False, 33, True)):
        layer = KSLinear(up, algo="kernel", dtype=dt, bs_last=bs_last, device="cuda")
        dense = layer.get_dense_product(torch.float64)
        x = torch.randn((layer.in_size, n) if bs_last else (n, layer.in_size), device="cuda").to(dt)
        side = torch.cuda.Stream()
        with torch.no_grad(), torch.cuda.stream(side):
            spare = torch.empty_like(layer(x))
            assert taken(layer, x, spare)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.no_grad(), torch.cuda.graph(graph):
            assert taken(layer, x, spare) == in_graph, (dt, bs_last, n)
            y = layer(x)
        for k in range(3):
            x.copy_(torch.randn(x.shape, device="cuda") * (k + 1))
            graph.replay()
            torch.cuda.synchronize()
            with torch.no_grad():
                eager = layer(x)
                bias = layer.bias.double()
                want = dense @ x.double() + bias if bs_last else x.double() @ dense.t() + bias
            for got in (y, eager):
                assert ((got.double() - want).norm() / want.norm()).item() <= TOL[dt], (dt, bs_last, n, k)
