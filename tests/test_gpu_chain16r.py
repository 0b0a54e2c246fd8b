"""Radix-16 chains in one launch (ksmm_chain16r.hip) against the float64 oracle, at the edges of its chunks of 16 and 32
rows, for every type, layout, number of factors and power-of-two stride, and rows off the 16-byte grid.

Tolerances are those of the other chain tests: fp32 1e-5; fp16 2e-3 (each factor rounds to 2^-11); e4m3 5e-3 against the
oracle on the dequantised operands."""
import ctypes
import math

import pytest
import torch

from oracle import ks_oracle as O

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn
CHAINS = [[(1, 16, 16, 1)] * 2, [(1, 16, 16, 8), (2, 16, 16, 4), (4, 16, 16, 2), (8, 16, 16, 1)],
          [(3, 16, 16, 16), (48, 16, 16, 1)], [(1, 16, 16, 64), (16, 16, 16, 4), (64, 16, 16, 1)], [(2, 16, 16, 32), (32, 16, 16, 2)]]
TOL = {torch.float32: 1e-5, torch.float16: 2e-3, FP8: 5e-3}


def taken(layer, x, y):
    """Whether the one launch takes the layer on x as it is."""
    from ksmm_amd import _lib
    from ksmm_amd.kernel import dtype_code

    d = (_lib.KsmmFactorDesc * len(layer.patterns))()
    for i, (f, p) in enumerate(zip(layer.factors, layer.patterns)):
        d[i].w, d[i].w_dtype, d[i].scale = f.data_ptr(), dtype_code(f.dtype), layer.w_scales[i]
        d[i].a, d[i].b, d[i].c, d[i].d = p
    return _lib.load().ksmm_chain_forward_fused(d, len(layer.patterns), x.data_ptr(), y.data_ptr(), x.numel() // layer.in_size,
                                                dtype_code(x.dtype), dtype_code(y.dtype), int(layer.bs_last), None,
                                                torch.cuda.current_stream().cuda_stream) == 0


def expected(dt, bs_last, features, n):
    """The rule of fused_rows_pay (ksmm_api.hip) for tensors on 16 bytes."""
    if features < 256:
        return n <= 4096
    return not bs_last or dt != FP8 or n <= 8192 or n % 16 != 0  # else the chain has the kernel of whole vectors


@pytest.mark.parametrize("dt", [torch.float32, torch.float16, FP8])
@pytest.mark.parametrize("bs_last", [False, True])
def test_chain_edges(dt, bs_last):
    from ksmm_amd import KSLinear, quantize_fp8

    gen = torch.Generator(device="cuda").manual_seed(5)
    for k, patterns in enumerate(CHAINS):
        ws = [(torch.rand(p, generator=torch.Generator().manual_seed(k)) * 2 - 1) / 4 for p in patterns]
        layer = KSLinear(patterns, weights=ws, algo="kernel", dtype=dt, bs_last=bs_last, device="cuda", act="gelu" if k % 2 else None)
        dense = layer.get_dense_product(torch.float64).cpu()
        for n in (1, 15, 16, 17, 33, 197, 4096, 4097, 8192, 8193, 8208):
            x = torch.randn((layer.in_size, n) if bs_last else (n, layer.in_size), generator=gen, device="cuda")
            x, scale = quantize_fp8(x) if dt == FP8 else (x.to(dt), None)
            scale = None if scale is None else float(scale)
            with torch.no_grad():
                y = layer(x, x_scale=scale)
                assert taken(layer, x, torch.empty_like(y)) == expected(dt, bs_last, layer.in_size, n), (patterns, n)
            cols = torch.arange(n) if n <= 200 else torch.cat([torch.arange(40), torch.arange(n // 2, n // 2 + 40), torch.arange(n - 40, n)])
            xs = (x.double().cpu() * (scale or 1.0)).index_select(1 if bs_last else 0, cols)
            z = dense @ xs if bs_last else xs @ dense.T
            z = z + layer.bias.double().cpu()
            if layer.act:
                z = z * 0.5 * (1 + torch.erf(z / math.sqrt(2)))
            err = O.rel_fro_error(y.double().cpu().index_select(1 if bs_last else 0, cols).numpy(), z.detach().numpy())
            assert err <= TOL[dt], (patterns, n, err)


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
def test_chain_off_16_bytes(dt):
    """Batch-size-last tensors that start one element behind a boundary are taken, batch-size-first ones go elsewhere."""
    from ksmm_amd import KSLinear

    patterns = CHAINS[3]
    for bs_last in (True, False):
        layer = KSLinear(patterns, algo="kernel", dtype=dt, bs_last=bs_last, device="cuda")
        for n in (33, 64):
            flat = torch.randn(1024 * n + 1, device="cuda").to(dt)
            x = flat[1:].view((1024, n) if bs_last else (n, 1024))
            with torch.no_grad():
                y = layer(x)
                assert taken(layer, x, torch.empty_like(y)) == bs_last
                assert O.rel_fro_error(y.double().cpu().numpy(), layer(x.clone()).double().cpu().numpy()) <= TOL[dt]


def test_chain_that_is_not_one():
    """Strides that are no power of two, other block sizes and wider chains stay on their kernels."""
    from ksmm_amd import KSLinear

    for patterns in ([(1, 16, 16, 3), (3, 16, 16, 1)], [(1, 16, 16, 128), (128, 16, 16, 1)], [(1, 32, 32, 4), (4, 32, 32, 1)]):
        layer = KSLinear(patterns, algo="kernel", dtype=torch.float16, device="cuda")
        x = torch.randn(64, layer.in_size, device="cuda", dtype=torch.float16)
        with torch.no_grad():
            y = layer(x)
        assert not taken(layer, x, torch.empty_like(y))
        want = x.double() @ layer.get_dense_product(torch.float64).T + layer.bias.double()
        assert O.rel_fro_error(y.double().cpu().numpy(), want.detach().cpu().numpy()) <= 2e-3
