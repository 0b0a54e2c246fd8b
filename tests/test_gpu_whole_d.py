"""Batch-size-first tiles that take all of d = 2, 3, 4 or 6 at once, at batches around their tiles, with blocks that fill their tiles of
outputs and blocks that do not, and with bias and GELU, against float64; every instance of the library is one of those run.

Tolerances: fp32 1e-5, fp16 and e4m3 operands 2e-3 (one rounding of the result to 2^-11; the operands are exact and the sums
fp32)."""
import ctypes
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn


PATTERNS = [(2, 192, 64, 3), (1, 32, 32, 3), (3, 80, 96, 3), (1, 144, 128, 3), (2, 64, 48, 6), (3, 128, 32, 6), (1, 208, 16, 6),
            (2, 128, 64, 2), (1, 208, 96, 2), (2, 64, 64, 4), (1, 144, 32, 4), (1, 256, 32, 3), (1, 192, 32, 2)]


@pytest.mark.parametrize("dts", [(torch.float32, torch.float32), (torch.float16, torch.float16), (FP8, FP8)])
@pytest.mark.parametrize("pattern", PATTERNS)
def test_whole_d(dts, pattern):
    from ksmm_amd import Kernel, _lib
    from ksmm_amd._lib import KsmmError
    from ksmm_amd.kernel import query_tile

    (a, b, c, d), (xt, wt) = pattern, dts
    w = (torch.rand(a * d * c, b, device="cuda") * 2 - 1).div(math.sqrt(c)).to(wt)
    wk = w.float().double().view(a, d, c, b)
    seen = set()
    for n in (1, 33, 63, 64, 65, 127, 129, 515):
        x = torch.randn(n, a * c * d, device="cuda").to(xt)
        flat = torch.full((a * b * d * n + 64,), 7.0, device="cuda", dtype=torch.float32 if xt == torch.float32 else torch.float16)
        y = flat[:a * b * d * n].view(n, a * b * d)
        xk = x.float().double().view(n, a, c, d)
        want = torch.stack([torch.stack([xk[:, i, :, j].contiguous() @ wk[i, j] for j in range(d)], -1) for i in range(a)], 1)
        want = want.reshape(n, -1)
        for i in range(128):
            variant = 3 << 24 | i
            try:
                tile = query_tile(n, pattern, xt, wt, False, _lib.ALGO_TILE, variant)
            except KsmmError:
                continue
            if tile["tile_d"] != d:
                continue
            seen.add(i)
            flat.fill_(7.0)
            Kernel.forward(x, w, False, a, b, c, d, out=y, algo=_lib.ALGO_TILE, variant=variant)
            err = ((y.double() - want).norm() / want.norm()).item()
            assert err <= (1e-5 if xt == torch.float32 else 2e-3), (n, i, err)
            assert bool((flat[a * b * d * n:] == 7.0).all())
    # (fp16 has other tiles for d = 2 and 4; fp32 with d = 2 and 6 takes full tiles only)
    takes = {torch.float16: d in (3, 6), torch.float32: d == 3 or b % 64 == 0, FP8: True}[xt]
    assert seen or not takes or c % (16 if d == 6 else 32)


def test_every_whole_d_instance_takes_one_of_the_patterns():
    """The patterns above reach all of these tiles, each with outputs that fill its last tile and outputs that do not where it takes both."""
    from ksmm_amd import _lib
    from ksmm_amd._lib import KsmmError
    from ksmm_amd.kernel import query_tile

    whole = _lib.load()["_ZN4ksmm13bf_inst_wholeEi"]
    whole.restype = ctypes.c_bool
    every, full, part = {i for i in range(128) if whole(i)}, set(), set()
    for dt in (torch.float32, torch.float16, FP8):
        for pattern in PATTERNS:
            for i in every:
                try:
                    t = query_tile(129, pattern, dt, dt, False, _lib.ALGO_TILE, 3 << 24 | i)
                except KsmmError:
                    continue
                assert t["tile_d"] == pattern[3]
                (part if pattern[1] % t["tile_m"] else full).add(i)
    assert len(every) >= 16 and full | part == every, every - full - part
    # (fp32 with d = 2 and 6 takes whole blocks of 64: their two tiles of 64 are never filled in part)
    assert full == every and len(every - part) == 2, (every - full, every - part)


@pytest.mark.parametrize("dt", [torch.float32, torch.float16, FP8])
def test_whole_d_epilogue(dt):
    """Bias and GELU of a layer whose factor the tiles take, and what they refuse: a stride or block off the vector."""
    from ksmm_amd import KSLinear, quantize_fp8

    for pattern in ((1, 192, 192, 3), (2, 80, 192, 3), (1, 72, 96, 3), (1, 100, 96, 3)):
        w4 = (torch.rand(pattern) * 2 - 1) / math.sqrt(pattern[2])
        layer = KSLinear([pattern], weights=[w4], algo="kernel", dtype=dt, device="cuda", act="gelu")
        dense = layer.get_dense_product(torch.float64)
        for n in (197, 1001):
            x = torch.randn(n, layer.in_size, device="cuda")
            x, scale = quantize_fp8(x) if dt == FP8 else (x.to(dt), None)
            with torch.no_grad():
                y = layer(x, x_scale=scale)
                z = x.double() * (float(scale) if scale is not None else 1.0) @ dense.T + layer.bias.double()
            want = z * 0.5 * (1 + torch.erf(z / math.sqrt(2)))
            assert ((y.double() - want).norm() / want.norm()).item() <= {torch.float32: 1e-5, torch.float16: 2e-3, FP8: 5e-3}[dt]


@pytest.mark.parametrize("dt", [torch.float32, torch.float16, FP8])
def test_whole_d_without_workspace_at_any_alignment(dt):
    """What asks for no workspace runs without one, on tensors that start an element behind 16 bytes as well, and writes nothing
    but its result; a chain on its intermediates alone."""
    from ksmm_amd import Kernel, KSLinear, _lib
    from ksmm_amd.kernel import dtype_code

    lib = _lib.load()
    yt = torch.float32 if dt == torch.float32 else torch.float16
    xd, yd, tol = dtype_code(dt), dtype_code(yt), 1e-5 if dt == torch.float32 else 2e-3
    for (a, b, c, d), n in [((1, 256, 256, 3), 2050), ((3, 80, 96, 3), 2051), ((2, 128, 32, 6), 2111), ((1, 192, 48, 2), 6304), ((2, 64, 256, 4), 4099)]:
        def tensor(size, off, dtype):
            return torch.empty(size + 64, device="cuda", dtype=dtype)[off:off + size]

        full_x = torch.randn(n * a * c * d, device="cuda").to(dt)
        full_w = ((torch.rand(a * d * c * b, device="cuda") * 2 - 1) / math.sqrt(c)).to(dt)
        xk, wk = full_x.float().double().view(n, a, c, d), full_w.float().double().view(a, d, c, b)
        want = torch.stack([torch.stack([xk[:, i, :, j].contiguous() @ wk[i, j] for j in range(d)], -1) for i in range(a)], 1).reshape(n, -1)
        need = lib.ksmm_factor_workspace(n, a, b, c, d, xd, xd, yd, 0)
        for offs in ((0, 0, 0), (1, 0, 0), (0, 1, 0), (0, 0, 1), (1, 3, 1)):
            x, w = tensor(full_x.numel(), offs[0], dt).copy_(full_x), tensor(full_w.numel(), offs[1], dt).copy_(full_w)
            flat = torch.full((want.numel() + 64,), 7.0, device="cuda", dtype=yt)
            y = flat[offs[2]:offs[2] + want.numel()]
            stream = torch.cuda.current_stream().cuda_stream
            rc = lib.ksmm_factor_forward_ws(x.data_ptr(), w.data_ptr(), y.data_ptr(), n, a, b, c, d, xd, xd, yd, 0, 1.0, None, 0, stream)
            assert rc == (0 if need == 0 else -9), (a, b, c, d, rc)
            if rc:
                continue
            err = ((y.view(n, -1).double() - want).norm() / want.norm()).item()
            assert err <= tol, ((a, b, c, d), offs, err)
            assert bool((flat[:offs[2]] == 7.0).all()) and bool((flat[offs[2] + want.numel():] == 7.0).all())
    if dt == FP8:
        return
    patterns, n = [(12, 64, 256, 1), (1, 256, 256, 3)], 2050
    layer = KSLinear(patterns, bias=False, algo="kernel", dtype=dt, device="cuda")
    flat = torch.randn(n * layer.in_size + 1, device="cuda").to(dt)
    for off in (0, 1):
        x = flat[off:off + n * layer.in_size].view(n, layer.in_size)
        with torch.no_grad():
            y = layer(x)
            want = x.double() @ layer.get_dense_product(torch.float64).t()
        assert ((y.double() - want).norm() / want.norm()).item() <= tol
