"""e4m3 chains with their weights decoded once (decode_pays in ksmm_api.hip) against the oracle and against the same
chain on a workspace without room for that; ragged batches, both layouts and an input that is quantised on the way.

Tolerance: 5e-3 against the oracle on the dequantised operands (fp16 intermediates and results); between the two
routes 1e-3, two such roundings of sums in another order."""
import ctypes

import pytest
import torch

from oracle import ks_oracle as O

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn
CASES = [([(3, 64, 256, 1), (1, 64, 64, 3)], False, 4800), ([(6, 64, 64, 1), (1, 768, 192, 2)], False, 10070),
         ([(6, 64, 64, 1), (1, 768, 192, 2)], True, 10080), ([(12, 64, 256, 1), (1, 256, 256, 3)], True, 10080),
         ([(12, 64, 256, 1), (1, 256, 256, 3)], False, 10070)]


@pytest.mark.parametrize("patterns,bs_last,n", CASES)
def test_decoded_weights(patterns, bs_last, n):
    from ksmm_amd import KSLinear, _lib, quantize_fp8
    from ksmm_amd.kernel import dtype_code

    lib = _lib.load()
    gen = torch.Generator(device="cuda").manual_seed(3)
    layer = KSLinear(patterns, algo="kernel", dtype=FP8, bs_last=bs_last, device="cuda", act="gelu")
    x = torch.randn((layer.in_size, n) if bs_last else (n, layer.in_size), generator=gen, device="cuda").half()
    codes, scale = quantize_fp8(x)
    d = (_lib.KsmmFactorDesc * len(patterns))()
    for i, (f, p) in enumerate(zip(layer.factors, patterns)):
        d[i].w, d[i].w_dtype = f.data_ptr(), dtype_code(f.dtype)
        d[i].scale = layer.w_scales[i] * (float(scale) if i == 0 else 1.0)
        d[i].a, d[i].b, d[i].c, d[i].d = p
    xd, yd = dtype_code(FP8), _lib.KSMM_F16
    asked = lib.ksmm_chain_workspace_layout(d, len(patterns), n, xd, yd, int(bs_last))
    weights = sum(a * b * c * e for a, b, c, e in patterns[1:])
    ep = _lib.KsmmEpilogue(bias=layer.bias.data_ptr(), act=_lib.ACT_GELU)
    out = []
    for ws_bytes in (asked, asked - 2 * weights):
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device="cuda")
        y = torch.empty((layer.out_size, n) if bs_last else (n, layer.out_size), dtype=torch.float16, device="cuda")
        rc = lib.ksmm_chain_forward_ep(d, len(patterns), codes.data_ptr(), y.data_ptr(), ws.data_ptr(), ws_bytes, n, xd, yd, int(bs_last),
                                       1, ctypes.byref(ep), torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        out.append(y.double())
    assert O.rel_fro_error(out[0].cpu().numpy(), out[1].cpu().numpy()) <= 1e-3
    with torch.no_grad():
        assert torch.equal(layer(codes, x_scale=float(scale)).double(), out[0])
        assert torch.equal(layer(x).double(), out[0])  # quantised on the way: the same codes and scale
    cols = torch.cat([torch.arange(40), torch.arange(n - 40, n)])
    xs = codes.float().double().cpu().index_select(1 if bs_last else 0, cols) * float(scale)
    dense = layer.get_dense_product(torch.float64).cpu()
    z = (dense @ xs if bs_last else xs @ dense.T) + layer.bias.detach().double().cpu()
    z = torch.nn.functional.gelu(z)
    assert O.rel_fro_error(out[0].cpu().index_select(1 if bs_last else 0, cols).numpy(), z.numpy()) <= 5e-3


def test_room_for_decoded_weights_is_asked_for_where_it_pays():
    from ksmm_amd import _lib

    lib = _lib.load()
    d = (_lib.KsmmFactorDesc * 2)()
    for i, (a, b, c, e) in enumerate([(6, 64, 64, 1), (1, 768, 192, 2)]):
        d[i].a, d[i].b, d[i].c, d[i].d, d[i].w_dtype, d[i].scale = a, b, c, e, _lib.KSMM_FP8_E4M3, 1.0
    need = lambda n: lib.ksmm_chain_workspace_layout(d, 2, n, _lib.KSMM_FP8_E4M3, _lib.KSMM_F16, 1)
    plain = lambda n: lib.ksmm_chain_workspace(d, 2, n, _lib.KSMM_F16)
    assert need(64) == plain(64)
    assert need(25088) == plain(25088) + 2 * 768 * 192 * 2


def test_the_entry_point_with_its_own_scratch_takes_what_it_took():
    """Up to what the chain alone needs, with room for decoded weights or without; beyond that it is refused."""
    from ksmm_amd import KSLinear, _lib
    from ksmm_amd.kernel import dtype_code

    lib = _lib.load()
    patterns = [(6, 64, 64, 1), (1, 768, 192, 2)]
    layer = KSLinear(patterns, algo="kernel", dtype=FP8, bs_last=True, device="cuda", bias=False)
    d = (_lib.KsmmFactorDesc * 2)()
    for i, (f, p) in enumerate(zip(layer.factors, patterns)):
        d[i].w, d[i].w_dtype, d[i].scale = f.data_ptr(), dtype_code(f.dtype), layer.w_scales[i]
        d[i].a, d[i].b, d[i].c, d[i].d = p
    xd, yd, room = dtype_code(FP8), _lib.KSMM_F16, lib.ksmm_static_scratch_bytes()
    most = max(n for n in range(16, 1 << 16, 16) if lib.ksmm_chain_workspace(d, 2, n, yd) <= room)
    asked = lambda n: lib.ksmm_chain_workspace_layout(d, 2, n, xd, yd, 1)
    assert asked(20000) <= room < asked(most)
    stream = torch.cuda.current_stream().cuda_stream
    for n, rc in ((20000, 0), (most, 0), (most + 16, -9)):
        codes = torch.randn(layer.in_size, n, device="cuda").to(FP8)
        y = torch.empty(layer.out_size, n, dtype=torch.float16, device="cuda")
        assert lib.ksmm_chain_forward_static(d, 2, codes.data_ptr(), y.data_ptr(), n, xd, yd, 1, 1, None, stream) == rc
        if rc == 0:
            with torch.no_grad():
                want = layer(codes, x_scale=1.0)
            assert O.rel_fro_error(y.double().cpu().numpy(), want.double().cpu().numpy()) <= 1e-3
