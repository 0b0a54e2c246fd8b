"""Two factors in one launch (ksmm_pair.hip) against the layer's dense product in float64: edges of the batch tiles of 16 and
32, output tiles filled in part, strides of one to four and of several groups, several blocks of the second factor, and
whole and ragged rows in either layout.

Tolerances are those of the other chain tests: fp32 1e-5; fp16 2e-3 (each factor rounds to 2^-11); e4m3 5e-3 against the
oracle on the dequantised operands."""
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
