"""Which kernels calls take that need no other one: results have the bits of the same call's usual kernel."""
import pytest
import torch

pytestmark = pytest.mark.gpu


# one shape per family and layout at full batches (and below): GEMM, stream, wave, rows, d > 1 tiles, k-loop, generic
@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("bs_last", [False, True])
@pytest.mark.parametrize("batch", [200, 8192])
def test_bias_needs_the_alignment_of_its_elements(dt, bs_last, batch):
    from ksmm_amd import Kernel

    gen = torch.Generator(device="cuda").manual_seed(5)
    for a, b, c, d in [(1, 1536, 384, 2), (4, 256, 64, 1), (6, 64, 64, 1), (1, 48, 48, 16), (1, 384, 384, 4), (1, 100, 36, 1),
                       (3, 4, 4, 16)]:
        x = torch.randn((a * c * d, batch) if bs_last else (batch, a * c * d), generator=gen, device="cuda").to(dt)
        w = torch.randn(a * d * c, b, generator=gen, device="cuda").to(dt)
        flat = torch.randn(a * b * d + 3, generator=gen, device="cuda").to(dt)
        for act in (None, "gelu"):
            for offset in (1, 2, 3):
                bias = flat[offset:offset + a * b * d]
                got = Kernel.forward(x, w, bs_last, a, b, c, d, bias=bias, act=act)
                assert torch.equal(got, Kernel.forward(x, w, bs_last, a, b, c, d, bias=bias.clone(), act=act)), (a, b, c, d, offset)
