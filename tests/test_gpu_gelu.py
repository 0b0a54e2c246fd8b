"""GELU in the far negative tail on the fp32 GEMM tiles (gelu_of in ksmm_gemm.hip): results there are small differences from
0, and in fp32 they are to be as exact as on every other kernel.

Tolerance: Abramowitz & Stegun 7.1.26 is off by at most 1.5e-7 / 2 in the tail, which is 4e-3 of the result at -6 (its worst on this
grid, evaluated in float32 steps, is 3.6e-3); 5e-3 leaves room for the hardware's exponential and reciprocal."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pattern,n", [((1, 256, 256, 3), 4096), ((1, 768, 192, 2), 4096), ((1, 1024, 1024, 1), 6272), ((1, 200, 512, 1), 6272)])
def test_far_tail_in_fp32(pattern, n):
    from ksmm_amd import Kernel, generate_factor
    from ksmm_amd.kernel import query_tile

    t = query_tile(n, pattern, torch.float32, torch.float32, True)
    assert (t["algo"], t["variant"] >> 24) == (3, 4), t  # a GEMM tile
    a, b, c, d = pattern
    w = generate_factor(a, b, c, d, "kernel", None, torch.float32, "cuda")
    z = torch.linspace(-6.0, -3.0, a * b * d, device="cuda")  # what the activation is applied to: x is 0
    y = Kernel.forward(torch.zeros(a * c * d, n, device="cuda"), w, True, a, b, c, d, bias=z, act="gelu")
    assert torch.equal(y, y[:, :1].expand_as(y))
    z = z.double().cpu()
    want = z * torch.special.erfc(-z / 2 ** 0.5) / 2
    assert ((y[:, 0].double().cpu() - want).abs() / want.abs()).max().item() <= 5e-3
