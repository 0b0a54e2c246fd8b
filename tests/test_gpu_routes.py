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


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("bs_last", [False, True])
def test_unaligned_tensors_between_aligned_ones(dt, bs_last):
    """The choice is remembered by sizes and by whether the tensors start on 16 bytes: calls of both kinds in
    turn get their own each time, whichever tensor is off, and agree with float64."""
    from ksmm_amd import Kernel
    from ksmm_amd.layer import from_kernel_format_to_dense

    gen = torch.Generator(device="cuda").manual_seed(6)
    for (a, b, c, d), batch in [((1, 96, 48, 2), 200), ((2, 64, 64, 1), 33), ((1, 3, 5, 4), 77), ((1, 256, 256, 2), 8200)]:
        def tensor(rows, cols, off):
            t = torch.empty(rows * cols + 1, device="cuda", dtype=dt)[off:off + rows * cols].view(rows, cols)
            return t.copy_(torch.randn(rows, cols, generator=gen, device="cuda"))

        w, x = [tensor(a * d * c, b, off) for off in (0, 1)], [tensor(*((a * c * d, batch) if bs_last else (batch, a * c * d)), off) for off in (0, 1)]
        w[1].copy_(w[0])
        x[1].copy_(x[0])
        k = from_kernel_format_to_dense(w[0].double(), (a, b, c, d))
        want = k @ x[0].double() if bs_last else x[0].double() @ k.t()
        bits = {}
        for _ in range(2):
            for i, j in ((0, 0), (1, 0), (0, 1), (1, 1)):
                y = Kernel.forward(x[i], w[j], bs_last, a, b, c, d)
                # sums of c products of type dt in fp32, one rounding: 2e-7 sqrt(c) in fp32, 2.9e-4 in fp16
                assert ((y.double() - want).norm() / want.norm()).item() <= (5e-6 if dt == torch.float32 else 4e-4)
                assert torch.equal(y, bits.setdefault((i, j), y)), (i, j)


@pytest.mark.parametrize("dts", [(torch.float32, torch.float32), (torch.float16, torch.float16), (torch.float8_e4m3fn, torch.float8_e4m3fn),
                                 (torch.float16, torch.float8_e4m3fn)])
@pytest.mark.parametrize("bs_last", [False, True])
def test_equal_rows_have_equal_bits(dts, bs_last):
    """A row's result does not depend on where in the batch it lies: every tile sums in the same order."""
    from ksmm_amd import Kernel

    gen = torch.Generator(device="cuda").manual_seed(7)
    # wide groups of blocks first, then a shape per family
    for a, b, c, d in [(1, 192, 192, 64), (2, 128, 128, 32), (1, 256, 64, 16), (1, 48, 48, 16), (3, 64, 64, 1), (1, 768, 192, 2), (1, 128, 128, 3),
                       (2, 96, 96, 4), (1, 64, 256, 6), (4, 192, 192, 1), (1, 100, 36, 1), (3, 4, 4, 16), (16, 16, 16, 4), (1, 451, 64, 1)]:
        w = (torch.randn(a * d * c, b, generator=gen, device="cuda") / c ** 0.5).to(dts[1])
        row = torch.randn(a * c * d, generator=gen, device="cuda").to(dts[0])
        for n in (33, 197, 1000, 2050, 8192):
            x = torch.empty((a * c * d, n) if bs_last else (n, a * c * d), device="cuda", dtype=dts[0])
            x.copy_(row[:, None] if bs_last else row)
            y = Kernel.forward(x, w, bs_last, a, b, c, d)
            assert bool((y == (y[:, :1] if bs_last else y[:1])).all()), (a, b, c, d, n)
