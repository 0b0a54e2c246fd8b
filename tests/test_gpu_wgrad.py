"""Weight gradients at the edges of their kernels: the batch-size-first kernel (ksmm_wgrad_bf.hip) and
the batch-size-last ones on rows of any length and alignment, against float64 products of the values
the device holds.

Tolerance: a gradient is a sum of n products rounded once to its type; the fp32 accumulation is off by
at most n * 2^-24 of the sum of the magnitudes, sqrt(n) * 2^-24 for inputs of random sign, so for
n <= 4200 the relative Frobenius error is below 1e-5 in fp32 and that of the last rounding, 2^-11 at
most, in fp16."""
import pytest
import torch

pytestmark = pytest.mark.gpu

TOL = {torch.float32: 1e-5, torch.float16: 5e-4}

# block edges of 16, 32, 48 and 64 and one more; d of one pass (1 .. 8) and in eights with an overlap (9,
# 12); blocks shared by a workgroup with a remainder; one row, one slab, a ragged one, several splits
CASES = [((1, 16, 16, 64), 130), ((5, 16, 9, 1), 333), ((3, 17, 33, 1), 64), ((7, 32, 20, 3), 129), ((1, 48, 144, 5), 1),
         ((2, 65, 64, 2), 31), ((1, 64, 129, 7), 97), ((2, 40, 24, 9), 261), ((1, 70, 130, 12), 40), ((1, 192, 64, 8), 515),
         ((3, 64, 64, 1), 4197), ((1, 451, 64, 1), 77), ((2, 130, 260, 4), 1030), ((1, 3, 500, 1), 50), ((1, 128, 128, 1), 3),
         ((1, 128, 256, 2), 777), ((2, 48, 48, 3), 2003)]


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("bs_last", [False, True])
@pytest.mark.parametrize("offset", [0, 1])
def test_weight_gradient_edges(dt, bs_last, offset):
    """``offset``: the operands start one element behind a 16-byte boundary."""
    from ksmm_amd import Kernel

    gen = torch.Generator(device="cuda").manual_seed(5)
    for (a, b, c, d), n in CASES:
        def tensor(features):
            t = torch.randn(offset + features * n, generator=gen, device="cuda").to(dt)[offset:]
            return t.view(features, n) if bs_last else t.view(n, features)

        x, dy = tensor(a * c * d), tensor(a * b * d)
        factor = torch.zeros(a * c * d, b, device="cuda", dtype=dt)
        got = Kernel.backward(dy, x, factor, bs_last, a, b, c, d, scale=0.5, need_input=False)[1]
        xs, ys = (x, dy) if bs_last else (x.t(), dy.t())
        xs = xs.double().reshape(a, c, d, n).permute(0, 2, 1, 3).reshape(a * d, c, n)
        ys = ys.double().reshape(a, b, d, n).permute(0, 2, 3, 1).reshape(a * d, n, b).contiguous()
        want = 0.5 * torch.bmm(xs, ys).reshape(a * d * c, b)
        err = ((got.double() - want).norm() / want.norm()).item()
        assert err <= TOL[dt], ((a, b, c, d), n, err)


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("d", [5, 6, 8, 11])
def test_weight_gradient_slab_counts(dt, d):
    """Workgroups of five to eight waves on 64 x 64 tiles hold two slabs (32 rows in fp16, 16 in fp32): none, one, an odd
    and an even number of whole ones, a remainder of one row."""
    from ksmm_amd import Kernel

    gen = torch.Generator(device="cuda").manual_seed(6)
    a, b, c = 2, 64, 80
    for n in (1, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 96, 97, 129, 160):
        x, dy = (torch.randn(n, a * s * d, generator=gen, device="cuda").to(dt) for s in (c, b))
        factor = torch.zeros(a * c * d, b, device="cuda", dtype=dt)
        got = Kernel.backward(dy, x, factor, False, a, b, c, d, need_input=False)[1]
        xs = x.t().double().reshape(a, c, d, n).permute(0, 2, 1, 3).reshape(a * d, c, n)
        ys = dy.t().double().reshape(a, b, d, n).permute(0, 2, 3, 1).reshape(a * d, n, b).contiguous()
        want = torch.bmm(xs, ys).reshape(a * d * c, b)
        err = ((got.double() - want).norm() / want.norm()).item()
        assert err <= TOL[dt], (n, err)


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", [(1, 128, 64, 2), (2, 64, 128, 1), (1, 120, 250, 1), (3, 17, 40, 3)])
def test_weight_gradient_slabs_batch_last(dt, shape):
    """Each tile of the batch-size-last GEMM kernel on no more than its first slab (64 columns in fp16, 32 in fp32), whole and
    ragged ones behind it, and several splits whose last one is short; rows that hold one vector only."""
    from ksmm_amd import Kernel

    gen = torch.Generator(device="cuda").manual_seed(8)
    a, b, c, d = shape
    for n in (4, 8, 9, 31, 32, 33, 63, 64, 65, 127, 128, 129, 130, 192, 200, 1025, 3001):
        x, dy = (torch.randn(a * s * d, n, generator=gen, device="cuda").to(dt) for s in (c, b))
        factor = torch.zeros(a * c * d, b, device="cuda", dtype=dt)
        got = Kernel.backward(dy, x, factor, True, a, b, c, d, need_input=False)[1]
        xs = x.double().reshape(a, c, d, n).permute(0, 2, 1, 3).reshape(a * d, c, n)
        ys = dy.double().reshape(a, b, d, n).permute(0, 2, 3, 1).reshape(a * d, n, b).contiguous()
        want = torch.bmm(xs, ys).reshape(a * d * c, b)
        err = ((got.double() - want).norm() / want.norm()).item()
        assert err <= TOL[dt], (n, err)


@pytest.mark.parametrize("d", [1, 2, 3, 4, 6])
def test_weight_gradient_wide(d):
    """Batch-size-first fp16 blocks of 48 and more (ksmm_wgrad_wide.hip): tiles of 64 and 128 filled and in part, no whole slab, whole
    ones and a remainder of one row, one split and several."""
    from ksmm_amd import Kernel

    gen = torch.Generator(device="cuda").manual_seed(8)
    for a, b, c in ((1, 64, 64), (3, 48, 56), (2, 128, 72), (1, 72, 128), (1, 200, 136), (5, 64, 192), (1, 520, 264)):
        for n in (1, 32, 63, 64, 65, 97, 129, 1025, 1100, 2304) if b * c < 20000 else (64, 1031, 4000):
            x, dy = (torch.randn(n, a * s * d, generator=gen, device="cuda").half() for s in (c, b))
            factor = torch.zeros(a * c * d, b, device="cuda", dtype=torch.float16)
            got = Kernel.backward(dy, x, factor, False, a, b, c, d, scale=0.5, need_input=False)[1]
            xs = x.t().double().reshape(a, c, d, n).permute(0, 2, 1, 3).reshape(a * d, c, n)
            ys = dy.t().double().reshape(a, b, d, n).permute(0, 2, 3, 1).reshape(a * d, n, b).contiguous()
            want = 0.5 * torch.bmm(xs, ys).reshape(a * d * c, b)
            err = ((got.double() - want).norm() / want.norm()).item()
            assert err <= TOL[torch.float16], ((a, b, c, d), n, err)


def test_weight_gradient_wide_bytes():
    """Rows behind a split's end and features behind a block's do not reach the sums: infinities there would."""
    from ksmm_amd import Kernel

    a, b, c, d, n = 2, 72, 56, 2, 1100
    gen = torch.Generator(device="cuda").manual_seed(9)
    rows = [torch.full((n + 200, a * s * d), float("inf"), device="cuda", dtype=torch.float16) for s in (c, b)]
    for r in rows:
        r[:n] = torch.randn(n, r.shape[1], generator=gen, device="cuda").half()
        r[:n].view(n, a, -1)[:, 1] = float("inf")  # the second block: its own gradient only
    factor = torch.zeros(a * c * d, b, device="cuda", dtype=torch.float16)
    got = Kernel.backward(rows[1][:n], rows[0][:n], factor, False, a, b, c, d, need_input=False)[1].view(a, -1)
    assert bool(got[0].isfinite().all()) and not bool(got[1].isfinite().any())


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("shape", [(2, 128, 64, 1), (2, 72, 130, 1), (1, 64, 192, 2), (2, 16, 16, 1), (1, 12, 9, 2), (2, 32, 32, 1), (1, 17, 30, 2),
                                   (2, 33, 32, 1)])
def test_weight_gradient_rows_end_where_the_batch_does(dt, shape):
    """Batch-size-last rows that no vector divides: what a vector reaches of the next row, and what a slab reaches of the next split, does
    not get into the sums: infinities there would."""
    from ksmm_amd import Kernel

    a, b, c, d = shape
    gen = torch.Generator(device="cuda").manual_seed(10)
    for n in (9, 33, 65, 130, 1025, 3001):
        pair = []
        for s in (c, b):
            t = torch.randn(a, s, d, n, generator=gen, device="cuda").to(dt)
            (t[1] if a == 2 else t[:, :, 1]).fill_(float("inf"))  # the other block: its rows lie behind (d = 2: between) the finite ones
            pair.append(t.view(a * s * d, n))
        factor = torch.zeros(a * c * d, b, device="cuda", dtype=dt)
        got = Kernel.backward(pair[1], pair[0], factor, True, a, b, c, d, need_input=False)[1].view(2, c, b)
        xs, ys = (t.view(a, s, d, n)[0, :, 0].double() for t, s in zip(pair, (c, b)))
        want = xs @ ys.t()
        assert ((got[0].double() - want).norm() / want.norm()).item() <= TOL[dt], n
        assert not bool(got[1].isfinite().any())
