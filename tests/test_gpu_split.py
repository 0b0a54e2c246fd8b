"""The split-K tiles (any b >= 4, c, d, batch and alignment) against the float64 oracle, and what the
automatic choice does with batches off the vector and below the measured table."""
import pytest
import torch

from tests.util import TOL, TORCH_DTYPE, round_to, seeded_input, seeded_weights
from oracle import ks_oracle as O

# remainders of the 64 (32) x 16 NT tile, of the 32 (16) input step and of four outputs per lane;
# d of every group width, alone and as a divisor
PATTERNS = [(1, 4, 4, 1), (2, 5, 7, 3), (3, 66, 33, 2), (2, 64, 64, 1), (1, 16, 16, 8), (2, 50, 40, 4),
            (1, 130, 72, 6), (1, 33, 200, 8), (2, 7, 1, 5), (1, 64, 96, 12), (2, 68, 32, 2), (1, 36, 24, 16), (1, 64, 520, 3)]
BATCHES = (1, 3, 16, 33, 67, 130)


def _operands(pattern, batch, prec, bs_last):
    """(input, factor, scale, oracle result); ``mix``: e4m3 weights on fp16 input."""
    from ksmm_amd import generate_factor

    a, b, c, d = pattern
    (w4,) = seeded_weights([pattern], seed=7)
    x = seeded_input(a * c * d, batch, bs_last, seed=8)
    wp, xp = ("fp8" if prec in ("fp8", "mix") else prec), ("fp16" if prec == "mix" else prec)
    wr, wq, ws = round_to(w4, wp)
    xr, xq, xs = round_to(x, xp)
    fac = generate_factor(a, b, c, d, "kernel", wq.float() if wq is not None else w4, TORCH_DTYPE[wp], "cuda")
    xin = (xq if xq is not None else x.to(TORCH_DTYPE[xp])).cuda()
    return xin, fac, (ws or 1.0) * (xs or 1.0), O.ks_apply_einsum(wr, xr, bs_last)


def _error(y, z):
    return O.rel_fro_error(y.float().cpu().numpy(), z)


@pytest.mark.gpu
@pytest.mark.parametrize("bs_last", [True, False])
@pytest.mark.parametrize("prec", ["fp32", "fp16", "fp8", "mix"])
def test_split_tiles_forced(prec, bs_last):
    from ksmm_amd import Kernel, _lib

    ran = set()
    for pattern in PATTERNS:
        for batch in BATCHES:
            xin, fac, scale, z = _operands(pattern, batch, prec, bs_last)
            for inst in range(80):
                for waves in (1, 3, 16):
                    try:
                        y = Kernel.forward(xin, fac, bs_last, *pattern, scale=scale, algo=3,
                                           variant=(5 << 24) | (waves << 8) | inst)
                    except _lib.KsmmError as e:
                        assert e.status == -6
                        continue
                    ran.add(inst)
                    assert _error(y, z) <= TOL.get(prec, TOL["fp8"]), (prec, bs_last, pattern, batch, inst, waves)
    assert len(ran) == (3 if bs_last else 17), sorted(ran)


@pytest.mark.gpu
@pytest.mark.parametrize("bs_last", [True, False])
@pytest.mark.parametrize("prec", ["fp32", "fp16", "fp8"])
def test_automatic_choice_on_small_and_ragged_batches(prec, bs_last):
    """With bias and GELU, on both sides of the batches where the choice changes, on tensors that
    start off a 16-byte boundary, and the same bits from call to call."""
    from ksmm_amd import Kernel

    for pattern in [(1, 768, 192, 2), (2, 96, 384, 4), (4, 16, 16, 4), (1, 198, 192, 3)]:
        for batch in (1, 8, 61, 512, 1003):
            xin, fac, scale, z = _operands(pattern, batch, prec, bs_last)
            bias = torch.linspace(-1, 1, z.shape[0 if bs_last else 1]).to(torch.float32 if prec == "fp32" else torch.float16)
            zb = torch.from_numpy(z) + (bias.double()[:, None] if bs_last else bias.double())
            want = torch.nn.functional.gelu(zb).numpy()
            y = Kernel.forward(xin, fac, bs_last, *pattern, scale=scale, bias=bias.cuda(), act="gelu")
            assert _error(y, want) <= TOL[prec], (prec, bs_last, pattern, batch)
            assert torch.equal(y, Kernel.forward(xin, fac, bs_last, *pattern, scale=scale, bias=bias.cuda(), act="gelu"))
            shifted = torch.empty(xin.numel() + 1, dtype=xin.dtype, device="cuda")[1:].view(xin.shape)
            shifted.copy_(xin)
            y = Kernel.forward(shifted, fac, bs_last, *pattern, scale=scale)
            assert _error(y, z) <= TOL[prec], (prec, bs_last, pattern, batch, "shifted")


def test_small_batches_fill_the_chip():
    """Host only: (1,1536,384,2) on one image of 196 rows was 8 workgroups of a 256 x 128 tile."""
    from ksmm_amd import query_tile

    for dt in (torch.float32, torch.float16, torch.float8_e4m3fn):
        for bs_last in (True, False):
            t = query_tile(196, (1, 1536, 384, 2), dt, None, bs_last)
            assert t["grid"] * t["threads"] >= 256 * 64, (dt, bs_last, t)
    # a batch no vector divides: reported as the generic family's, and forced back by that number
    t = query_tile(197, (1, 1536, 384, 2), torch.float16, None, True)
    assert t["algo"] == 1 and t["variant"] >= 16
    assert query_tile(197, (1, 1536, 384, 2), torch.float16, None, True, algo=1, variant=t["variant"]) == t
