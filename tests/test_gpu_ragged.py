"""k-loop tiles on batch-size-last rows that no 16-byte vector divides: every instance, at batches around a vector and a
tile, with blocks that fill its tiles and blocks that do not (b and c tails), against float64.

Tolerances: fp32 1e-5, fp16 2e-3, e4m3 5e-3 on the dequantised operands (one rounding of the result; the sums
are fp32)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn
TOL = {torch.float32: 1e-5, torch.float16: 2e-3, FP8: 5e-3}


@pytest.mark.parametrize("dt", [torch.float32, torch.float16, FP8])
@pytest.mark.parametrize("pattern", [(2, 192, 64, 1), (1, 256, 100, 3), (2, 96, 33, 2), (1, 75, 40, 2)])
def test_ragged_rows(dt, pattern):
    from ksmm_amd import Kernel, _lib, generate_factor
    from ksmm_amd._lib import KsmmError

    a, b, c, d = pattern
    vec = 16 // torch.empty(0, dtype=dt).element_size()
    w4 = torch.empty(a, b, c, d).uniform_(-1, 1) / c ** 0.5
    w = generate_factor(a, b, c, d, "kernel", w4, torch.float32, "cuda").to(dt)
    wk = w.float().double().cpu().view(a, d, c, b)
    taken = 0
    for n in (vec, vec + 1, 2 * vec - 1, 127, 129, 255, 257, 261, 515):
        x = torch.randn(a * c * d, n, device="cuda").to(dt)
        want = torch.einsum("adcb,acdn->abdn", wk, x.float().double().cpu().view(a, c, d, n)).reshape(a * b * d, n)
        for i in range(128):
            try:
                y = Kernel.forward(x, w, True, a, b, c, d, algo=_lib.ALGO_TILE, variant=i | 1 << 8)
            except KsmmError:
                continue
            taken += 1
            err = ((y.double().cpu() - want).norm() / want.norm()).item()
            assert err <= TOL[dt], (n, i, err)
            if n % vec:  # as an ordinary instance it refuses such rows, as ever
                with pytest.raises(KsmmError):
                    Kernel.forward(x, w, True, a, b, c, d, algo=_lib.ALGO_TILE, variant=i)
    assert taken >= 9


def test_rows_of_neighbours_stay_as_they_are():
    """The last vector of a row is stored with its end: nothing behind the tensor, and no row's end, is touched."""
    from ksmm_amd import Kernel, generate_factor

    a, b, c, d, n = 4, 192, 192, 1, 6501
    w = generate_factor(a, b, c, d, "kernel", None, torch.float16, "cuda")
    x = torch.randn(a * c * d, n, device="cuda", dtype=torch.float16)
    flat = torch.full((a * b * d * n + 64,), 7.0, device="cuda", dtype=torch.float16)
    y = flat[:a * b * d * n].view(a * b * d, n)
    Kernel.forward(x, w, True, a, b, c, d, out=y)
    assert bool((flat[a * b * d * n:] == 7.0).all())
    want = torch.einsum("acb,acn->abn", w.double().view(a, c, b), x.double().view(a, c, n)).reshape(a * b, n)
    assert ((y.double() - want).norm() / want.norm()).item() <= 2e-3
    assert (y[:, -9:].double() - want[:, -9:]).abs().max().item() <= 2e-2


def test_ragged_rows_run_on_the_tiles():
    from ksmm_amd.kernel import query_tile

    for dt in (torch.float32, torch.float16, FP8):
        t = query_tile(6501, (1, 256, 256, 3), torch.float16 if dt == FP8 else dt, dt, True)
        v = t["variant"] - 16  # reported as the generic family's: no kernel of its own at full batches
        assert t["algo"] == 1 and v >> 8 == 1, t
