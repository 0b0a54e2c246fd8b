"""What the native call of KSLinear must leave as the Python path has it: a bias that is no plain
parameter, flags that are truthy without being ``True``, and the error of a full device."""
import pytest
import torch

PATTERNS = [(2, 32, 16, 2), (1, 64, 128, 1)]


def _layer(bs_last, **kw):
    from ksmm_amd import KSLinear

    torch.manual_seed(0)
    return KSLinear(PATTERNS, algo="kernel", dtype=torch.float32, bs_last=bs_last, device="cuda", **kw)


def _input(bs_last):
    gen = torch.Generator().manual_seed(1)
    return torch.randn((64, 96) if bs_last else (96, 64), generator=gen).cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("bs_last", [True, False])
def test_bias_that_is_pruned(bs_last):
    from torch.nn.utils import prune

    layer, x = _layer(bs_last, bias=True), _input(bs_last)
    with torch.no_grad():
        want = layer(x) - layer.bias
        mask = torch.zeros_like(layer.bias)
        mask[::2] = 1
        prune.custom_from_mask(layer, "bias", mask)
        # the sum and its rounding are the same up to the last bits of |y| + |bias|
        torch.testing.assert_close(layer(x), want + layer.bias_orig * mask, rtol=1e-6, atol=2e-6)


@pytest.mark.gpu
@pytest.mark.parametrize("bs_last", [True, False])
@pytest.mark.parametrize("for_good", [False, True])
def test_factor_that_is_pruned(bs_last, for_good):
    """Factors of one shape: unpruned or out of order they would fit as well."""
    from ksmm_amd import KSLinear
    from ksmm_amd.layer import from_kernel_format_to_abcd
    from torch.nn.utils import prune

    patterns = [(1, 16, 16, 4), (4, 16, 16, 1)]
    layer = KSLinear(patterns, algo="kernel", dtype=torch.float32, bs_last=bs_last, device="cuda")
    prune.l1_unstructured(layer.factors, "0", 0.5)
    if for_good:
        prune.remove(layer.factors, "0")
    with torch.no_grad():
        ref = KSLinear(patterns, weights=[from_kernel_format_to_abcd(f, p).cpu() for f, p in zip(layer.factors, patterns)],
                       algo="einsum", dtype=torch.float64, bs_last=bs_last, device="cuda")
        ref.bias.copy_(layer.bias)
        x = _input(bs_last)
        # two sums of 16 products in fp32
        torch.testing.assert_close(layer(x).double(), ref(x.double()), rtol=1e-5, atol=1e-5)


@pytest.mark.gpu
@pytest.mark.parametrize("bs_last", [True, False])
def test_flags_need_not_be_bool(bs_last):
    with torch.no_grad():
        x = _input(bs_last)
        assert torch.equal(_layer(int(bs_last), bias=True, fuse=1)(x), _layer(bs_last, bias=True, fuse=True)(x))


@pytest.mark.gpu
def test_full_device_raises_out_of_memory():
    layer, x = _layer(True, bias=False), torch.zeros(64, 1 << 16, device="cuda")
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    before = torch.cuda.memory_reserved()
    total = torch.cuda.get_device_properties(0).total_memory
    torch.cuda.set_per_process_memory_fraction((before + 4096) / total)
    try:
        with torch.no_grad(), pytest.raises(torch.cuda.OutOfMemoryError):
            layer(x)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    with torch.no_grad():
        assert not layer(x).any()


@pytest.mark.gpu
def test_native_module_loads():
    from ksmm_amd import _lib

    assert _lib.native().__name__ == "ksmm_amd._native"
