"""e4m3 layers that quantise their input (ksmm_quant.hip) against the same steps as tensor operations: the
codes and the scale are the same, so the results have the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu

FP8 = torch.float8_e4m3fn

# one chain per kernel family: fused butterfly, dense blocks of either layout, ragged ones, small ones
LAYERS = [[(1, 16, 16, 16), (16, 16, 16, 1)], [(2, 128, 64, 1), (1, 192, 128, 2)], [(1, 37, 21, 3)], [(1, 48, 48, 4)],
          [(3, 8, 16, 8)], [(1, 96, 96, 64)], [(4, 256, 64, 1)]]


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
@pytest.mark.parametrize("bs_last", [False, True])
def test_quantised_inputs_give_the_same_bits(dt, bs_last):
    from ksmm_amd import KSLinear, quantize_fp8

    gen = torch.Generator(device="cuda").manual_seed(11)
    with torch.no_grad():
        for patterns in LAYERS:
            layer = KSLinear(patterns, algo="kernel", dtype=FP8, bs_last=bs_last, device="cuda", act="gelu")
            for n in (1, 7, 64, 197, 1031, 4096):
                for offset in (0, 1):
                    x = (3 * torch.randn(offset + layer.in_size * n, generator=gen, device="cuda")).to(dt)[offset:]
                    x = x.view((layer.in_size, n) if bs_last else (n, layer.in_size))
                    codes, scale = quantize_fp8(x)
                    assert torch.equal(layer(x), layer(codes, x_scale=float(scale))), (patterns, n, offset)


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
def test_one_launch_and_two_give_the_same_codes(dt):
    """Sizes around the 384 KB up to which one launch takes the input, whole runs of 16 values and not; the largest
    value is the last, which the last thread alone sees."""
    from ksmm_amd import KSLinear, quantize_fp8

    edge = (384 << 10) // (2 if dt == torch.float16 else 4)
    w = torch.eye(8).reshape(1, 8, 8, 1)
    with torch.no_grad():
        layer = KSLinear([(1, 8, 8, 1)], weights=[w], bias=False, algo="kernel", dtype=FP8, device="cuda")
        for rows in (1, 2, 3, 2049, edge // 8 - 1, edge // 8, edge // 8 + 1):
            x = torch.randn(rows, 8, device="cuda").to(dt)
            x[-1, -1] = -9.5
            codes, scale = quantize_fp8(x)
            assert float(scale) == pytest.approx(9.5 / 448, rel=1e-3)
            assert torch.equal(layer(x), layer(codes, x_scale=float(scale))), rows


@pytest.mark.parametrize("dt", [torch.float32, torch.float16])
def test_quantisation_of_special_values(dt):
    """Zeros, one value, infinities, NaN, denormals, halfway codes: a layer of the identity shows the codes."""
    from ksmm_amd import KSLinear, quantize_fp8

    inf, nan = float("inf"), float("nan")
    halfway = [(m + 0.5) / 8 * 2.0 ** e for e in range(-9, 9) for m in range(8, 15)] + [448.0]
    rows = [[0.0], [-0.0, 0.0], [1.0, -0.3], [inf, 1.0, -inf], [nan, 700.0, -470.0, 464.0, 5.0], [6e-8, -1e-7, 3e-6], halfway,
            [-v for v in halfway], [65504.0, 1e-3, -7.5]]
    if dt == torch.float32:
        rows += [[1e-44, 1e-45], [3e38, -1e30, 1.0], [1e-38, -1e-39]]
    w = torch.eye(128).reshape(1, 128, 128, 1)
    with torch.no_grad():
        layer = KSLinear([(1, 128, 128, 1)], weights=[w], bias=False, algo="kernel", dtype=FP8, device="cuda")
        for row in rows:
            x = torch.zeros(64, 128, device="cuda", dtype=dt)
            x.view(-1)[:len(row)] = torch.tensor(row, device="cuda", dtype=dt)
            codes, scale = quantize_fp8(x)
            assert torch.equal(torch.nan_to_num(layer(x)), torch.nan_to_num(layer(codes, x_scale=float(scale)))), row
            assert torch.equal(layer(x).isnan(), layer(codes, x_scale=float(scale)).isnan()), row


def test_quantising_layers_replay_in_a_graph():
    from ksmm_amd import KSLinear

    with torch.no_grad():
        layers = [KSLinear(p, algo="kernel", dtype=FP8, device="cuda") for p in ([(4, 64, 64, 1)], [(1, 96, 128, 2)])]
        x = torch.randn(197, 256, device="cuda", dtype=torch.float16)
        side = torch.cuda.Stream()
        with torch.cuda.stream(side):
            layers[1](layers[0](x))
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = layers[1](layers[0](x))
        for k in range(4):
            x.copy_(torch.randn(197, 256, device="cuda") * (k + 1))
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y, layers[1](layers[0](x))), k


@pytest.mark.parametrize("dt,exponents", [(torch.float16, range(-22, 15, 4)), (torch.float32, (-120, -53, -52, -51, -20, 0, 33, 67, 68, 69, 120))])
def test_scales_with_and_without_a_division(dt, exponents):
    """Scales from 2^-60 to 2^60 take the quotient by residuals, others divide: the same bits."""
    from ksmm_amd import KSLinear, quantize_fp8

    gen = torch.Generator(device="cuda").manual_seed(12)
    w = torch.eye(128).reshape(1, 128, 128, 1)
    with torch.no_grad():
        layer = KSLinear([(1, 128, 128, 1)], weights=[w], bias=False, algo="kernel", dtype=FP8, device="cuda")
        for e in exponents:
            x = torch.rand(512, 128, generator=gen, device="cuda") * 2 - 1
            x[::2] *= torch.exp2(-20 * torch.rand(256, 128, generator=gen, device="cuda"))
            x = (x * 2.0 ** e).to(dt)
            codes, scale = quantize_fp8(x)
            layer.w_scales[0] = 2.0 ** -e  # fp16 results in range
            got, want = layer(x), layer(codes, x_scale=float(scale))
            assert torch.equal(got.nan_to_num(), want.nan_to_num()), (dt, e)
