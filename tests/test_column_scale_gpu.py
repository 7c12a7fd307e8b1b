"""int8 and int4 with a scale per column: the sums take the scale in fp32, the weights are not rounded.  Against float64, in the
small-batch kernels and the tiled GEMM."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _inputs(M, N, K, bits, seed):
    from relax_amd import ops

    g = torch.Generator(device="cuda").manual_seed(seed)
    q = torch.randint(-128, 128, (K, N * bits // 8), device="cuda", dtype=torch.int8, generator=g)
    codes = q.double() if bits == 8 else torch.stack([(q << 4) >> 4, q >> 4], -1).flatten(1).double()
    return torch.randn(M, K, device="cuda", generator=g).half(), ops.ft_preprocess_weight(q, 80, bits == 4), codes, g


# one, two, four and eight column blocks, slabs of 16 .. 64 rows, activations in registers (K = 6144), K that ends inside a step; the
# tiled GEMM with halves of K and without, and 256 x 256 tiles
@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("M,N,K", [(4, 16448, 6144), (8, 1024, 4160), (16, 9280, 2048), (20, 8256, 2048), (24, 1024, 2048), (40, 4160, 1088), (64, 22016, 512),
                                   (100, 1024, 4160), (300, 4160, 2048), (1100, 4160, 1088)])
def test_only_the_result_is_rounded(bits, M, N, K):
    from relax_amd import ops

    x, B, codes, g = _inputs(M, N, K, bits, M + N)
    s = (torch.rand(N, device="cuda", generator=g) * 0.009 + 0.001).half()
    y = ops.fpA_intB_gemm(x, B, s, weight_nbit=bits)
    exact = (x.double() @ codes) * s.double()
    # an fp16 number is off by up to half a step, in root mean square by a step / sqrt(12); a tenth more for the sums in fp32 (a
    # rounding of the weights adds four tenths)
    step = torch.exp2(torch.floor(torch.log2(exact.abs().clamp_min(2.0**-14))) - 10)
    miss, rounding = (y.double() - exact).norm().item(), (step.norm() / 12**0.5).item()
    assert miss <= 1.1 * rounding, miss / rounding


@pytest.mark.parametrize("bits", [8, 4])
@pytest.mark.parametrize("M", [8, 40, 300])
def test_weights_beyond_fp16(bits, M):
    """A scale with which the largest weights are no fp16 numbers: here the product is what it is, the dequantized weight infinite."""
    from relax_amd import ops

    N, K = 256, 512
    x, B, codes, _ = _inputs(M, N, K, bits, M)
    x *= 2.0**-14
    s = torch.full((N,), 1000.0 if bits == 8 else 10000.0, device="cuda").half()
    y = ops.fpA_intB_gemm(x, B, s, weight_nbit=bits)
    exact = (x.double() @ codes) * s.double()
    assert exact.abs().max() < 65504
    mass = (x.double().abs() @ codes.abs()) * s.double()
    assert ((y.double() - exact).abs() <= exact.abs() * 2.0**-11 + mass * 2.0**-20).all()
    w = ops.intb_dequantize(B, s, bits)
    assert torch.isinf(w).any()
