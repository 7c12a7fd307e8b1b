"""Slabs of 24 and 48 rows in every format of the small-batch kernel, with one, two and four column blocks and eight wavefronts, and
with three and twelve: workgroups whose last columns lie past N, fewer steps of K than wavefronts along it, K that ends
inside a step; and the choice by shape."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fmt", ["q4f16_1", "gptq64", "int8", "int4", "int4x64"])
@pytest.mark.parametrize("M,N,K,nw,stages,waves", [
    (17, 64, 64, 3, 2, 12), (19, 128, 576, 3, 3, 12), (24, 320, 4160, 3, 0, 12),
    (17, 64, 2048, 1, 2, 1), (24, 320, 2112, 1, 3, 1),
    (33, 64, 64, 1, 2, 1), (40, 320, 1088, 2, 3, 1), (48, 128, 4224, 2, 0, 1), (39, 192, 4160, 4, 2, 1), (47, 128, 192, 1, 3, 1),
    (21, 8256, 2112, 0, 0, 0), (40, 4160, 1088, 0, 0, 0)])
def test_against_the_oracle(fmt, M, N, K, nw, stages, waves):
    from oracle import wq_oracle as oracle
    from relax_amd import _lib, ops
    from tests import gpu_util as u
    from tests import test_gptq_gpu, test_intb_gpu

    _lib.lib().wq_debug_set_skinny_config(nw, stages, waves)
    try:
        if fmt.startswith("int"):
            test_intb_gpu._run(ops, u, oracle, M, N, K, int(fmt[3]), seed=M + N, group_size=64 if fmt.endswith("x64") else -1)
        elif fmt == "gptq64":
            x, qw, qz, s, g_idx = oracle.make_gptq_inputs(M, N, K, 64, seed=M + N)
            y = ops.gptq_linear(ops.gptq_prepare(*map(u.dev, (qw, qz, s, g_idx))), u.dev(x))
            u.assert_close(u.host(y), test_gptq_gpu._ref_linear(oracle, qw, qz, s, g_idx, x), f"{fmt} {M}x{N}x{K}")
        else:
            for k in (K, K - 32):  # an odd number of groups per column too
                x, W, S = oracle.make_q4g32_inputs(M, N, k, seed=M + N)
                y = ops.q4g32_linear(u.dev(W), u.dev(S), u.dev(x))
                u.assert_close(u.host(y), oracle.q4g32_linear(W, S, x, nthreads=8), f"{fmt} {M}x{N}x{k}")
    finally:
        _lib.lib().wq_debug_set_skinny_config(0, 0, 0)


# (formats, M, column tiles per CU, tiles beside that (Format B: fours), K, slab rows / 8, wavefronts side by side, wavefronts or 0: either count)
ONE, TWO = ("q4f16_1", "int4"), ("int8",)  # pieces of a weight tile
EDGES = [
    # 17 .. 24 rows, two to three tiles per CU: twelve wavefronts from K = 2048 on
    (ONE + TWO, 17, 2, 4, 2048, 3, 3, 12), (ONE + TWO, 24, 3, 0, 2048, 3, 3, 12), (ONE + TWO, 24, 2, 0, 2048, 4, 2, 0), (ONE + TWO, 24, 3, 4, 2048, 4, 4, 0),
    (ONE, 24, 3, 0, 1984, 4, 4, 0), (TWO, 24, 3, 0, 1984, 3, 3, 6), (ONE + TWO, 25, 3, 0, 2048, 4, 4, 0), (ONE + TWO, 16, 3, 0, 2048, 2, 0, 0),
    # ... four to six
    (ONE + TWO, 20, 4, 4, 128, 3, 3, 6), (ONE + TWO, 20, 6, 0, 128, 3, 3, 6), (ONE + TWO, 20, 4, 0, 128, 4, 4, 0),
    # ... one column block, int8
    (TWO, 17, 0, 64, 2048, 3, 1, 8), (TWO, 24, 0, 64, 2048, 3, 1, 8), (TWO, 25, 0, 64, 2048, 4, 1, 0), (TWO, 24, 0, 64, 1984, 4, 1, 0), (ONE, 24, 0, 64, 2048, 4, 1, 0),
    # 33 .. 48 rows, one, two and four column blocks
    (ONE + TWO, 32, 0, 64, 512, 4, 1, 0), (ONE + TWO, 33, 0, 64, 512, 6, 1, 0), (ONE + TWO, 48, 0, 64, 512, 6, 1, 0), (ONE + TWO, 49, 0, 64, 512, 8, 1, 0),
    (ONE, 40, 1, 4, 4096, 6, 2, 0), (ONE, 41, 1, 4, 4096, 8, 2, 0), (ONE, 48, 1, 4, 4160, 6, 2, 0), (TWO, 33, 1, 4, 4160, 8, 2, 0),
    (ONE, 48, 2, 4, 512, 6, 4, 0), (TWO, 40, 2, 4, 512, 6, 4, 0), (TWO, 41, 2, 4, 512, 8, 4, 0), (ONE, 49, 2, 4, 512, 8, 4, 0),
]


@pytest.mark.parametrize("formats,M,per_cu,more,K,TH,NW,waves", EDGES)
def test_the_choice_by_shape_at_its_edges(formats, M, per_cu, more, K, TH, NW, waves):
    """Which form ran (TH 0, NW 0: not looked at), and that it is right: sums against float64 with the output's and a weight's rounding."""
    import torch

    from relax_amd import _lib, ops

    g = torch.Generator(device="cuda").manual_seed(M + K)
    N = 16 * (per_cu * torch.cuda.get_device_properties(0).multi_processor_count + more)
    x = torch.randn(M, K, device="cuda", generator=g).half()
    for fmt in formats:
        if fmt == "q4f16_1":
            W = torch.randint(-(2**31), 2**31 - 1, (N, K // 8), device="cuda", dtype=torch.int32, generator=g)
            S = (torch.rand(N, K // 32, device="cuda", generator=g) * 0.015 + 0.005).half()
            w = (((W[:, :, None] >> torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)) & 15).flatten(1).double() - 7) * S.double().repeat_interleave(32, 1)
            y = ops.q4g32_linear(W, S, x)
        else:
            bits = int(fmt[3])
            q = torch.randint(-128, 128, (K, N * bits // 8), device="cuda", dtype=torch.int8, generator=g)
            S = (torch.rand(N, device="cuda", generator=g) * 0.015 + 0.005).half()
            codes = q.double() if bits == 8 else torch.stack([(q << 4) >> 4, q >> 4], -1).flatten(1).double()
            w = codes.t() * S.double()[:, None]
            y = ops.fpA_intB_gemm(x, ops.ft_preprocess_weight(q, 80, bits == 4), S, weight_nbit=bits)
        torch.cuda.synchronize()
        form = _lib.lib().wq_debug_small_batch_form()
        got = (form >> 16, form >> 8 & 255, form & 255)
        assert got[0] == TH and NW in (0, got[1]) and waves in (0, got[2]), (fmt, got)
        exact, mass = x.double() @ w.t(), x.double().abs() @ w.abs().t()
        assert ((y.double() - exact).abs() <= exact.abs() * 2.0**-11 + mass * 2.0**-11).all(), fmt
