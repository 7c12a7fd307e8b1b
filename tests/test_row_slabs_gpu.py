"""Slabs of 24 and 48 rows in every format of the small-batch kernel, with one, two and four column blocks and eight wavefronts, and
with three and twelve: workgroups whose last columns lie past N, fewer steps of K than wavefronts along it, K that ends
inside a step, and (the last) the choice by shape."""
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
