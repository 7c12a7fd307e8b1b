"""The tiled GEMM where the loads that its K loop issues past the last step would land in the LDS that the results are
staged in: rings of three slots with K / 64 % 3 == 2 (320, 704, 896), rings of four with 1, 3 and 2, whole tiles and row
slices, one workgroup per CU and two.  x = identity returns the dequantized weights, so a result that such a load
overwrote is not a weight any more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KS = [320, 704, 896]


@pytest.fixture(scope="module")
def env():
    import torch

    assert torch.cuda.is_available(), "these tests need a GPU"
    from relax_amd import _lib, ops
    from tests import gpu_util

    yield ops, gpu_util, _lib.lib()
    _lib.lib().wq_debug_set_gemm_tail_split(1)
    _lib.lib().wq_debug_set_gemm_config(0)


def _each(lib, cfgs):
    """Every tile configuration, with the last round cut into row slices and not."""
    for cfg in cfgs:
        for split in (1, 0):
            lib.wq_debug_set_gemm_config(cfg)
            lib.wq_debug_set_gemm_tail_split(split)
            yield cfg, split
    lib.wq_debug_set_gemm_tail_split(1)
    lib.wq_debug_set_gemm_config(0)


@pytest.mark.parametrize("K", KS)
@pytest.mark.parametrize("nbit,group", [(8, -1), (8, 64), (4, -1), (4, 64)])
def test_fpA_intB(env, oracle, nbit, group, K):
    ops, u, lib = env
    for N in (192, 8256):
        _, A, s = oracle.make_intb_inputs(1, N, K, nbit, seed=K + nbit, group_size=group)
        want = oracle.intb_dequant(A, s, nbit, group)
        B, ds, x = ops.ft_preprocess_weight(u.dev(A), 80, nbit == 4), u.dev(s), u.dev(np.eye(K, dtype=np.float16))
        for cfg, split in _each(lib, (11, 17, 18)):
            got = u.host(ops.fpA_intB_gemm(x, B, ds, weight_nbit=nbit, group_size=group))
            np.testing.assert_array_equal(got, want, err_msg=f"N={N} cfg={cfg} split={split}")


@pytest.mark.parametrize("K", [128, 192] + [k + 32 for k in KS])
def test_q4f16_1_with_weights_in_lds(env, oracle, K):
    """K < 256, and K % 64 == 32, whose last half step lies behind the loop."""
    ops, u, lib = env
    for N in (300, 8200):
        _, W, S = oracle.make_q4g32_inputs(1, N, K, seed=K)
        want = oracle.q4g32_dequant(W, S).T
        dW, dS, x = u.dev(W), u.dev(S), u.dev(np.eye(K, dtype=np.float16))
        for cfg, split in _each(lib, (11, 17, 18)):
            got = u.host(ops.q4g32_linear(dW, dS, x, kernel="gemm"))
            np.testing.assert_array_equal(got, want, err_msg=f"N={N} cfg={cfg} split={split}")


@pytest.mark.parametrize("K", KS)
def test_autogptq_with_a_group_of_64(env, oracle, K):
    ops, u, lib = env
    for N in (264, 8200):
        _, qw, qz, s, g_idx = oracle.make_gptq_inputs(1, N, K, 64, seed=K, act_order=False)
        w = ops.gptq_prepare(u.dev(qw), u.dev(qz), u.dev(s), u.dev(g_idx))
        got = u.host(ops.gptq_linear(w, u.dev(np.eye(K, dtype=np.float16))))
        np.testing.assert_array_equal(got, oracle.gptq_dequant(qw, qz, s, g_idx), err_msg=f"N={N}")


@pytest.mark.parametrize("K", KS)
def test_weights_packed_along_n(env, oracle, K):
    ops, u, lib = env
    for N in (160, 8224):
        _, W, S = oracle.make_q4g32_inputs(1, K, N, seed=K)
        W_nk, ST = ops.q4n32_prepare(u.dev(W), u.dev(S))
        for cfg, split in _each(lib, (11, 17, 18)):
            got = u.host(ops.q4n32_linear(W_nk, ST, u.dev(np.eye(K, dtype=np.float16))))
            np.testing.assert_array_equal(got, oracle.q4g32_dequant(W, S), err_msg=f"N={N} cfg={cfg} split={split}")


def test_weights_packed_along_n_with_64_bit_addresses(env):
    """There the loads past the end read the last step again, from memory.  One activation per row is not zero."""
    import torch

    ops, _, _ = env
    M, N, K = 130, 32, (1 << 23) + 192
    g = torch.Generator(device="cuda").manual_seed(5)
    W_nk = torch.randint(-2**31, 2**31 - 1, (N, K // 8), dtype=torch.int32, device="cuda", generator=g)
    ST = (torch.rand((1, K), device="cuda", generator=g) * 0.015 + 0.005).half()
    x = torch.zeros((M, K), dtype=torch.float16, device="cuda")
    ks = torch.cat([torch.tensor([0, K - 129, K - 128, K - 65, K - 64, K - 1]),
                    torch.randint(0, K, (M - 6,), generator=torch.Generator().manual_seed(6))]).cuda()
    x[torch.arange(M, device="cuda"), ks] = 1.0
    y = ops.q4n32_linear(W_nk, ST, x)
    codes = (W_nk[:, ks // 8] >> (4 * (ks % 8)).int()[None, :]) & 15
    assert torch.equal(y, ((codes.half() - 7) * ST[:, ks]).t())
