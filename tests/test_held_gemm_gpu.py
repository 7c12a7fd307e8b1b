"""The small-batch kernel that keeps the activations in registers (up to 16 rows of q4f16_1 and AutoGPTQ), against float64."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# one wavefront's run of 1 .. 5 pieces of 256 k; K that ends inside a piece, inside a run and before the last run; N of part
# of a tile, and of more rounds over the CUs than tiles in flight, odd and even
SHAPES = [(16, 64), (33, 576), (12300, 320), (8200, 2112), (130, 4096), (47, 4352), (259, 6208), (100, 8192)]
CASES = [(M, N, K) for M in (3, 8, 9, 16) for N, K in SHAPES] + [(2, 70, 8256), (8, 260, 10240)]
# two rounds of long runs, where the next tile's codes are requested into the registers that are being read
CASES += [(M, 16 * 256 + 40, K) for M in (3, 8, 9, 16) for K in (4352, 6208, 8192)]


def _codes(words):  # [N, K/8] -> [N, K]
    return ((words[:, :, None] >> torch.arange(0, 32, 4, device="cuda", dtype=torch.int32)) & 15).flatten(1).double()


@pytest.mark.parametrize("fmt", ["q4f16_1", "gptq"])
@pytest.mark.parametrize("M,N,K", CASES)
def test_against_float64(fmt, M, N, K):
    from relax_amd import _lib, ops

    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    half = lambda *s, lo=0.0, hi=1.0: (torch.rand(s, device="cuda", generator=g) * (hi - lo) + lo).half()
    words = lambda *s: torch.randint(-(2**31), 2**31 - 1, s, device="cuda", dtype=torch.int32, generator=g)
    if fmt == "gptq":
        N, K = N // 8 * 8, (K + 127) // 128 * 128
        gs = 256 if K % 512 == 0 else 128
        qw, qz, s, g_idx = words(K // 8, N), words(K // gs, N // 8), half(K // gs, N, lo=0.005, hi=0.02), torch.arange(K, dtype=torch.int32) // gs
        prep = ops.gptq_prepare(qw, qz, s, g_idx.cuda())
        zero = _codes(qz) + 1
        q = _codes(qw.t().contiguous())
        w = (q - zero.repeat_interleave(gs, 0).t()) * s.double().repeat_interleave(gs, 0).t()
        run = lambda x, r: ops.gptq_linear(prep, x, residual=r)
    else:
        W, S = words(N, K // 8), half(N, K // 32, lo=0.005, hi=0.02)
        w = (_codes(W) - 7) * S.double().repeat_interleave(32, 1)
        run = lambda x, r: ops.q4g32_linear(W, S, x, residual=r, kernel="small_batch")
    x = torch.randn(M, K, device="cuda", generator=g).half()
    x[0] *= 2.0**-13  # a row of small numbers loses nothing
    res = torch.randn(M, N, device="cuda", generator=g).half()
    tall = x.clone()
    tall[M - 1, K // 2] = 5000.0
    odd = x.clone()
    odd[0, K - 1], odd[M - 1, 3] = float("inf"), float("nan")
    _lib.lib().wq_debug_set_skinny_config(0, 0, 2)
    try:
        plain, with_res, y_tall, y_odd = run(x, None), run(x, res), run(tall, None), run(odd, None)
        torch.cuda.synchronize()
    finally:
        _lib.lib().wq_debug_set_skinny_config(0, 0, 0)

    def close(y, a, r, unit):
        # rounding of y (2^-11 of it, 2^-25 where it is no normal number), and per product `unit`: the sums' 24 bits and the
        # alignment of the products in the matrix core, 2^-17, or a weight rounded to fp16, 2^-11
        exact, mass = a.double() @ w.t(), a.double().abs() @ w.abs().t()
        room = exact.abs() * 2.0**-11 + 2.0**-25 + mass * unit
        if r is not None:  # the product is rounded, then the sum
            exact = exact + r.double()
            room = room + exact.abs() * 2.0**-11 + room * 2.0**-11
        bad = (y.double() - exact).abs() - room
        assert bad.max().item() <= 0, f"{bad.max().item():.3e}"

    close(plain, x, None, 2.0**-17)
    close(with_res, x, res, 2.0**-17)
    close(y_tall, tall, None, 2.0**-11)
    assert torch.isnan(y_odd[M - 1]).all()
    if M > 2:
        close(y_odd[1 : M - 1], odd[1 : M - 1], None, 2.0**-11)
    want = w[:, K - 1].sign() * float("inf")  # the sign of the weight, no number where it is zero
    np.testing.assert_array_equal(y_odd[0].float().cpu().numpy(), want.float().cpu().numpy())


# (format, M, column tiles per CU, tiles beside that, K, whether the kernel takes it): each bound of the rule from both sides
EDGES = [
    # K above 4096 and four tiles per CU
    ("q4f16_1", 16, 4, 0, 4160, True), ("q4f16_1", 16, 4, -1, 4160, False), ("q4f16_1", 16, 4, 0, 4096, False),
    ("gptq", 16, 4, 0, 4224, True), ("gptq", 16, 4, -1, 4224, False),
    # up to 8 rows: two tiles per CU, K of 4352 or (AutoGPTQ) 3072
    ("q4f16_1", 8, 2, 1, 4352, True), ("q4f16_1", 8, 2, 0, 4352, False), ("q4f16_1", 8, 2, 1, 4288, False), ("q4f16_1", 9, 2, 1, 4352, False),
    ("gptq", 8, 2, 1, 3072, True), ("gptq", 8, 2, 0, 3072, False), ("gptq", 8, 2, 1, 2944, False), ("gptq", 9, 2, 1, 3072, False),
    # ... five tiles per CU, K of 3840
    ("q4f16_1", 3, 5, 0, 3840, True), ("q4f16_1", 3, 5, -1, 3840, False), ("q4f16_1", 3, 5, 0, 3776, False),
    # more than 8 rows: five tiles per CU, K above 3072
    ("q4f16_1", 9, 5, 0, 3136, True), ("q4f16_1", 9, 5, -1, 3136, False), ("q4f16_1", 9, 5, 0, 3072, False),
    ("gptq", 16, 5, 0, 3200, True), ("gptq", 16, 5, -1, 3200, False), ("gptq", 16, 5, 0, 3072, False),
    # ... AutoGPTQ, two tiles per CU, K above 3840 that fills 15/16 of its pieces
    ("gptq", 9, 2, 1, 3968, True), ("gptq", 9, 2, 0, 3968, False), ("gptq", 9, 2, 1, 3840, False), ("gptq", 9, 2, 1, 5760, False),
    ("gptq", 9, 2, 1, 5888, True),
]


@pytest.mark.parametrize("fmt,M,per_cu,more,K,held", EDGES)
def test_the_choice_by_shape_at_its_edges(fmt, M, per_cu, more, K, held):
    """Which kernel ran, and that it is right: without rounded weights (2^-17 of a product, the alignment in the matrix core) where
    this one did, and with them (2^-11) where another."""
    from relax_amd import _lib, ops

    g = torch.Generator(device="cuda").manual_seed(3)
    N = 16 * (per_cu * torch.cuda.get_device_properties(0).multi_processor_count + more)
    x = torch.randn(M, K, device="cuda", generator=g).half()
    W = torch.randint(-(2**31), 2**31 - 1, (K // 8, N), device="cuda", dtype=torch.int32, generator=g)
    if fmt == "gptq":
        s = (torch.rand(K // 128, N, device="cuda", generator=g) * 0.015 + 0.005).half()
        z = torch.randint(-(2**31), 2**31 - 1, (K // 128, N // 8), device="cuda", dtype=torch.int32, generator=g)
        w = (_codes(W.t().contiguous()) - (_codes(z) + 1).repeat_interleave(128, 0).t()) * s.double().repeat_interleave(128, 0).t()
        y = ops.gptq_linear(ops.gptq_prepare(W, z, s, torch.arange(K, dtype=torch.int32, device="cuda") // 128), x)
    else:
        Wt, s = W.t().contiguous(), (torch.rand(N, K // 32, device="cuda", generator=g) * 0.015 + 0.005).half()
        w = (_codes(Wt) - 7) * s.double().repeat_interleave(32, 1)
        y = ops.q4g32_linear(Wt, s, x)
    torch.cuda.synchronize()
    assert (_lib.lib().wq_debug_small_batch_form() == 1) == held
    exact, mass = x.double() @ w.t(), x.double().abs() @ w.abs().t()
    assert ((y.double() - exact).abs() <= exact.abs() * 2.0**-11 + mass * (2.0**-17 if held else 2.0**-11)).all()


@pytest.mark.parametrize("path", ["q4f16_1", "gptq", "list"])
@pytest.mark.parametrize("M", [3, 16])
def test_weights_that_are_exact(path, M):
    """Scales that are powers of two: a weight is an fp16 number, so nothing but the result is rounded in any way of computing
    it.  The sums may add a fifth of that rounding (squares add: 2 %); they are a tenth or less."""
    from relax_amd import _lib, ops

    N, K = 4096, 4096
    g = torch.Generator(device="cuda").manual_seed(M)
    words = lambda *s: torch.randint(-(2**31), 2**31 - 1, s, device="cuda", dtype=torch.int32, generator=g)
    x = torch.randn(M, K, device="cuda", generator=g).half()
    _lib.lib().wq_debug_set_skinny_config(0, 0, 2)
    try:
        if path == "gptq":
            qw, qz = words(K // 8, N), words(K // 128, N // 8)
            s = torch.exp2(torch.randint(-9, -5, (K // 128, N), device="cuda", generator=g).float()).half()
            y = ops.gptq_linear(ops.gptq_prepare(qw, qz, s, torch.arange(K, device="cuda", dtype=torch.int32) // 128), x)
            w = (_codes(qw.t().contiguous()) - (_codes(qz) + 1).repeat_interleave(128, 0).t()) * s.double().repeat_interleave(128, 0).t()
        else:
            W, S = words(N, K // 8), torch.exp2(torch.randint(-9, -5, (N, K // 32), device="cuda", generator=g).float()).half()
            w = (_codes(W) - 7) * S.double().repeat_interleave(32, 1)
            if path == "list":
                y = torch.zeros(M, N, device="cuda", dtype=torch.float16)
                lin = ops.Q4G32GemvList([(W, S, x, y)], M=M)
                lin.run()
                lin.status()
            else:
                y = ops.q4g32_linear(W, S, x, kernel="small_batch")
        torch.cuda.synchronize()
    finally:
        _lib.lib().wq_debug_set_skinny_config(0, 0, 0)
    exact = x.double() @ w.t()
    miss, rounding = (y.double() - exact).norm().item(), (exact.half().double() - exact).norm().item()
    assert miss <= 1.02 * rounding, miss / rounding
