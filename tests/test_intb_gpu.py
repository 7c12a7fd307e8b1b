"""GPU parity of the format-B (fp16 x int8/int4) path against the CPU oracle, through the C ABI."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GOLD = os.path.join(os.path.dirname(__file__), "golden", "ft_layout_vectors.npz")


@pytest.fixture(scope="module")
def ops():
    import torch

    assert torch.cuda.is_available(), "these tests need a GPU"
    from relax_amd import ops as _ops

    return _ops


@pytest.fixture(scope="module")
def u():
    from tests import gpu_util

    return gpu_util


@pytest.mark.parametrize("case", ["int8_64x64", "int8_128x192", "int8_256x64", "int4_64x64", "int4_128x192", "int4_256x128"])
def test_device_preprocess_matches_golden(ops, u, case):
    g = np.load(GOLD)
    a, want = g[case + "_in"], g[case + "_out"]
    got = u.host(ops.ft_preprocess_weight(u.dev(a), 80, case.startswith("int4")))
    assert np.array_equal(got, want)


@pytest.mark.parametrize("is_int4", [False, True])
def test_device_preprocess_large_and_experts(ops, u, oracle, is_int4):
    rng = np.random.default_rng(17)
    a = rng.integers(-128, 128, size=(2, 512, 320)).astype(np.int8)
    got = u.host(ops.ft_preprocess_weight(u.dev(a), 80, is_int4))
    assert np.array_equal(got, oracle.ft_preprocess(a, is_int4, 80))
    a = rng.integers(-128, 128, size=(8192, 1024 if not is_int4 else 512)).astype(np.int8)
    got = u.host(ops.ft_preprocess_weight(u.dev(a), 80, is_int4))
    assert np.array_equal(got, oracle.ft_preprocess(a, is_int4, 80))


@pytest.mark.parametrize("nbit", [8, 4])
def test_dequant_exhaustive_bit_exact(ops, u, oracle, nbit):
    """every code x every fp16 scale bit pattern, through preprocess + device dequantize."""
    all_s = np.arange(65536, dtype=np.uint32).astype(np.uint16).view(np.float16)
    ncode = 256 if nbit == 8 else 16
    lo = -128 if nbit == 8 else -8
    K = 256  # codes repeat down the rows; K must be a multiple of 64
    codes = (np.arange(K) % ncode + lo).astype(np.int64)
    for start in range(0, 65536, 16384):
        s = all_s[start:start + 16384]
        N = s.size
        q = np.repeat(codes[:, None], N, axis=1)
        if nbit == 8:
            A = q.astype(np.int8)
        else:
            A = ((q[:, 0::2] & 15) | ((q[:, 1::2] & 15) << 4)).astype(np.uint8).view(np.int8)
        want = oracle.intb_dequant(A, s, nbit)
        P = ops.ft_preprocess_weight(u.dev(A), 80, nbit == 4)
        got = u.host(ops.intb_dequantize(P, u.dev(s), nbit))
        nan = np.isnan(want)
        assert np.array_equal(got.view(np.uint16)[~nan], want.view(np.uint16)[~nan])
        assert np.all(np.isnan(got[nan]))


@pytest.mark.parametrize("nbit", [8, 4])
def test_dequant_finegrained(ops, u, oracle, nbit):
    _, A, s = oracle.make_intb_inputs(1, 128, 256, nbit, seed=4, group_size=64)
    P = ops.ft_preprocess_weight(u.dev(A), 80, nbit == 4)
    got = u.host(ops.intb_dequantize(P, u.dev(s), nbit, group_size=64))
    assert np.array_equal(got.view(np.uint16), oracle.intb_dequant(A, s, nbit, 64).view(np.uint16))


def _run(ops, u, oracle, M, N, K, nbit, seed, group_size=-1, **ep):
    x, A, s = oracle.make_intb_inputs(M, N, K, nbit, seed=seed, group_size=group_size)
    rng = np.random.default_rng(seed + 1)
    kw, okw = {}, {}
    if ep.get("bias") == "row":
        b = rng.standard_normal(N).astype(np.float16)
        kw["bias"], okw["bias"] = u.dev(b), b
    elif ep.get("bias") == "full":
        b = rng.standard_normal((M, N)).astype(np.float16)
        kw["bias"], okw["bias"], okw["bias_stride"] = u.dev(b), b, N
    if ep.get("residual"):
        r = rng.standard_normal((M, N)).astype(np.float16)
        kw["residual"], okw["residual"] = u.dev(r), r
        kw["binary_op"] = okw["binary_op"] = ep.get("binary_op", "plus")
        kw["unary_op"] = okw["unary_op"] = ep.get("unary_op", "identity")
    act = ep.get("activation", "identity")
    P = ops.ft_preprocess_weight(u.dev(A), 80, nbit == 4)
    got = u.host(ops.fpA_intB_gemm(u.dev(x), P, u.dev(s), weight_nbit=nbit, activation=act, group_size=group_size, **kw))
    ref = oracle.intb_linear(x, A, s, nbit, group_size=group_size, activation=act, nthreads=8, **okw)
    u.assert_close(got, ref, f"intb nbit={nbit} M={M} N={N} K={K} g={group_size} {ep}")


@pytest.mark.parametrize("nbit", [8, 4])
@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 16, 33, 128, 300])
def test_gemm_vs_oracle_shapes(ops, u, oracle, nbit, M):
    print(f"intb nbit={nbit} M={M}", flush=True)
    _run(ops, u, oracle, M, 256, 512, nbit, seed=M)
    _run(ops, u, oracle, M, 64, 64, nbit, seed=M + 50)
    _run(ops, u, oracle, M, 192, 4096, nbit, seed=M + 100)


@pytest.mark.parametrize("nbit", [8, 4])
@pytest.mark.parametrize("M", [1, 4, 64])
def test_gemm_finegrained(ops, u, oracle, nbit, M):
    _run(ops, u, oracle, M, 128, 512, nbit, seed=M + 7, group_size=64)


@pytest.mark.parametrize("nbit", [8, 4])
@pytest.mark.parametrize("M", [2, 48, 100, 130])
@pytest.mark.parametrize("ep", [
    dict(bias="row"), dict(bias="full"), dict(bias="row", activation="relu"), dict(bias="row", activation="silu"),
    dict(bias="row", activation="gelu"), dict(residual=True), dict(bias="row", residual=True, binary_op="plus"),
    dict(bias="row", residual=True, binary_op="multiply", unary_op="relu"),
    dict(bias="row", activation="silu", residual=True, binary_op="plus", unary_op="relu"),
], ids=lambda d: "-".join(f"{k}={v}" for k, v in d.items()))
def test_gemm_epilogues(ops, u, oracle, nbit, M, ep):
    _run(ops, u, oracle, M, 128, 256, nbit, seed=M + 3, **ep)


@pytest.mark.parametrize("nw,stages,waves", [(1, 2, 0), (2, 3, 0), (4, 4, 0), (8, 3, 0), (0, 0, 0), (0, 0, 1), (0, 0, 2)])
@pytest.mark.parametrize("nbit", [8, 4])
@pytest.mark.parametrize("group_size", [-1, 64])
def test_small_batch_work_splits(ops, u, oracle, nbit, group_size, nw, stages, waves):
    """3 <= M <= 64 runs the matrix-core streaming kernel; every work split of it, ragged M,
    K not a multiple of its 128-k step."""
    from relax_amd import _lib

    _lib.lib().wq_debug_set_skinny_config(nw, stages, waves)
    try:
        for M, N, K in [(3, 64, 64), (8, 320, 448), (9, 128, 4096), (16, 320, 448), (24, 64, 1024),
                        (32, 2048, 512), (40, 320, 448), (64, 192, 2112), (16, 4288, 8192), (5, 8192, 5184)]:
            print(f"intb small batch nbit={nbit} g={group_size} nw={nw} waves={waves} M={M} N={N} K={K}", flush=True)
            _run(ops, u, oracle, M, N, K, nbit, seed=M + nw, group_size=group_size)
    finally:
        _lib.lib().wq_debug_set_skinny_config(0, 0, 0)


@pytest.mark.parametrize("nbit", [8, 4])
@pytest.mark.parametrize("group_size", [-1, 64])
@pytest.mark.parametrize("M,N,K,nw,stages", [(17, 64, 64, 3, 2), (19, 320, 448, 3, 3), (24, 2048, 512, 3, 2), (21, 192, 2112, 3, 0),
                                             (18, 8256, 576, 0, 0), (23, 16448, 512, 0, 0)])
def test_slabs_of_24_rows(ops, u, oracle, nbit, group_size, M, N, K, nw, stages):
    """17 .. 24 rows with three wavefronts side by side, forced and (the last two) by shape."""
    from relax_amd import _lib

    _lib.lib().wq_debug_set_skinny_config(nw, stages, 0)
    try:
        _run(ops, u, oracle, M, N, K, nbit, seed=M, group_size=group_size)
    finally:
        _lib.lib().wq_debug_set_skinny_config(0, 0, 0)


@pytest.mark.parametrize("stages", [2, 3, 4])
@pytest.mark.parametrize("group_size", [-1, 64])
@pytest.mark.parametrize("M,N,K", [(17, 64, 512), (24, 192, 1024), (25, 64, 1536), (32, 320, 4608), (32, 192, 576), (29, 64, 64)])
def test_int8_two_column_blocks(ops, u, oracle, group_size, M, N, K, stages):
    """int8, 17 .. 32 rows, two wavefronts side by side: the weights of a later step are requested behind the products
    where K comes out even (K % 512 == 0: one step, as many as the ring holds, more), with the activations elsewhere."""
    from relax_amd import _lib

    _lib.lib().wq_debug_set_skinny_config(2, stages, 1)
    try:
        _run(ops, u, oracle, M, N, K, 8, seed=M + K, group_size=group_size)
    finally:
        _lib.lib().wq_debug_set_skinny_config(0, 0, 0)


@pytest.mark.parametrize("rows", [0, 1, 2])
@pytest.mark.parametrize("nbit", [8, 4])
@pytest.mark.parametrize("group_size", [-1, 64])
def test_one_and_two_rows_on_either_kernel(ops, u, oracle, nbit, group_size, rows):
    """M <= 2: the automatic choice (the streaming kernel for wide matrices, the small-batch kernel for narrow
    ones, where whole columns per wavefront leave the machine short of wavefronts) and the streaming kernel asked
    for by the test hook, with one and two column groups per wavefront."""
    from relax_amd import _lib

    _lib.lib().wq_debug_set_gemv_config(rows, 0)
    try:
        for M, N, K in [(1, 64, 64), (2, 64, 128), (1, 320, 448), (2, 320, 4096), (1, 4096, 1024), (2, 4096, 1024),
                        (1, 16384, 256), (2, 16384, 256), (1, 1024, 11008)]:
            print(f"intb rows={rows} nbit={nbit} g={group_size} M={M} N={N} K={K}", flush=True)
            _run(ops, u, oracle, M, N, K, nbit, seed=M + N + rows, group_size=group_size, bias="row")
    finally:
        _lib.lib().wq_debug_set_gemv_config(0, 0)


@pytest.mark.parametrize("nbit", [8, 4])
def test_65_to_128_rows_in_two_small_batch_passes(ops, u, oracle, nbit):
    """65 .. 96 rows of a small matrix, and up to 128 where a GEMM cannot halve K or (int8, a scale per 64, long K) gains
    nothing by it, run as two passes of the small-batch kernel (64 rows, then the rest), others as a tiled GEMM: both
    sides of the rule, with an epilogue that reads per-row operands."""
    for M, N, K, g in [(65, 4096, 256, -1), (96, 1024, 1024, 64), (128, 1024, 1024, 64), (100, 512, 192, 64),
                       (128, 1024, 8320, 64), (96, 5120, 8192, -1), (97, 5120, 8192, -1), (128, 4160, 512, 64)]:
        print(f"intb two passes nbit={nbit} M={M} N={N} K={K} g={g}", flush=True)
        _run(ops, u, oracle, M, N, K, nbit, seed=M + N, group_size=g, bias="full")
        _run(ops, u, oracle, M, N, K, nbit, seed=M + N + 1, group_size=g, bias="row", residual=True, binary_op="multiply")


@pytest.mark.parametrize("ways", [2, 4, 8])
@pytest.mark.parametrize("nbit", [8, 4])
@pytest.mark.parametrize("group_size", [-1, 64])
def test_streaming_kernel_with_k_split(ops, u, oracle, nbit, group_size, ways):
    """2, 4 or 8 wavefronts share a column group and split K (what one row of a narrow int4 matrix gets by itself):
    K shorter than the split, K that does not divide by it, one and two rows, ragged last workgroup."""
    from relax_amd import _lib

    L = _lib.lib()
    L.wq_debug_set_intb_gemv_k_split(ways)
    L.wq_debug_set_gemv_config(2, 0)
    try:
        for M, N, K in [(1, 64, 64), (2, 64, 128), (1, 320, 448), (1, 4096, 1024), (2, 1024, 4096), (1, 8192, 2112),
                        (1, 5120, 13824)]:
            print(f"intb k split {ways} nbit={nbit} g={group_size} M={M} N={N} K={K}", flush=True)
            _run(ops, u, oracle, M, N, K, nbit, seed=M + N + ways, group_size=group_size, bias="row", residual=True)
        L.wq_debug_set_gemv_config(1, 0)
        _run(ops, u, oracle, 1, 1024, 4096, nbit, seed=ways, group_size=group_size)
    finally:
        L.wq_debug_set_gemv_config(0, 0)
        L.wq_debug_set_intb_gemv_k_split(0)


@pytest.mark.parametrize("nbit", [8, 4])
def test_one_row_of_a_narrow_matrix(ops, u, oracle, nbit):
    """The automatic choice at M = 1 over widths on both sides of every threshold (int4: the streaming kernel with
    its own split of K; int8: the small-batch kernel below 8 wavefronts per CU)."""
    for N, K in [(1024, 4096), (4096, 4096), (5120, 13824), (8192, 8192), (12288, 4096), (22016, 4096)]:
        for g in (-1, 64):
            print(f"intb narrow nbit={nbit} g={g} N={N} K={K}", flush=True)
            _run(ops, u, oracle, 1, N, K, nbit, seed=N + K, group_size=g)


@pytest.mark.parametrize("cfg", [1, 2, 3, 4, 11, 12, 17, 18])
@pytest.mark.parametrize("nbit", [8, 4])
def test_gemm_tile_configurations(ops, u, oracle, nbit, cfg):
    """every tile shape of the register-staged (1-4) and the LDS-staged (11, 12, 17, 18) kernel, ragged M,
    N smaller than a tile, a bias per row and one per element."""
    from relax_amd import _lib

    _lib.lib().wq_debug_set_gemm_config(cfg)
    try:
        for M, N, K in [(70, 64, 64), (130, 320, 448), (257, 192, 1024), (300, 576, 512)]:
            print(f"intb cfg={cfg} nbit={nbit} M={M} N={N} K={K}", flush=True)
            _run(ops, u, oracle, M, N, K, nbit, seed=M + cfg)
        _run(ops, u, oracle, 100, 128, 256, nbit, seed=cfg, bias="row", activation="gelu", residual=True,
             binary_op="multiply", unary_op="relu")
        _run(ops, u, oracle, 100, 128, 256, nbit, seed=cfg + 1, bias="full")
        # fine-grained (group-64) scales through the same tiles
        for M, N, K in [(70, 64, 64), (130, 320, 448), (300, 576, 512)]:
            print(f"intb cfg={cfg} nbit={nbit} g=64 M={M} N={N} K={K}", flush=True)
            _run(ops, u, oracle, M, N, K, nbit, seed=M + cfg + 1, group_size=64)
        _run(ops, u, oracle, 100, 128, 256, nbit, seed=cfg + 2, group_size=64, bias="row", activation="relu")
    finally:
        _lib.lib().wq_debug_set_gemm_config(0)


@pytest.mark.parametrize("cfg", [4, 11, 17, 18, 19])
@pytest.mark.parametrize("activation", ["identity", "relu", "silu", "gelu"])
def test_gemm_epilogue_operands_at_any_address_and_stride(ops, u, oracle, cfg, activation):
    """A bias per element with rows of N and of N + 3 halves, and bias, residual and output one half off a 16-byte
    boundary; nothing before or behind the output is written."""
    import torch
    from relax_amd import _lib

    M, N, K = 300, 192, 256
    rng = np.random.default_rng(cfg)
    x, A, s = oracle.make_intb_inputs(M, N, K, 8, seed=cfg)
    P, dx, ds = ops.ft_preprocess_weight(u.dev(A), 80, False), u.dev(x), u.dev(s)
    row, res = rng.standard_normal(N).astype(np.float16), rng.standard_normal((M, N)).astype(np.float16)

    def off(a):  # the same values, two bytes off
        buf = torch.zeros(a.size + 8, dtype=torch.float16, device="cuda")
        buf[1:1 + a.size] = u.dev(a).reshape(-1)
        return buf

    L, act = _lib.lib(), ops.ACTIVATIONS[activation]
    L.wq_debug_set_gemm_config(cfg)
    try:
        for stride in (N, N + 3):
            full = rng.standard_normal((M, stride)).astype(np.float16)
            b, y = off(full), torch.zeros(M * N + 16, dtype=torch.float16, device="cuda")
            rc = L.wq_fpA_intB_gemm(dx.data_ptr(), P.data_ptr(), ds.data_ptr(), b[1:].data_ptr(), y[9:].data_ptr(), act, M, N,
                                    K, -1, stride, 8, 0, 0, torch.cuda.current_stream().cuda_stream)
            assert rc == 0
            ref = oracle.intb_linear(x, A, s, 8, bias=np.ascontiguousarray(full[:, :N]), bias_stride=N,
                                     activation=activation, nthreads=8)
            got = u.host(y)
            u.assert_close(got[9:9 + M * N].reshape(M, N), ref, f"cfg {cfg} {activation} stride {stride}")
            assert not got[:9].any() and not got[9 + M * N:].any()
        b, r, y = off(row), off(res), torch.zeros(M * N + 16, dtype=torch.float16, device="cuda")
        rc = L.wq_fpA_intB_gemm_residual(dx.data_ptr(), P.data_ptr(), ds.data_ptr(), b[1:].data_ptr(), r[1:].data_ptr(),
                                         y[9:].data_ptr(), act, ops.BINARY_OPS["plus"], ops.UNARY_OPS["relu"], M, N, K, -1, 8,
                                         0, 0, torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        ref = oracle.intb_linear(x, A, s, 8, bias=row, residual=res, activation=activation, binary_op="plus",
                                 unary_op="relu", nthreads=8)
        got = u.host(y)
        u.assert_close(got[9:9 + M * N].reshape(M, N), ref, f"cfg {cfg} {activation} residual")
        assert not got[:9].any() and not got[9 + M * N:].any()
    finally:
        L.wq_debug_set_gemm_config(0)


# K of one step per set of wavefronts, of fewer steps than the ring has slots, and of more
@pytest.mark.parametrize("K", [128, 256, 384, 1152])
@pytest.mark.parametrize("group_size", [-1, 64])
@pytest.mark.parametrize("nbit", [8, 4])
def test_k_halves_in_one_workgroup(ops, u, oracle, nbit, group_size, K):
    """128 x 128 tiles whose K-steps two sets of wavefronts share: whole tiles and row slices of them."""
    from relax_amd import _lib

    _lib.lib().wq_debug_set_gemm_config(19)
    try:
        for split in (1, 0):
            _lib.lib().wq_debug_set_gemm_tail_split(split)
            for M, N in [(70, 64), (130, 320), (300, 192)]:
                _run(ops, u, oracle, M, N, K, nbit, seed=M + K, group_size=group_size)
                _run(ops, u, oracle, M, N, K, nbit, seed=M + K + 1, group_size=group_size, bias="row", activation="gelu",
                     residual=True)
    finally:
        _lib.lib().wq_debug_set_gemm_tail_split(1)
        _lib.lib().wq_debug_set_gemm_config(0)


@pytest.mark.parametrize("M", [1, 16, 128, 256, 512])
def test_int8_full_size_sampled(ops, u, oracle, M):
    """K=8192, N=28672 int8 per-channel.  The oracle checks a sample of output columns
    (columns are independent given x), the one-hot test checks the layout end to end."""
    import torch

    K, N = 8192, 28672
    rng = np.random.default_rng(M)
    x = rng.standard_normal((M, K), dtype=np.float32).astype(np.float16)
    dA = torch.randint(-127, 128, (K, N), dtype=torch.int8, device="cuda")
    s = rng.uniform(0.001, 0.01, size=N).astype(np.float16)
    print(f"int8 full size M={M}", flush=True)
    P = ops.ft_preprocess_weight(dA, 80, False)
    got = u.host(ops.fpA_intB_gemm(u.dev(x), P, u.dev(s), weight_nbit=8))
    cols = np.concatenate([np.arange(0, 64), np.arange(14000, 14064), np.arange(N - 64, N)])
    A_cols = u.host(dA[:, torch.from_numpy(cols).cuda()].contiguous())
    # rows from every row tile of the kernels that serve these M (128 x 128, 256 x 128 and 256 x 256 tiles by M)
    rows = np.unique(np.clip(np.array([0, 7, 8, 15, 31, 32, 63, 64, 127, 128, 129, 255, 256, 300, 383, 384, 511]), 0, M - 1))
    ref = oracle.intb_linear(x[rows], A_cols, s[cols], 8, nthreads=8)
    u.assert_close(got[rows][:, cols], ref, f"int8 full M={M}")
    if M > 2:
        # every 61st row against the streaming kernel (an independent kernel), all columns
        pick = np.arange(0, M, 61)
        for r in pick:
            yv = u.host(ops.fpA_intB_gemm(u.dev(x[r:r + 1]), P, u.dev(s), weight_nbit=8))
            u.assert_close(got[r:r + 1], yv, f"int8 full M={M} row {r} vs gemv")
    if M == 1:
        # the reordered layout of the whole matrix (224 MiB), bit for bit against the oracle
        want_P = oracle.ft_preprocess(u.host(dA), False, 80)
        assert np.array_equal(u.host(P), want_P)
        del want_P
        xh = np.zeros((1, K), np.float16)
        xh[0, 4321] = 1
        y = u.host(ops.fpA_intB_gemm(u.dev(xh), P, u.dev(s), weight_nbit=8))
        want = (u.host(dA[4321]).astype(np.float16) * s)
        assert np.array_equal(y[0].view(np.uint16), want.view(np.uint16))


def test_reference_fixture_chain(ops, u, oracle):
    """The reference's own small test case (tests/python/relax/test_codegen_cutlass.py:1559-1609):
    np.random.seed(0); x = randn(64,64); y = normal(0, 0.002, (128,64)); bias = randn(1,128);
    residual = randn(64,128); encode -> preprocess -> fused GEMM, compared with the UNQUANTIZED
    np.dot(x, y.T) + bias (+ residual) at the reference's rtol = atol = 1e-2."""
    np.random.seed(0)
    x = np.random.randn(64, 64).astype("float16")
    y = np.random.normal(0, 0.002, size=(128, 64)).astype("float16")
    bias = np.random.randn(1, 128).astype("float16")
    residual = np.random.randn(64, 128).astype("float16")
    for nbit, tol in ((4, 1e-2), (8, 1e-2)):
        w, s = oracle.intb_encode(y, nbit)
        P = ops.ft_preprocess_weight(u.dev(w), 80, nbit == 4)
        out = u.host(ops.fpA_intB_gemm(u.dev(x), P, u.dev(s), bias=u.dev(bias), weight_nbit=nbit))
        ref = np.dot(x, y.transpose()) + bias
        np.testing.assert_allclose(out, ref, rtol=tol, atol=tol)
        out = u.host(ops.fpA_intB_gemm(u.dev(x), P, u.dev(s), bias=u.dev(bias), residual=u.dev(residual),
                                       weight_nbit=nbit, binary_op="plus"))
        np.testing.assert_allclose(out, ref + residual, rtol=tol, atol=tol)


def test_argument_errors(ops, u, oracle):
    from relax_amd._lib import WqError

    x, A, s = oracle.make_intb_inputs(2, 64, 64, 8, seed=0)
    P = ops.ft_preprocess_weight(u.dev(A), 80, False)
    with pytest.raises(WqError, match="group_size"):
        ops.fpA_intB_gemm(u.dev(x), P, u.dev(np.tile(s, 2)), weight_nbit=8, group_size=32)
    with pytest.raises(ValueError):
        ops.fpA_intB_gemm(u.dev(x[:, :32].copy()), P, u.dev(s), weight_nbit=8)
    with pytest.raises(ValueError):
        ops.fpA_intB_gemm(u.dev(x), P, u.dev(s[:10].copy()), weight_nbit=8)


@pytest.mark.parametrize("nbit", [8, 4])
def test_grouped_gemv_with_scales_at_any_alignment(ops, u, oracle, nbit):
    """group-64 scales: the streaming kernel fetches them as 8- or 16-byte vectors when the buffer is
    16-byte aligned and one by one otherwise; both must give the same result."""
    import torch

    M, N, K = 2, 192, 512
    x, A, s = oracle.make_intb_inputs(M, N, K, nbit, seed=5, group_size=64)
    P = ops.ft_preprocess_weight(u.dev(A), 80, nbit == 4)
    ref = oracle.intb_linear(x, A, s, nbit, group_size=64)
    aligned = u.dev(s)
    backing = torch.empty(s.size + 2, dtype=torch.float16, device="cuda")
    shifted = backing[2:].view(s.shape)  # 4 bytes past a 16-byte boundary
    shifted.copy_(aligned)
    assert aligned.data_ptr() % 16 == 0 and shifted.data_ptr() % 16 == 4
    got_a = ops.fpA_intB_gemm(u.dev(x), P, aligned, weight_nbit=nbit, group_size=64)
    got_s = ops.fpA_intB_gemm(u.dev(x), P, shifted, weight_nbit=nbit, group_size=64)
    assert torch.equal(got_a, got_s)
    u.assert_close(u.host(got_a), ref, f"grouped gemv int{nbit}")


@pytest.mark.parametrize("K", [192, 11008])
@pytest.mark.parametrize("group_size", [-1, 64])
@pytest.mark.parametrize("nbit", [8, 4])
def test_infinite_activations_where_the_steps_do_not_come_out_even(ops, u, nbit, group_size, K):
    """The small-batch kernel multiplies the first activations of a row once, not again by the zero weights past K."""
    import torch

    N = 128
    q = torch.full((K, N if nbit == 8 else N // 2), 3 if nbit == 8 else 0x33, dtype=torch.int8, device="cuda")
    B = ops.ft_preprocess_weight(q, 80, nbit == 4)
    s = torch.full((N,) if group_size <= 0 else (K // 64, N), 0.01, dtype=torch.float16, device="cuda")
    for M in (3, 16, 40, 64, 96):
        x = np.random.default_rng(M).standard_normal((M, K)).astype(np.float16)
        x[1, 0], x[2, 7] = np.inf, -np.inf
        got = u.host(ops.fpA_intB_gemm(u.dev(x), B, s, weight_nbit=nbit, group_size=group_size))
        assert np.all(got[1] == np.inf) and np.all(got[2] == -np.inf), M
        assert np.all(np.isfinite(got[3:])) and np.all(np.isfinite(got[0])), M


@pytest.mark.parametrize("M", [1, 40, 300])
def test_gelu_over_its_range(ops, u, M):
    """x[m] = (v, 0, ...), w = 1: gelu(v) itself, against 64 bits.  Bound: the rounding to fp16 (2^-11 of the value,
    2^-25 below the smallest normal number) and 2e-5 for the fp32 evaluation (1e-5 at v = -5.5)."""
    import torch
    from scipy.special import erfc

    N = K = 64
    v = np.concatenate([np.linspace(-8, 8, 64 * M - 5), [0.0, 100.0, -100.0, 60000.0, -60000.0]])
    v = v.astype(np.float16)[:: 64][:M] if M > 1 else np.array([-3.25], np.float16)
    if M > 4:
        v[:4] = [60000.0, -60000.0, 0.0, -5.5]
    x = np.zeros((M, K), np.float16)
    x[:, 0] = v
    q = torch.zeros((K, N), dtype=torch.int8, device="cuda")
    q[0] = 1
    B = ops.ft_preprocess_weight(q, 80, False)
    got = u.host(ops.fpA_intB_gemm(u.dev(x), B, torch.ones(N, dtype=torch.float16, device="cuda"), weight_nbit=8,
                                   activation="gelu", group_size=-1)).astype(np.float64)
    v = v.astype(np.float64)[:, None]
    ref = 0.5 * v * erfc(-v / np.sqrt(2))
    assert np.all(np.abs(got - ref) <= np.abs(ref) * (2.0**-11 + 2e-5) + 2.0**-25)
