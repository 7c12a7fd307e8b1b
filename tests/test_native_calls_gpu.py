"""The native form of the linears of ops.py: it takes plain calls, gives what the general path gives, and leaves every other call
to the general path."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def env():
    from relax_amd import _lib, ops

    g = torch.Generator(device="cuda").manual_seed(1)
    half = lambda *s: (torch.rand(s, device="cuda", generator=g) - 0.5).half()
    words = lambda *s: torch.randint(-(2**31), 2**31 - 1, s, device="cuda", dtype=torch.int32, generator=g)
    N, K = 256, 512
    prep = lambda order: ops.gptq_prepare(words(K // 8, N), words(K // 128, N // 8), half(K // 128, N), order)
    rows = torch.arange(K, device="cuda", dtype=torch.int32) // 128
    B = torch.randint(-128, 127, (K, N), device="cuda", dtype=torch.int8, generator=g)
    forms = {
        "q4": (lambda x, **k: ops.q4g32_linear(W, S, x, **k)),
        "intb": (lambda x, **k: ops.fpA_intB_gemm(x, B, half_scales, weight_nbit=8, activation="silu", **k)),
        "gptq": (lambda x, **k: ops.gptq_linear(plain, x, **k)),
        "gptq-order": (lambda x, **k: ops.gptq_linear(ordered, x, **k)),
    }
    W, S, half_scales = words(N, K // 8), half(N, K // 32), half(N)
    plain, ordered = prep(rows), prep(rows.flip(0).contiguous())
    return _lib, ops, forms, half, N, K


class _Watch:  # every call with its answer
    def __init__(self, monkeypatch, module):
        self.answers = []
        self.real = module
        for name in ("q4g32_linear", "fpA_intB_gemm", "gptq_linear"):
            setattr(self, name, lambda *a, f=getattr(module, name): self.answers.append(f(*a)) or self.answers[-1])


@pytest.mark.parametrize("form", ["q4", "intb", "gptq", "gptq-order"])
@pytest.mark.parametrize("shape", [(1,), (3, 5), (70,)])
def test_taken_and_left(env, monkeypatch, form, shape):
    from torch.utils._python_dispatch import TorchDispatchMode

    _lib, ops, forms, half, N, K = env
    run, x, bias, res = forms[form], half(*shape, K), half(N), half(*shape, N)
    watch = _Watch(monkeypatch, _lib.calls())
    monkeypatch.setattr(_lib, "_calls", watch)

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Sub(torch.Tensor):
        pass

    for kw in ({}, {"bias": bias}, {"residual": res}, {"bias": bias, "residual": res}):
        y = run(x, **kw)
        assert watch.answers[-1] is y and y.shape == (*shape, N) and y.dtype == torch.float16
        with Mode():  # watched: the general path
            want = run(x, **kw)
        assert watch.answers[-1] is None and torch.equal(y, want)
        assert torch.equal(run(x.as_subclass(Sub), **kw), want) and watch.answers[-1] is None
        out = torch.empty_like(y)
        assert run(x, out=out, **kw) is out and torch.equal(out, want)
    n = len(watch.answers)
    for bad in (x.float(), x.cpu(), half(*shape, K + 8), half(*shape, 2 * K)[..., ::2]):
        with pytest.raises(ValueError):
            run(bad)
        assert watch.answers[-1] is None
    with pytest.raises(ValueError):
        run(x, residual=half(*shape, N + 1))
    assert watch.answers[n:] == [None] * 5
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        y = run(x)
    torch.cuda.current_stream().wait_stream(side)
    assert watch.answers[-1] is y and torch.equal(y, run(x))


@pytest.mark.parametrize("form", ["q4", "intb", "gptq", "gptq-order"])
@pytest.mark.parametrize("rows", [1, 70])
def test_a_short_bias_is_refused(env, form, rows):
    from torch.utils._python_dispatch import TorchDispatchMode

    class Mode(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    _, _, forms, half, N, K = env
    x, bias = half(rows, K), half(N)[: N - 1]
    with pytest.raises(ValueError):
        forms[form](x, bias=bias)
    with Mode(), pytest.raises(ValueError):  # the general path
        forms[form](x, bias=bias)


def test_gptq_linear_refuses_host_tensors_to_write_to(env):
    _, ops, forms, half, N, K = env
    for form in ("gptq", "gptq-order"):
        x = half(3, K)
        for kw in ({"out": half(3, N).cpu()}, {"workspace": torch.empty(1 << 16, dtype=torch.uint8)}):
            with pytest.raises(ValueError):
                forms[form](x, **kw)
        out = torch.empty(3, N, dtype=torch.float16, pin_memory=True)  # which the device can write
        assert forms[form](x, out=out) is out
        torch.cuda.synchronize()
        assert torch.equal(out, forms[form](x).cpu())
