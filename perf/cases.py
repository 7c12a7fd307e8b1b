"""The measured workloads of the weight-only quantized linear path.

Each case is one call (or one list launch) of the torch front end as a serving program makes it: weights are packed,
reordered and kept on the device, activations and the output tensor are new for every call.  Shapes are those of
bench.py and of the tests: the linears of a Llama-2-7B-shaped decoder layer (4096 -> 12288, 4096 -> 4096,
4096 -> 22016, 11008 -> 4096) and the 8192 -> 28672 matrix of the fpA_intB configuration.
"""
import math

import torch

from relax_amd import ops

GROUP = 32  # q4f16_1


def listed():
    return [
        # one decode linear called by itself (o_proj): a small matrix, so launch latency and the host path count
        {"name": "decode_one", "kind": "q4", "M": 1, "N": 4096, "K": 4096, "bias": False, "residual": False},
        # the four linears of a decoder layer for one sequence, one launch
        {"name": "decode_layer", "kind": "list", "M": 1, "hidden": 4096, "ffn": 11008, "layers": 1},
        # one decode step of the whole 32-layer stack for a batch of 8 sequences
        {"name": "decode_stack_b8", "kind": "list", "M": 8, "hidden": 4096, "ffn": 11008, "layers": 32},
        # rows of several drafted tokens or of a ragged small batch through the fused qkv projection
        {"name": "rows_19", "kind": "q4", "M": 19, "N": 12288, "K": 4096, "bias": False, "residual": True},
        # a short prompt, or a chunk of one, through a projection with bias
        {"name": "chunk_200", "kind": "q4", "M": 200, "N": 11008, "K": 4096, "bias": True, "residual": False},
        # prefill of 2048 tokens, down projection with the residual add
        {"name": "prefill_2048", "kind": "q4", "M": 2048, "N": 4096, "K": 11008, "bias": False, "residual": True},
        # prefill of a large batch of prompts, fused gate / up projection
        {"name": "prefill_8192", "kind": "q4", "M": 8192, "N": 22016, "K": 4096, "bias": False, "residual": False},
        # fpA_intB, int8 per column: decode of one sequence with a bias
        {"name": "int8_decode", "kind": "intb", "M": 1, "N": 28672, "K": 8192, "nbit": 8, "group": -1, "bias": True,
         "activation": "identity", "residual": False},
        # fpA_intB, int8 per column: a batch of 128 with bias and gelu fused
        {"name": "int8_gelu_128", "kind": "intb", "M": 128, "N": 28672, "K": 8192, "nbit": 8, "group": -1, "bias": True,
         "activation": "gelu", "residual": False},
        # fpA_intB, int4 with a scale per 64 rows: a prompt of 500 tokens, residual add fused
        {"name": "int4_group_500", "kind": "intb", "M": 500, "N": 28672, "K": 8192, "nbit": 4, "group": 64, "bias": False,
         "activation": "identity", "residual": True},
        # an AutoGPTQ layer stored in activation order, a batch of 8
        {"name": "gptq_order_8", "kind": "gptq", "M": 8, "N": 12288, "K": 4096, "group": 128, "order": True,
         "residual": False},
        # quantizing a weight when a model is loaded
        {"name": "quantize", "kind": "encode", "N": 11008, "K": 4096},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["q4", "q4", "q4", "q4", "list", "list", "intb", "intb", "intb", "gptq", "encode"])
    if kind == "list":
        hidden = 128 * _log_int(rng, 8, 64)
        ffn = 32 * int(hidden * rng.uniform(2.0, 3.6) / 32)
        per_layer = 0.5625 * hidden * (4 * hidden + 3 * ffn)
        return {"kind": kind, "M": _log_int(rng, 1, 32), "hidden": hidden, "ffn": ffn,
                "layers": min(_log_int(rng, 1, 32), max(1, int(3.0e9 / per_layer)))}
    K = 32 * _log_int(rng, 32, 448)
    N = _log_int(rng, 1024, 28672)
    if kind == "q4":
        if rng.random() < 0.8:
            N = N // 8 * 8
        if rng.random() < 0.7:
            K = (K + 63) // 64 * 64
        M = min(_log_int(rng, 1, 8192), int(7.0e11 / (2.0 * N * K)))
        return {"kind": kind, "M": M, "N": N, "K": K, "bias": rng.random() < 0.4, "residual": rng.random() < 0.4}
    if kind == "intb":
        N, K = (N + 63) // 64 * 64, (K + 63) // 64 * 64
        M = min(_log_int(rng, 1, 2048), int(7.0e11 / (2.0 * N * K)))
        return {"kind": kind, "M": M, "N": N, "K": K, "nbit": rng.choice([8, 8, 4]), "group": rng.choice([-1, -1, 64]),
                "bias": rng.random() < 0.5, "activation": rng.choice(["identity", "identity", "relu", "silu", "gelu"]),
                "residual": rng.random() < 0.4}
    if kind == "gptq":
        return {"kind": kind, "M": _log_int(rng, 1, 512), "N": N // 8 * 8, "K": (K + 127) // 128 * 128, "group": 128,
                "order": rng.random() < 0.5, "residual": rng.random() < 0.4}
    return {"kind": kind, "N": N, "K": K}


def _layer_shapes(case):
    h, f = case["hidden"], case["ffn"]
    return (("qkv", 3 * h, h), ("o", h, h), ("gate_up", 2 * f, h), ("down", h, f))


class _Random:
    """Inputs on the device, from the seed alone."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda")
        self.g.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(shape, device="cuda", dtype=torch.float16, generator=self.g)

    def uniform(self, lo, hi, *shape):
        return (torch.rand(shape, device="cuda", generator=self.g) * (hi - lo) + lo).to(torch.float16)

    def words(self, *shape):
        return torch.randint(-2**31, 2**31 - 1, shape, dtype=torch.int32, device="cuda", generator=self.g)

    def q4(self, N, K):
        return self.words(N, K // 8), self.uniform(0.005, 0.02, N, K // GROUP)


def _prepare_list(case, r):
    # qkv reads the hidden state (the down projection of the layer before), o the attention output, gate / up the
    # output of o, down the gated activations; what attention and gating would compute comes in as data
    M, h, f, L = case["M"], case["hidden"], case["ffn"], case["layers"]
    hidden, attn, act = r.normal(M, h), r.normal(L, M, h), r.normal(L, M, f)
    out = {name: torch.empty((L, M, N), device="cuda", dtype=torch.float16) for name, N, _ in _layer_shapes(case)}
    linears = []
    for l in range(L):
        x = {"qkv": out["down"][l - 1] if l else hidden, "o": attn[l], "gate_up": out["o"][l], "down": act[l]}
        for name, N, K in _layer_shapes(case):
            linears.append((*r.q4(N, K), x[name], out[name][l]))
    return {"list": ops.Q4G32GemvList(linears, M=M), "out": out}


def prepare(case, seed):
    r = _Random(seed)
    s = {"case": case}
    kind, M, N, K = case["kind"], case.get("M"), case.get("N"), case.get("K")
    if kind == "list":
        s.update(_prepare_list(case, r))
        return s
    if kind == "encode":
        s["Wf"] = (r.normal(N, K) * 0.05).contiguous()
        return s
    s["x"] = r.normal(M, K)
    s["bias"] = r.normal(N) if case.get("bias") else None
    s["residual"] = r.normal(M, N) if case.get("residual") else None
    if kind == "q4":
        s["W"], s["S"] = r.q4(N, K)
    elif kind == "intb":
        nbit, group = case["nbit"], case["group"]
        lo = -127 if nbit == 8 else -128
        q = torch.randint(lo, 128, (K, N if nbit == 8 else N // 2), dtype=torch.int8, device="cuda", generator=r.g)
        s["B"] = ops.ft_preprocess_weight(q, 80, nbit == 4)
        s["scales"] = r.uniform(0.001, 0.01, *((N,) if group <= 0 else (K // group, N)))
    elif kind == "gptq":
        G = K // case["group"]
        g_idx = torch.arange(K, device="cuda", dtype=torch.int32) // case["group"]
        if case["order"]:
            g_idx = g_idx[torch.randperm(K, device="cuda", generator=r.g)].contiguous()
        s["w"] = ops.gptq_prepare(r.words(K // 8, N), r.words(G, N // 8), r.uniform(0.005, 0.02, G, N), g_idx)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "q4":
        return ops.q4g32_linear(s["W"], s["S"], s["x"], bias=s["bias"], residual=s["residual"])
    if kind == "list":
        s["list"].run()
        return s["out"]
    if kind == "intb":
        return ops.fpA_intB_gemm(s["x"], s["B"], s["scales"], bias=s["bias"], residual=s["residual"],
                                 weight_nbit=case["nbit"], activation=case["activation"], group_size=case["group"])
    if kind == "gptq":
        return ops.gptq_linear(s["w"], s["x"], residual=s["residual"])
    return ops.q4g32_encode(s["Wf"])


def _linear_work(M, N, K, weight_bytes, extra=0):
    return weight_bytes + 2.0 * (M * K + M * N + extra), 2.0 * M * N * K


def work(case):
    kind = case["kind"]
    if kind == "encode":
        N, K = case["N"], case["K"]
        return {"bytes": N * K * (2.0 + 0.5 + 2.0 / GROUP), "flops": 0.0}
    M = case["M"]
    if kind == "list":
        parts = [_linear_work(M, N, K, N * K * (0.5 + 2.0 / GROUP)) for _, N, K in _layer_shapes(case)]
        return {"bytes": case["layers"] * sum(p[0] for p in parts), "flops": case["layers"] * sum(p[1] for p in parts)}
    N, K = case["N"], case["K"]
    extra = (N if case.get("bias") else 0) + (M * N if case.get("residual") else 0)
    if kind == "q4":
        w = N * K * (0.5 + 2.0 / GROUP)
    elif kind == "intb":
        w = N * K * case["nbit"] / 8.0 + 2.0 * N * (1 if case["group"] <= 0 else K // case["group"])
    else:
        w = N * K * 0.5 + 2.5 * N * (K // case["group"]) + (4.0 * K if case["order"] else 0)
    b, f = _linear_work(M, N, K, w, extra)
    return {"bytes": b, "flops": f}


def tolerance(case):
    # codes and scales of the quantizer are exact by definition
    if case["kind"] == "encode":
        return "exact"
    # fp16 outputs of fp32 sums.  Against the same product in 64 bits: 2.1e-4 where every weight is rounded to fp16
    # once, 2.8e-4 where the scale is factored out of a group, 3.0e-4 with a residual added in fp16; the largest
    # single difference 1.2e-3 .. 2.0e-3 of the root mean square.  Four times that.
    return {"rel": 1.2e-3, "max": 8e-3}
