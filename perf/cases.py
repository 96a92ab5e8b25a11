"""The calls whose speed this package is judged by, as a serving program makes them.

A case is one pass of one of five paths, named by ``op``:

* ``dynamic_quant``  per-token int8 quantisation of an activation matrix [M, K], optionally with smooth scales;
* ``quant_matmul``   int8 activations [M, K] x int8 weight stored [N, K], per-token and per-channel scales, bf16 or fp16 out;
* ``linear_quant``   the ``LinearQuant`` module as constructed by default: int32 bias, no per-token scales, fp16 out;
* ``weight_quant``   bf16 / fp16 activations x int8 (per channel) or int4 (groups of 128) weight, either through the operator
                     with the weight along N ("kn") or through the layout ``LinearWeightQuant`` stores ("nk");
* ``mlp``            a W8A8 decoder MLP: quantise, gate|up product, SwiGLU + quantise, down product.

M is the number of tokens in flight: 1 for one sequence being decoded, tens to a few hundred for a decode batch, any number
up to a few thousand for a prefill.  K and N are layer widths.
"""
from __future__ import annotations

import math

import torch

import pytorch_amd as pa
from pytorch_amd.contrib.module import LinearQuant, LinearWeightQuant

_DT = {"bf16": torch.bfloat16, "fp16": torch.float16}
_GROUP = 128                       # int4 scale groups
_MAX_TOKENS = 2048
# no drawn case does more than the largest listed one (int8 operations of the MLP at 2048 tokens); 16-bit products count
# several times because the card is that much slower at them
_MAX_INT8_MACS = 3 * 2048 * 4096 * 14336
_MAX_16BIT_MACS = 4.0e10


def listed():
    return [
        # one new token's activations before a projection: the smallest call of a decode step
        {"name": "dq_one_token", "op": "dynamic_quant", "M": 1, "K": 4096, "dtype": "bf16", "smooth": False},
        # a prefill's activations: the quantisation in front of every W8A8 projection
        {"name": "dq_prefill", "op": "dynamic_quant", "M": 2048, "K": 4096, "dtype": "bf16", "smooth": False},
        # fused q|k|v projection of a small decode batch
        {"name": "qmm_decode_16", "op": "quant_matmul", "M": 16, "K": 4096, "N": 6144, "dtype": "bf16", "bias": False},
        # down projection of a large decode batch
        {"name": "qmm_decode_128", "op": "quant_matmul", "M": 128, "K": 14336, "N": 4096, "dtype": "bf16", "bias": False},
        # up projection of a prefill with bias: the W8A8 benchmark shape
        {"name": "qmm_prefill_1024", "op": "quant_matmul", "M": 1024, "K": 4096, "N": 11008, "dtype": "bf16", "bias": True},
        # a prompt of arbitrary length through the module's own forward
        {"name": "linear_quant_777", "op": "linear_quant", "M": 777, "K": 11008, "N": 4096},
        # weight-only int8 decode of a wide model's up projection, weight [K, N]
        {"name": "w8a16_decode_16", "op": "weight_quant", "M": 16, "K": 8192, "N": 28672, "bits": 8, "layout": "kn", "dtype": "bf16"},
        # weight-only int4 decode of one sequence, and of a large batch
        {"name": "w4a16_one_token", "op": "weight_quant", "M": 1, "K": 4096, "N": 14336, "bits": 4, "layout": "kn", "dtype": "bf16"},
        {"name": "w4a16_decode_128", "op": "weight_quant", "M": 128, "K": 4096, "N": 14336, "bits": 4, "layout": "kn", "dtype": "bf16"},
        # weight-only int8 prefill through the module, float16
        {"name": "w8a16_module_1024", "op": "weight_quant", "M": 1024, "K": 11264, "N": 1664, "bits": 8, "layout": "nk", "dtype": "fp16"},
        # a whole W8A8 MLP, decode batch and prefill
        {"name": "mlp_decode_64", "op": "mlp", "M": 64, "K": 4096, "N": 14336},
        {"name": "mlp_prefill_2048", "op": "mlp", "M": 2048, "K": 4096, "N": 14336},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, step=128):
    """A layer width: mostly a multiple of 128, now and then one that is only a multiple of 16."""
    w = _log_int(rng, lo, hi)
    step = 16 if rng.random() < 0.25 and step == 128 else step
    return max(lo, w // step * step)


def draw(rng):
    op = rng.choice(["dynamic_quant", "quant_matmul", "quant_matmul", "linear_quant", "weight_quant", "weight_quant", "mlp"])
    m = _log_int(rng, 1, _MAX_TOKENS)
    if op == "dynamic_quant":
        k = _width(rng, 1024, 14336)
        if rng.random() < 0.15:
            k += rng.randrange(1, 16)                    # a row length no vector width divides
        return {"op": op, "M": m, "K": k, "dtype": rng.choice(["bf16", "fp16"]), "smooth": rng.random() < 0.3}
    if op == "mlp":
        k = _width(rng, 1024, 4096, 256)
        n = int(k * rng.uniform(2.5, 3.5)) // 256 * 256
        return {"op": op, "M": m, "K": k, "N": n}
    if op == "weight_quant":
        bits, layout = rng.choice([4, 8]), rng.choice(["kn", "nk"])
        k = _width(rng, 1024, 14336, _GROUP if bits == 8 else 256)
        n = _width(rng, 1024, 16384)
        m = max(1, min(m, int(_MAX_16BIT_MACS / (k * n))))
        return {"op": op, "M": m, "K": k, "N": n, "bits": bits, "layout": layout, "dtype": rng.choice(["bf16", "fp16"])}
    k, n = _width(rng, 1024, 14336), _width(rng, 1024, 28672)
    m = max(1, min(m, int(_MAX_INT8_MACS / (k * n))))
    if op == "linear_quant":
        return {"op": op, "M": m, "K": k, "N": n}
    return {"op": op, "M": m, "K": k, "N": n, "dtype": rng.choice(["bf16", "fp16"]), "bias": rng.random() < 0.5}


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(int(seed))
    op, M, K = case["op"], case["M"], case["K"]

    def normal(*shape):
        return torch.randn(*shape, generator=g, device=dev)

    def uniform(lo, hi, *shape):
        return torch.rand(*shape, generator=g, device=dev) * (hi - lo) + lo

    def codes(*shape):
        # what symmetric quantisation leaves of bell-shaped values: the row's largest sits near 4 sigma = 127
        return torch.empty(*shape, device=dev, dtype=torch.float16).normal_(0.0, 32.0, generator=g).round_().clamp_(-127, 127).to(torch.int8)

    def activations(dtype):
        x = normal(M, K)
        return torch.where(torch.rand(M, K, generator=g, device=dev) < 1e-3, x * 50.0, x).to(dtype)   # a few outliers

    if op == "dynamic_quant":
        dt = _DT[case["dtype"]]
        return {"op": op, "x": activations(dt), "smooth": uniform(0.5, 2.0, K).to(dt) if case["smooth"] else None}
    if op == "quant_matmul":
        N, dt = case["N"], _DT[case["dtype"]]
        return {"op": op, "x": codes(M, K), "w": codes(N, K).t(), "scale": uniform(1e-3, 1e-2, N),
                "pertoken": uniform(1e-3, 1e-2, M), "dtype": dt,
                "bias": (normal(N) * 0.02).to(dt if dt == torch.bfloat16 else torch.float32) if case["bias"] else None}
    if op == "linear_quant":
        N = case["N"]
        mod = LinearQuant(K, N, bias=True, output_dtype=torch.float16)
        mod.weight.data, mod.scale.data = codes(N, K), uniform(1e-5, 1e-4, N)
        mod.bias.data = torch.randint(-20000, 20000, (N,), generator=g, device=dev, dtype=torch.int32)
        return {"op": op, "x": codes(M, K), "mod": mod}
    if op == "weight_quant":
        N, dt, bits = case["N"], _DT[case["dtype"]], case["bits"]
        groups = K // _GROUP if bits == 4 else 1
        nk = case["layout"] == "nk"
        rows, cols = (N, K) if nk else (K, N)
        if bits == 8:
            w = torch.randint(-127, 128, (rows, cols), generator=g, device=dev, dtype=torch.int8)
        else:
            w = torch.randint(-2 ** 31, 2 ** 31, (rows, cols // 8), generator=g, device=dev, dtype=torch.int64).to(torch.int32)
        pshape = (groups, N) if bits == 4 and not nk else (N, groups) if bits == 4 else (N,)
        off = 4.0 if bits == 8 else 2.0
        x, scale, offset = normal(M, K).to(dt), uniform(1e-3, 1e-2, *pshape).to(dt), uniform(-off, off, *pshape).to(dt)
        if nk:
            mod = LinearWeightQuant(K, N, bias=False, antiquant_offset=True, antiquant_group_size=_GROUP if bits == 4 else 0,
                                    device="meta")
            mod.weight = torch.nn.Parameter(w, requires_grad=False)
            mod.antiquant_scale = torch.nn.Parameter(scale, requires_grad=False)
            mod.antiquant_offset = torch.nn.Parameter(offset, requires_grad=False)
            return {"op": op, "x": x, "mod": mod}
        return {"op": op, "x": x, "mod": None, "w": w, "scale": scale, "offset": offset, "group": _GROUP if bits == 4 else 0}
    N = case["N"]
    return {"op": op, "x": normal(M, K).to(torch.bfloat16), "w1": codes(2 * N, K).t(), "w2": codes(K, N).t(),
            "s1": uniform(1e-4, 1e-3, 2 * N), "s2": uniform(1e-4, 1e-3, K)}


def run(state):
    op, x = state["op"], state["x"]
    if op == "dynamic_quant":
        return pa.npu_dynamic_quant(x, smooth_scales=state["smooth"])
    if op == "quant_matmul":
        return pa.npu_quant_matmul(x, state["w"], state["scale"], pertoken_scale=state["pertoken"], bias=state["bias"],
                                   output_dtype=state["dtype"])
    if op == "linear_quant":
        return state["mod"](x)
    if op == "weight_quant":
        if state["mod"] is not None:
            return state["mod"](x)
        return pa.npu_weight_quant_batchmatmul(x, state["w"], state["scale"], state["offset"], None, None, None, state["group"])
    xq, xs = pa.npu_dynamic_quant(x)
    gu = pa.npu_quant_matmul(xq, state["w1"], state["s1"], pertoken_scale=xs, output_dtype=torch.bfloat16)
    aq, a_s = pa.npu_swiglu_quant(gu, activate_left=True, quant_mode=1)
    return pa.npu_quant_matmul(aq, state["w2"], state["s2"], pertoken_scale=a_s, output_dtype=torch.bfloat16)


def work(case):
    op, M, K = case["op"], case["M"], case["K"]
    if op == "dynamic_quant":
        return {"bytes": 3 * M * K + 4 * M + (2 * K if case["smooth"] else 0), "flops": 3 * M * K}
    N = case["N"]
    if op == "mlp":
        return {"bytes": 3 * K * N + 4 * (2 * N + K) + 4 * M * K, "flops": 6 * M * K * N}
    if op == "quant_matmul":
        bias = 0 if not case["bias"] else 2 * N if case["dtype"] == "bf16" else 4 * N
        return {"bytes": M * K + K * N + 2 * M * N + 4 * (M + N) + bias, "flops": 2 * M * K * N}
    if op == "linear_quant":
        return {"bytes": M * K + K * N + 2 * M * N + 8 * N, "flops": 2 * M * K * N}
    groups = K // _GROUP if case["bits"] == 4 else 1
    return {"bytes": 2 * M * K + K * N * case["bits"] // 8 + 2 * M * N + 4 * groups * N, "flops": 2 * M * K * N}


def tolerance(case):
    if case["op"] == "dynamic_quant":
        return "exact"                                   # codes and scales are defined bit for bit
    if case["op"] == "mlp":
        return {"rel": 1e-2, "max": 0.1}                 # one ulp of the bf16 activation may move an int8 code
    half = case["op"] == "linear_quant" or case["dtype"] == "fp16"
    # 32-bit (or exact integer) sums and one rounding to the output type: a few values land on the other side of a tie
    return {"rel": 5e-4, "max": 2e-3} if half else {"rel": 4e-3, "max": 1.6e-2}
