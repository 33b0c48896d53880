"""The work that a user of this package has it do, as cases that can be timed and compared.

Every case is one layer (or half-layer) of a model served or evaluated in fp8, through the public entry points of
``flag_gems``, with what a serving program holds between calls (quantized weights and their scales, norm weights, the
RoPE cache) made beforehand:

  linear  one fp8 linear: quantize the activations per token and 128-group, multiply by the block-scaled weight
  mlp     a dense MLP: RMSNorm + quantizer, gate/up product, SiLU-and-mul + quantizer, down product
  scaled  a linear with one scale per token and one per output channel (fp8 or int8 operands, optional bias)
  moe     an expert layer: routing (softmax top-k, or DeepSeek-V3's group-limited top-k), then the fused experts
  oproj   DeepSeek-V4's grouped output projection: inverse RoPE + quantizer, then the batched "bhr,hdr->bhd" product

``rows`` is the number of tokens: 1 to a few dozen while decoding, hundreds to thousands while a prompt is processed.
"""
import math

import numpy as np
import torch

import flag_gems

_BLOCK = [128, 128]
_TYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # one token through DeepSeek-V3's fused q_a / kv_a projection: the smallest weight and the shortest launch, where
        # latency and what the host does per call count
        {"name": "linear_decode_1", "kind": "linear", "rows": 1, "n": 2112, "k": 7168, "type": "bf16", "ue8m0": False},
        # a decode batch of 61 sequences against DeepSeek-V3's largest projection: weight-bound, ragged row count
        {"name": "linear_batch_61", "kind": "linear", "rows": 61, "n": 7168, "k": 16384, "type": "bf16", "ue8m0": False},
        # a chunk of a prompt, or a large decode batch, between the weight-bound and the matrix-bound sizes
        {"name": "linear_chunk_333", "kind": "linear", "rows": 333, "n": 4608, "k": 7168, "type": "bf16", "ue8m0": False},
        # a whole prompt through the largest projection: matrix-bound
        {"name": "linear_prefill_4096", "kind": "linear", "rows": 4096, "n": 7168, "k": 16384, "type": "bf16", "ue8m0": False},
        # Llama-3-8B's MLP while decoding for 16 sequences: four launches, two large weights
        {"name": "mlp_decode_16", "kind": "mlp", "rows": 16, "hidden": 4096, "inter": 14336, "type": "bf16", "ue8m0": False},
        # DeepSeek-V3's MLP (one of eight tensor-parallel shards) on a ragged prompt, with the power-of-two scales that its
        # later checkpoints ask for
        {"name": "mlp_prefill_1000", "kind": "mlp", "rows": 1000, "hidden": 7168, "inter": 2304, "type": "bf16", "ue8m0": True},
        # per-token x per-channel fp8 linear with bias on a prompt chunk (cutlass_scaled_mm, 8192 x 8192)
        {"name": "scaled_fp8_256", "kind": "scaled", "rows": 256, "n": 8192, "k": 8192, "operand": "fp8", "bias": True, "type": "bf16"},
        # the same with int8 operands and no bias for a decode batch, fp16 results
        {"name": "scaled_int8_32", "kind": "scaled", "rows": 32, "n": 8192, "k": 8192, "operand": "int8", "bias": False, "type": "fp16"},
        # Mixtral-8x7B's expert layer while decoding: a few rows per expert, every expert's weights read
        {"name": "moe_8_decode_24", "kind": "moe", "rows": 24, "experts": 8, "hidden": 4096, "inter": 14336, "top_k": 2, "groups": 0, "type": "bf16"},
        # many small experts while decoding (512, top 10): about one row per expert that is hit
        {"name": "moe_512_decode_48", "kind": "moe", "rows": 48, "experts": 512, "hidden": 4096, "inter": 1024, "top_k": 10, "groups": 0, "type": "bf16"},
        # Mixtral's expert layer on a long prompt: matrix-bound, skewed expert loads
        {"name": "moe_8_prefill_4096", "kind": "moe", "rows": 4096, "experts": 8, "hidden": 4096, "inter": 14336, "top_k": 2, "groups": 0, "type": "bf16"},
        # attention output of a 500-token prompt chunk, 128 heads of 512 in 8 groups, onto 1024 columns per group
        {"name": "oproj_chunk_500", "kind": "oproj", "rows": 500, "heads": 128, "groups": 8, "d": 1024, "type": "bf16"},
    ]


def _spread(rng, lo, hi, step=1):
    """A whole number in [lo, hi], spread over its logarithm, rounded to a multiple of ``step``."""
    v = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return int(min(hi, max(lo, round(v / step) * step)))


# (n, k) of the linears in the benchmark and the tests: DeepSeek-V3, Llama-3 8B, Llama-3 70B, Qwen-2.5
_LINEARS = [(2112, 7168), (24576, 1536), (32768, 512), (7168, 16384), (4608, 7168), (7168, 2304), (576, 7168),
            (6144, 4096), (4096, 4096), (28672, 4096), (4096, 14336), (10240, 8192), (8192, 8192), (5120, 5120)]
_MLPS = [(4096, 14336), (7168, 2304), (8192, 3584), (5120, 1664), (4096, 1792)]
# experts, hidden, intermediate, top_k, groups of the router (0: softmax)
_LAYERS = [(8, 4096, 14336, 2, 0), (512, 4096, 1024, 10, 0), (256, 7168, 256, 8, 8), (64, 2048, 1408, 6, 0), (128, 2048, 768, 8, 0), (16, 4096, 6400, 2, 0)]
_MOST_FLOPS = 2.0 * 4096 * 2 * 3 * 4096 * 14336  # the largest listed case: Mixtral's layer on 4096 tokens


def _flops(c):
    if c["kind"] in ("linear", "scaled"):
        return 2.0 * c["rows"] * c["n"] * c["k"]
    if c["kind"] == "mlp":
        return 6.0 * c["rows"] * c["hidden"] * c["inter"]
    if c["kind"] == "moe":
        return 6.0 * c["rows"] * c["top_k"] * c["hidden"] * c["inter"]
    return 2.0 * c["rows"] * c["heads"] * 512 * c["d"]


def draw(rng):
    while True:
        kind = rng.choice(["linear", "linear", "linear", "linear", "mlp", "mlp", "scaled", "scaled", "moe", "moe", "moe", "oproj"])
        c = {"kind": kind, "rows": _spread(rng, 1, 4096)}
        if kind in ("linear", "scaled"):
            if rng.random() < 0.5:
                c["n"], c["k"] = rng.choice(_LINEARS)
            else:
                c["n"], c["k"] = _spread(rng, 512, 32768, 64), _spread(rng, 512, 16384, 128)
        if kind == "linear":
            c["ue8m0"] = rng.random() < 0.25
        elif kind == "scaled":
            c["operand"] = rng.choice(["fp8", "fp8", "int8"])
            c["bias"] = rng.random() < 0.5
        elif kind == "mlp":
            c["hidden"], c["inter"] = rng.choice(_MLPS) if rng.random() < 0.5 else (_spread(rng, 1024, 8192, 128), _spread(rng, 1024, 14336, 128))
            c["ue8m0"] = rng.random() < 0.25
        elif kind == "moe":
            c["experts"], c["hidden"], c["inter"], c["top_k"], c["groups"] = rng.choice(_LAYERS)
        else:
            c["heads"], c["groups"] = rng.choice([(128, 8), (64, 8), (64, 4), (16, 2)])
            c["d"] = rng.choice([512, 1024])
        c["type"] = rng.choice(["bf16", "bf16", "bf16", "fp16"])
        if _flops(c) <= _MOST_FLOPS:
            return c


def _rand(g, shape, std, dtype=torch.bfloat16):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32).mul_(std).to(dtype)


def _weight(g, n, k, ue8m0=False):
    """A linear's weight as a checkpoint holds it: e4m3fn codes and one scale per 128 x 128 block."""
    return flag_gems.per_block_cast_to_fp8(_rand(g, (n, k), 0.02), ue8m0, 128)


def _skew(experts):
    """Exponent of the experts' popularity: Zipf-like for Mixtral's few, mild where many experts are trained to balance."""
    return 1.1 if experts <= 16 else 0.2


def _expert_weights(g, experts, n, k):
    q = torch.empty((experts, n, k), device="cuda", dtype=torch.float8_e4m3fn)
    s = torch.empty((experts, -(-n // 128), k // 128), device="cuda", dtype=torch.float32)
    for e in range(experts):
        w = torch.empty((n, k), device="cuda", dtype=torch.bfloat16).normal_(0.0, 0.02, generator=g)
        q[e], s[e] = flag_gems.per_block_cast_to_fp8(w, False, 128)
    return q, s


def prepare(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind, rows, dtype = case["kind"], case["rows"], _TYPES[case["type"]]
    s = {"kind": kind, "case": case, "dtype": dtype}
    if kind == "linear":
        s["x"] = _rand(g, (rows, case["k"]), 1.0, dtype)
        s["w"], s["ws"] = _weight(g, case["n"], case["k"], case["ue8m0"])
    elif kind == "mlp":
        h, i = case["hidden"], case["inter"]
        s["x"] = _rand(g, (rows, h), 1.0, dtype)
        s["norm"] = (1.0 + _rand(g, (h,), 0.1, torch.float32)).to(dtype)
        s["w13"], s["w13s"] = _weight(g, 2 * i, h, case["ue8m0"])
        s["w2"], s["w2s"] = _weight(g, h, i, case["ue8m0"])
    elif kind == "scaled":
        n, k = case["n"], case["k"]
        x, w = _rand(g, (rows, k), 1.0, torch.float32), _rand(g, (n, k), 0.02, torch.float32)
        top, to = (448.0, torch.float8_e4m3fn) if case["operand"] == "fp8" else (127.0, torch.int8)
        s["sa"], s["sb"] = x.abs().amax(1, keepdim=True) / top, (w.abs().amax(1, keepdim=True) / top).t().contiguous()
        x, w = x / s["sa"], w / s["sb"].t()
        if to is torch.int8:
            x, w = x.round_(), w.round_()
        s["a"], s["b"] = x.to(to), w.to(to).t()  # b: [k, n], column-major
        s["bias"] = _rand(g, (n,), 1.0, dtype) if case["bias"] else None
    elif kind == "moe":
        e, h, i = case["experts"], case["hidden"], case["inter"]
        s["x"] = _rand(g, (rows, h), 1.0, dtype)
        # experts are not equally popular: popularity falls off as a power of the rank, the ranks dealt out at random
        skew = -_skew(e) * torch.log(1.0 + torch.randperm(e, generator=g, device="cuda").float())
        s["logits"] = _rand(g, (rows, e), 1.0, torch.float32) + skew
        s["router_bias"] = _rand(g, (e,), 0.01, torch.float32)
        s["w1"], s["w1s"] = _expert_weights(g, e, 2 * i, h)
        s["w2"], s["w2s"] = _expert_weights(g, e, h, i)
    else:
        heads, groups = case["heads"], case["groups"]
        s["o"] = _rand(g, (rows, heads, 512), 1.0, dtype)
        s["positions"] = torch.randint(0, 4096, (rows,), generator=g, device="cuda", dtype=torch.int64)
        angle = torch.arange(4096, device="cuda", dtype=torch.float32)[:, None] * 10000.0 ** (-torch.arange(32, device="cuda").float() / 32)
        s["cos_sin"] = torch.cat([angle.cos(), angle.sin()], dim=1).contiguous()
        d, r = case["d"], heads // groups * 512
        w, ws = _expert_weights(g, groups, d, r)
        s["w"], s["ws"] = w, ws
    return s


def _linear(xq, xs, w, ws, dtype, ue8m0):
    return flag_gems.w8a8_block_fp8_matmul(xq, w, xs, ws, _BLOCK, dtype, scales_are_powers_of_two=ue8m0)


def run(s):
    case, kind, dtype = s["case"], s["kind"], s["dtype"]
    if kind == "linear":
        xq, xs = flag_gems.per_token_group_quant_fp8(s["x"], 128, scale_ue8m0=case["ue8m0"])
        return _linear(xq, xs, s["w"], s["ws"], dtype, case["ue8m0"])
    if kind == "mlp":
        u = case["ue8m0"]
        xq, xs = flag_gems.rms_norm_per_token_group_quant_fp8(s["x"], s["norm"], 128, 1e-6, scale_ue8m0=u)
        gate_up = _linear(xq, xs, s["w13"], s["w13s"], dtype, u)
        aq, a_s = flag_gems.silu_and_mul_per_token_group_quant_fp8(gate_up, 128, scale_ue8m0=u)
        return _linear(aq, a_s, s["w2"], s["w2s"], dtype, u)
    if kind == "scaled":
        c = torch.empty((case["rows"], case["n"]), device="cuda", dtype=dtype)
        flag_gems.cutlass_scaled_mm(c, s["a"], s["b"], s["sa"], s["sb"], s["bias"])
        return c
    if kind == "moe":
        rows, k = case["rows"], case["top_k"]
        if case["groups"]:
            weights, ids = flag_gems.grouped_topk(s["logits"], case["groups"], 4, k, True, 2.5, s["router_bias"], 1)
        else:
            weights = torch.empty((rows, k), device="cuda", dtype=torch.float32)
            ids = torch.empty((rows, k), device="cuda", dtype=torch.int32)
            flag_gems.topk_softmax(weights, ids, torch.empty_like(ids), s["logits"], True)
        y = flag_gems.fused_experts_impl(s["x"], s["w1"], s["w2"], weights, ids, use_fp8_w8a8=True, block_shape=_BLOCK,
                                         w1_scale=s["w1s"], w2_scale=s["w2s"])
        return {"y": y, "weights": weights, "ids": ids}
    oq, o_s = flag_gems.fused_inv_rope_fp8_quant(s["o"], s["positions"], s["cos_sin"], case["groups"], case["heads"] // case["groups"])
    return flag_gems.fp8_einsum("bhr,hdr->bhd", oq, o_s, s["w"], s["ws"], _BLOCK, dtype)


def _experts_hit(experts, rows, k):
    """How many experts some token chooses (the others' weights are not read), under prepare()'s distribution."""
    rng = np.random.default_rng(0)
    skew = -_skew(experts) * np.log(1.0 + np.arange(experts))
    logits = rng.standard_normal((min(rows, 1024), experts), dtype=np.float32) + skew
    return len(np.unique(np.argpartition(-logits, k - 1, axis=1)[:, :k]))


def work(case):
    rows = case["rows"]
    kind = case["kind"]
    if kind == "linear":
        n, k = case["n"], case["k"]
        moved = 2 * rows * k + n * k + 4 * -(-n // 128) * (k // 128) + 2 * rows * n
    elif kind == "mlp":
        h, i = case["hidden"], case["inter"]
        moved = 4 * rows * h + 3 * h * i + 12 * h * i // 16384
    elif kind == "scaled":
        n, k = case["n"], case["k"]
        moved = rows * k + n * k + 4 * (rows + n) + 2 * rows * n + (2 * n if case["bias"] else 0)
    elif kind == "moe":
        e, h, i, k = case["experts"], case["hidden"], case["inter"], case["top_k"]
        hit = _experts_hit(e, rows, k)
        moved = 4 * rows * h + 4 * rows * e + 3 * hit * h * i
    else:
        r = case["heads"] * 512
        moved = 2 * rows * r + r * case["d"] + 2 * rows * case["groups"] * case["d"]
    return {"bytes": float(moved), "flops": _flops(case)}


def tolerance(case):
    # One product against the same sums in float64: relative error up to 3.3e-4, largest error 0.0151 (a bf16 step or two
    # next to a power of two).  Two products with a quantizer between them: 2.3e-3 and 0.043, a code of the second operand
    # that rounds the other way.  Four times that.
    return {"rel": 1e-2, "max": 0.17} if case["kind"] in ("mlp", "moe") else {"rel": 1.3e-3, "max": 0.06}
