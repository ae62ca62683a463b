"""The work whose speed this framework is judged by: what a program that runs quantized linear layers and mixtures of
experts on one MI355X asks of it, through the public entry points, from one decode step to a large prefill.

A case is a dict: its ``kind`` says which part of a model it is, the rest are sizes, types and options.

  nvfp4_linear  activations are quantized to NVFP4 with a calibrated global scale and multiplied with NVFP4 weights
  mxfp8_linear  the same in MXFP8 (e4m3 with e8m0 scales per 32)
  nvfp4_mlp     two NVFP4 layers in a row; the first one's product leaves its GEMM quantized to NVFP4
  nvfp4_moe     a SwiGLU expert layer: gate and up projections, silu(gate) * up quantized, down projection
  nvfp4_expert_linear  one expert projection through the registered operator of the inference layers
  expert_mm     one expert projection in bf16 or f16
  quantize      a tensor is quantized: NVFP4 with a global scale computed on the way, or MXFP8

Sizes are those of the repository's benchmark and tests and whatever lies between them.  Expert loads are drawn from an
even or a Zipf(1.1) routing; which expert has which load depends on the seed, the loads themselves only on the case, so
that a case costs the same for every seed.
"""
import math
import random

import torch

from fuser_amd import nvf_cutlass, ops
from fuser_amd.custom_ops import compute_auxiliary_tensors, f16a_nvfp4weight_scaled_grouped_mm

DEV = "cuda"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BYTES = {"bf16": 2, "f16": 2, "f32": 4}
FP4 = 0.5 + 1 / 16  # bytes per element of an NVFP4 tensor: payload and block scales
FP8 = 1 + 1 / 32    # ... of an MXFP8 tensor


def listed():
    return [
        # one decode step of 16 sequences through a dense projection: launches and latency
        dict(name="nvfp4_linear_decode", kind="nvfp4_linear", m=16, n=4096, k=4096, dtype="bf16"),
        # a prefill of 2048 tokens through an up projection
        dict(name="nvfp4_linear_prefill", kind="nvfp4_linear", m=2048, n=14336, k=4096, dtype="bf16"),
        # a decode step of a large batch that is no multiple of a tile, down projection, f16
        dict(name="mxfp8_linear_decode", kind="mxfp8_linear", m=100, n=4096, k=14336, dtype="f16"),
        # a ragged number of tokens through a layer whose K is no multiple of 128
        dict(name="mxfp8_linear_ragged", kind="mxfp8_linear", m=1000, n=5760, k=2880, dtype="bf16"),
        # the headline size of the dense GEMM, with the quantization of its activations
        dict(name="mxfp8_linear_large", kind="mxfp8_linear", m=8192, n=8192, k=8192, dtype="bf16"),
        # up and down projection of a feed-forward block for a chunk of 512 tokens, the product between them kept in NVFP4
        dict(name="nvfp4_mlp_chunk", kind="nvfp4_mlp", m=512, hidden=4096, inter=14336, dtype="bf16"),
        # a prefill of 8192 tokens, 8 of 256 experts each
        dict(name="nvfp4_moe_prefill", kind="nvfp4_moe", m=65536, hidden=7168, inter=2048, experts=256, zipf=True, dtype="bf16"),
        # a decode step of 64 sequences over the same experts
        dict(name="nvfp4_moe_decode", kind="nvfp4_moe", m=512, hidden=7168, inter=2048, experts=256, zipf=True, dtype="bf16"),
        # a chunk of 500 tokens, 4 of 32 experts each, widths that are no multiple of the large tiles
        dict(name="nvfp4_expert_linear_chunk", kind="nvfp4_expert_linear", m=2000, n=5760, k=2880, experts=32, zipf=False,
             dtype="bf16"),
        # a prefill over 8 experts in bf16
        dict(name="expert_mm_prefill", kind="expert_mm", m=8192, n=14336, k=4096, experts=8, zipf=True, dtype="bf16"),
        # a decode step of 64 sequences, 2 of 8 experts each, in bf16
        dict(name="expert_mm_decode", kind="expert_mm", m=128, n=14336, k=4096, experts=8, zipf=False, dtype="bf16"),
        # all activations of a prefill quantized with a scale of their own
        dict(name="nvfp4_quantize_large", kind="quantize", rows=65536, cols=7168, fmt="nvfp4", dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi, steps):
    """A width between lo and hi, a multiple of one of `steps`: mostly of the larger ones, as model widths are."""
    step = rng.choice(steps)
    return min(hi, max(lo, -(-_log(rng, lo, hi) // step) * step)) // step * step


def draw(rng):
    """A case of the same kinds and ranges, redrawn while it would cost more than four fifths of the largest listed one."""
    largest = [max(work(c)[key] for c in listed()) for key in ("bytes", "flops")]
    while True:
        case = _any_case(rng)
        w = work(case)
        if w["bytes"] <= 0.8 * largest[0] and w["flops"] <= 0.8 * largest[1]:
            return case


def _any_case(rng):
    kind = rng.choice(["nvfp4_linear", "mxfp8_linear", "nvfp4_mlp", "nvfp4_moe", "nvfp4_expert_linear", "expert_mm", "quantize"])
    half = rng.choice(["bf16", "bf16", "f16"])
    if kind in ("nvfp4_linear", "mxfp8_linear"):
        steps = [32, 64, 128, 256, 512]
        return dict(kind=kind, m=_log(rng, 1, 8192), n=_width(rng, 1024, 16384, steps), k=_width(rng, 1024, 16384, steps), dtype=half)
    if kind == "nvfp4_mlp":
        steps = [64, 128, 256, 512]
        return dict(kind=kind, m=_log(rng, 1, 4096), hidden=_width(rng, 1024, 8192, steps), inter=_width(rng, 2048, 16384, steps),
                    dtype=half)
    if kind == "quantize":
        fmt = rng.choice(["nvfp4", "mxfp8"])
        return dict(kind=kind, rows=_log(rng, 16, 65536), cols=_width(rng, 1024, 8192, [32, 64, 128, 512, 1024]), fmt=fmt,
                    dtype=rng.choice(["bf16", "bf16", "f16", "f32"]))
    experts = rng.choice([8, 16, 32, 64, 128, 256])
    m = _log(rng, max(16, experts // 2), 65536)
    zipf = rng.choice([False, True])
    if kind == "nvfp4_moe":
        return dict(kind=kind, m=m, hidden=_width(rng, 1024, 7168, [128, 256, 512]), inter=_width(rng, 512, 4096, [128, 256, 512]),
                    experts=experts, zipf=zipf, dtype="bf16")
    if kind == "nvfp4_expert_linear":
        return dict(kind=kind, m=m, n=_width(rng, 1024, 8192, [128, 256, 512]), k=_width(rng, 1024, 7168, [64, 128, 512]),
                    experts=experts, zipf=zipf, dtype="bf16")
    experts = min(experts, 64)
    return dict(kind=kind, m=_log(rng, 16, 16384), n=_width(rng, 1024, 14336, [8, 64, 128, 256, 512]),
                k=_width(rng, 1024, 7168, [8, 64, 128, 512]), experts=experts, zipf=zipf, dtype=half)


def _loads(case):
    """Rows of every expert, in no particular order: `m` draws from an even or a Zipf(1.1) distribution."""
    rng = random.Random(case["m"] * 1009 + case["experts"])
    weights = [1.0 / (e + 1) ** 1.1 if case["zipf"] else 1.0 for e in range(case["experts"])]
    sizes = [0] * case["experts"]
    for e in rng.choices(range(case["experts"]), weights, k=case["m"]):
        sizes[e] += 1
    return sizes


def _generator(seed):
    gen = torch.Generator(device=DEV)
    gen.manual_seed(seed)
    return gen


def _normal(gen, shape, dtype, std=1.0):
    return torch.randn(shape, generator=gen, device=DEV, dtype=dtype).mul_(std)


def _scalar(value):
    return torch.tensor(value, dtype=torch.float32, device=DEV)


W_STD = 0.02  # standard deviation of the synthetic weights
A_SCALE = 2688.0 / 6.0  # calibrated global scale of N(0, 1) activations: 448 * 6 over a largest value of 6


def _nvfp4_weights(gen, n, k, experts=0):
    """-> (payload, block scales, what the product is multiplied with to undo the global scale)."""
    gs = _scalar(2688.0 / (6.0 * W_STD))
    if not experts:
        return (*ops.nv_block_quantize(_normal(gen, (n, k), torch.bfloat16, W_STD), gs, True), 1.0 / float(gs))
    q = torch.empty((experts, n, k // 2), dtype=torch.uint8, device=DEV)
    s = torch.empty((experts, n, -(-(k // 16) // 4) * 4), dtype=torch.uint8, device=DEV)
    for e in range(0, experts, 16):
        part = _normal(gen, (min(16, experts - e) * n, k), torch.bfloat16, W_STD)
        pq, ps = ops.nv_block_quantize(part, gs, True)
        q[e:e + 16].view(-1, k // 2).copy_(pq.view(torch.uint8))
        s[e:e + 16].view(-1, s.size(2)).copy_(ps.view(torch.uint8))
    return q.view(torch.float4_e2m1fn_x2), s.view(torch.float8_e4m3fn), torch.full((experts,), 1.0 / float(gs), device=DEV)


def _routing(case, seed):
    """-> (first row of every expert, rows of every expert), int32 on the device."""
    sizes = _loads(case)
    random.Random(seed).shuffle(sizes)
    sizes = torch.tensor(sizes, dtype=torch.int32)
    starts = torch.cumsum(sizes, 0, dtype=torch.int32) - sizes
    return starts.to(DEV), sizes.to(DEV)


def prepare(case, seed):
    kind, gen, dtype = case["kind"], _generator(seed), DTYPES[case["dtype"]]
    st = dict(kind=kind, dtype=dtype)
    if kind == "quantize":
        st.update(x=_normal(gen, (case["rows"], case["cols"]), dtype), fmt=case["fmt"])
    elif kind == "nvfp4_linear":
        wq, ws, inv = _nvfp4_weights(gen, case["n"], case["k"])
        st.update(x=_normal(gen, (case["m"], case["k"]), dtype), gs=_scalar(A_SCALE), wq=wq, ws=ws, alpha=_scalar(inv / A_SCALE))
    elif kind == "mxfp8_linear":
        wq, ws = ops.nv_block_quantize(_normal(gen, (case["n"], case["k"]), torch.bfloat16, W_STD), None, True, 32, torch.float8_e4m3fn)
        st.update(x=_normal(gen, (case["m"], case["k"]), dtype), wq=wq, ws=ws, alpha=_scalar(1.0))
    elif kind == "nvfp4_mlp":
        up_q, up_s, inv = _nvfp4_weights(gen, case["inter"], case["hidden"])
        down_q, down_s, _ = _nvfp4_weights(gen, case["hidden"], case["inter"])
        mid_scale = 2688.0 / (6.0 * W_STD * math.sqrt(case["hidden"]))
        st.update(x=_normal(gen, (case["m"], case["hidden"]), dtype), gs=_scalar(A_SCALE), up_q=up_q, up_s=up_s, down_q=down_q,
                  down_s=down_s, up_alpha=_scalar(inv / A_SCALE), mid_gs=_scalar(mid_scale), down_alpha=_scalar(inv / mid_scale))
    elif kind == "nvfp4_moe":
        g, hidden, inter = case["experts"], case["hidden"], case["inter"]
        starts, _ = _routing(case, seed)
        strides = [torch.full((g,), width, dtype=torch.int64, device=DEV) for width in (hidden, inter)]
        st.update(x=_normal(gen, (case["m"], hidden), dtype), starts=starts, hidden=hidden, inter=inter, strides=strides,
                  gate=_nvfp4_weights(gen, inter, hidden, g), up=_nvfp4_weights(gen, inter, hidden, g),
                  down=_nvfp4_weights(gen, hidden, inter, g))
    elif kind == "nvfp4_expert_linear":
        starts, _ = _routing(case, seed)
        wq, ws, alphas = _nvfp4_weights(gen, case["n"], case["k"], case["experts"])
        st.update(x=_normal(gen, (case["m"], case["k"]), dtype), starts=starts, n=case["n"], wq=wq.transpose(1, 2), ws=ws, alphas=alphas)
    else:
        g, n, k = case["experts"], case["n"], case["k"]
        starts, sizes = _routing(case, seed)
        problem_sizes = torch.stack([sizes, torch.full_like(sizes, n), torch.full_like(sizes, k)], dim=1).contiguous()
        st.update(x=_normal(gen, (case["m"], k), dtype), w=_normal(gen, (g, n, k), dtype, W_STD), starts=starts,
                  problem_sizes=problem_sizes, ab=torch.full((g,), k, dtype=torch.int64, device=DEV),
                  c=torch.full((g,), n, dtype=torch.int64, device=DEV))
    return st


def run(st):
    kind, x, dtype = st["kind"], st["x"], st["dtype"]
    if kind == "quantize":
        if st["fmt"] == "nvfp4":
            gs = ops.compute_nvfp4_global_scale(x)
            q, s = ops.nv_block_quantize(x, gs, True)
            return q.view(torch.uint8), s.view(torch.uint8), gs
        q, s = ops.nv_block_quantize(x, None, True, 32, torch.float8_e4m3fn)
        return q.view(torch.uint8), s.view(torch.uint8)
    if kind == "nvfp4_linear":
        q, s = ops.nv_block_quantize(x, st["gs"], True)
        return nvf_cutlass.nvfp4_scaled_mm(q, st["wq"], s, st["ws"], st["alpha"], dtype)
    if kind == "mxfp8_linear":
        q, s = ops.nv_block_quantize(x, None, True, 32, torch.float8_e4m3fn)
        return nvf_cutlass.mxfp8_scaled_mm(q, st["wq"], s, st["ws"], st["alpha"], dtype)
    if kind == "nvfp4_mlp":
        q, s = ops.nv_block_quantize(x, st["gs"], True)
        q, s = nvf_cutlass.nvfp4_scaled_mm_blockscale(q, st["up_q"], s, st["up_s"], st["up_alpha"], st["mid_gs"])
        return nvf_cutlass.nvfp4_scaled_mm(q, st["down_q"], s, st["down_s"], st["down_alpha"], dtype)
    if kind == "nvfp4_moe":
        starts, (hs, is_) = st["starts"], st["strides"]
        offsets, sizes = compute_auxiliary_tensors(x, starts, st["inter"])
        q, s = ops.nv_grouped_block_quantize(x, starts, offsets)
        gate, up = (nvf_cutlass.nvfp4_scaled_grouped_mm(q, wq, s, ws, alphas, hs, is_, sizes, starts, offsets, dtype)
                    for wq, ws, alphas in (st["gate"], st["up"]))
        offsets, sizes = compute_auxiliary_tensors(up, starts, st["hidden"])
        q, s = ops.silu_mul_nv_grouped_block_quantize(gate, up, starts, offsets)
        wq, ws, alphas = st["down"]
        return nvf_cutlass.nvfp4_scaled_grouped_mm(q, wq, s, ws, alphas, is_, hs, sizes, starts, offsets, dtype)
    if kind == "nvfp4_expert_linear":
        offsets, sizes = compute_auxiliary_tensors(x, st["starts"], st["n"])
        return f16a_nvfp4weight_scaled_grouped_mm(x, st["wq"], st["ws"], st["alphas"], st["starts"], offsets, sizes)
    return nvf_cutlass.grouped_mm(x, st["w"], st["ab"], st["c"], st["problem_sizes"], st["starts"])


def work(case):
    """The activations as they come in, the weights (of the experts that have rows), the result; 2 m n k."""
    kind, size = case["kind"], BYTES[case["dtype"]]
    if kind == "quantize":
        n = case["rows"] * case["cols"]
        # (an NVFP4 global scale has to be known before the first block is quantized, but what has been read for it may
        # still be on the chip: the input counts once)
        return {"bytes": n * (size + (FP4 if case["fmt"] == "nvfp4" else FP8)), "flops": 0}
    m = case["m"]
    active = sum(s > 0 for s in _loads(case)) if "experts" in case else 1
    if kind in ("nvfp4_mlp", "nvfp4_moe"):
        weights = 3 if kind == "nvfp4_moe" else 2
        hidden, inter = case["hidden"], case["inter"]
        return {"bytes": 2 * m * hidden * size + weights * active * hidden * inter * FP4, "flops": 2 * weights * m * hidden * inter}
    n, k = case["n"], case["k"]
    weight = {"nvfp4_linear": FP4, "nvfp4_expert_linear": FP4, "mxfp8_linear": FP8, "expert_mm": 2}[kind]
    return {"bytes": m * (k + n) * size + active * n * k * weight, "flops": 2 * m * n * k}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    # Measured against the same path with its sums in another order (64- or 128-wide pieces of K shuffled in both operands).
    # 16-bit experts: rel 6e-5, max 7.8e-3 - about 4 results in 10000 lie close enough to a rounding boundary to end one
    # 16-bit step away.  MXFP8: rel 4e-6, max 5e-3.  NVFP4: no difference, because block scales this close to each other
    # make every fp32 sum exact; an implementation whose sums are rounded is off by what the 16-bit experts show.
    if kind in ("nvfp4_mlp", "nvfp4_moe"):
        # ... and by a few e2m1 codes where the product between the layers is quantized again
        return {"rel": 1e-3, "max": 5e-2}
    return {"rel": 2.4e-4, "max": 1.6e-2}
