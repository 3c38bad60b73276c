"""The calls that a serving engine makes of this library, as timing cases.

One case is one layer call on one GPU: a dense projection in one of the three quantized formats, or one MoE block, with
the activations, packed weights and scales that an engine holds in HBM at that point.  The activation quantizers belong to
the call where the layer runs them (block fp8, W4A8), and so do routing and alignment in a MoE block.  Weights are packed
once, as the loader does.
"""
import torch

from ksanallm_amd import lib as L
from ksanallm_amd import ops

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}


def listed():
    return [
        # one sequence decoding: attention projection of a 4096-wide GPTQ model, the smallest call there is
        dict(name="gptq_f16_4096x4096_m1", op="w4a16", quant="gptq", dtype="f16", group=128, m=1, n=4096, k=4096),
        # a few sequences decoding: gate / up projection of an AWQ model
        dict(name="awq_bf16_14336x4096_m8", op="w4a16", quant="awq", dtype="bf16", group=128, m=8, n=14336, k=4096),
        # a full decode batch through the down projection: few columns, long k
        dict(name="awq_bf16_4096x14336_m32", op="w4a16", quant="awq", dtype="bf16", group=128, m=32, n=4096, k=14336),
        # a large decode batch together with a short prompt: a ragged number of rows
        dict(name="awq_bf16_14336x4096_m150", op="w4a16", quant="awq", dtype="bf16", group=128, m=150, n=14336, k=4096),
        # prefill of several prompts: the largest dense call
        dict(name="gptq_f16_25600x5120_m4096", op="w4a16", quant="gptq", dtype="f16", group=128, m=4096, n=25600, k=5120),
        # block-fp8 dense MLP: decode batch, mixed batch, prefill
        dict(name="fp8_bf16_18432x7168_m16", op="fp8", dtype="bf16", m=16, n=18432, k=7168),
        dict(name="fp8_bf16_18432x7168_m200", op="fp8", dtype="bf16", m=200, n=18432, k=7168),
        dict(name="fp8_bf16_7168x18432_m4096", op="fp8", dtype="bf16", m=4096, n=7168, k=18432),
        # W4A8 at a large decode batch
        dict(name="w4a8_bf16_25600x5120_m64", op="w4a8", dtype="bf16", m=64, n=25600, k=5120),
        # int4 experts: one sequence decoding, and a chunk of a prompt with a few rows per expert
        dict(name="moe_int4_bf16_t1", op="moe_int4", dtype="bf16", t=1, experts=256, top_k=8, hidden=7168, inter=2048),
        dict(name="moe_int4_bf16_t512", op="moe_int4", dtype="bf16", t=512, experts=256, top_k=8, hidden=7168, inter=2048),
        # block-fp8 experts: prefill, a ragged number of tokens
        dict(name="moe_fp8_bf16_t4000", op="moe_fp8", dtype="bf16", t=4000, experts=256, top_k=8, hidden=7168, inter=2048),
    ]


def _log(rng, lo, hi, step=1):
    """A multiple of step in [lo, hi], spread over the logarithm."""
    v = lo * (hi / lo) ** rng.random()
    return min(hi // step * step, max(-(-lo // step) * step, round(v / step) * step))


def draw(rng):
    op = rng.choice(["w4a16", "w4a16", "w4a16", "fp8", "fp8", "w4a8", "moe_int4", "moe_int4", "moe_fp8"])
    dtype = rng.choice(["f16", "bf16"])
    biggest = max((work(c)["flops"] for c in listed() if not c["op"].startswith("moe")))
    while True:
        if op.startswith("moe"):
            case = dict(op=op, dtype=dtype, t=_log(rng, 1, 4000), experts=rng.choice([8, 16, 32, 64, 128, 256]),
                        top_k=rng.choice([2, 4, 6, 8]), hidden=_log(rng, 1024, 7168, 128), inter=_log(rng, 512, 2048, 128))
            return case
        case = dict(op=op, dtype=dtype, m=_log(rng, 1, 8192), n=_log(rng, 1024, 28672, 32), k=_log(rng, 1024, 28672, 128))
        if op == "w4a16":
            case.update(quant=rng.choice(["gptq", "awq"]), group=rng.choice([128, 128, 128, 64]))
        # the weight of one projection of one rank, and no more work than the largest listed dense call
        if case["n"] * case["k"] <= 57344 * 8192 // 2 and work(case)["flops"] <= biggest:
            return case


def _touched(case):
    """Experts that a batch reaches, in expectation: every token takes top_k different ones, uniformly."""
    return case["experts"] * (1.0 - (1.0 - case["top_k"] / case["experts"]) ** case["t"])


def work(case):
    op = case["op"]
    if op.startswith("moe"):
        t, h, i = case["t"], case["hidden"], case["inter"]
        per_expert = 3 * h * i // 2 + 3 * h * i // 128 * 2 if op == "moe_int4" else 3 * h * i + 3 * h * i // (128 * 128) * 4
        return {"bytes": int(_touched(case) * per_expert + 2 * t * h * 2 + t * case["experts"] * 4),
                "flops": 6 * t * case["top_k"] * h * i}
    m, n, k = case["m"], case["n"], case["k"]
    weight = n * k if op == "fp8" else n * k // 2
    if op == "w4a16":
        groups = k // case["group"]
        weight += groups * n * 2 + (groups * n // 2 if case["quant"] == "awq" else 0)
    elif op == "w4a8":
        weight += k // 128 * n * 2
    else:
        weight += (n + 127) // 128 * (k // 128) * 4
    return {"bytes": weight + 2 * m * k + 2 * m * n, "flops": 2 * m * n * k}


def tolerance(case):
    """About four times the distance of the path's result from the same path in 64 bits.

    A dense call is off by the rounding of its output alone (1.7e-3 in bf16, 2.1e-4 in fp16) or of its weights and its
    output (2.2e-3, 2.8e-4).  A MoE block rounds its weights, the activation's output and every expert's share (5.6e-3,
    6.1e-4).  Block-fp8 experts quantize the activation's output again, where one step of the 16-bit type moves a value
    to the next e4m3 code (1.6e-2 in bf16).
    """
    f16 = case["dtype"] == "f16"
    if case["op"] == "moe_fp8":
        return {"rel": 1.5e-2 if f16 else 3e-2}
    if case["op"] == "moe_int4":
        return {"rel": 2.4e-3 if f16 else 2e-2}
    return {"rel": 1.1e-3 if f16 else 7e-3}


# ------------------------------------------------------------------------------------------------- inputs
def _activations(g, rows, k, dtype, std, outliers):
    x = torch.randn((rows, k), generator=g, device="cuda") * std
    if outliers:   # one value in a hundred twenty times as large, as hidden states have them
        x = torch.where(torch.rand((rows, k), generator=g, device="cuda") < 0.01, x * 20, x)
    return x.to(DTYPES[dtype])


def _uniform(g, shape, lo, hi, dtype):
    return (torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo).to(dtype)


def _fp8_weight(g, n, k):
    """e4m3 codes and fp32 block scales of a weight ~ N(0, 0.02^2), one scale = amax / 448 per 128 x 128 block."""
    rows = -(-n // 128) * 128
    w = torch.randn((rows // 128, 128, k // 128, 128), generator=g, device="cuda") * 0.02
    s = w.abs().amax(dim=(1, 3)) / 448.0
    q = (w / s[:, None, :, None]).to(torch.float8_e4m3fn).view(torch.uint8).view(rows, k)[:n]
    return q.contiguous(), s.contiguous()


def _prepare_w4a16(case, g):
    m, n, k, group = case["m"], case["n"], case["k"], case["group"]
    dt = DTYPES[case["dtype"]]
    awq = case["quant"] == "awq"
    shape, layout = ((k, n // 8), L.SRC_AWQ) if awq else ((k // 8, n), L.SRC_GPTQ)
    codes = torch.randint(-2**31, 2**31 - 1, shape, generator=g, device="cuda", dtype=torch.int32)
    scales = _uniform(g, (k // group, n), 0.003, 0.015, dt)
    zeros = None
    if awq:
        zp = torch.randint(6, 10, (k // group, n), generator=g, device="cuda", dtype=torch.uint8)
        zeros = ops.repack_zeros(zp, L.ZERO_U8_GN, k, n, group)
    return {"x": _activations(g, m, k, case["dtype"], 1.0 if m <= 512 else 0.5, False),
            "w": ops.repack_weight(codes, layout, 1, k, n),
            "s": ops.repack_scales(scales, L.SCALE_GN, 1, k, n, group), "z": zeros}


def _prepare_fp8(case, g):
    q, s = _fp8_weight(g, case["n"], case["k"])
    return {"x": _activations(g, case["m"], case["k"], case["dtype"], 1.0, True), "w": ops.fp8_repack_weight(q), "s": s}


def _prepare_w4a8(case, g):
    m, n, k = case["m"], case["n"], case["k"]
    codes = torch.randint(0, 256, (k, n // 2), generator=g, device="cuda", dtype=torch.uint8)
    return {"x": _activations(g, m, k, case["dtype"], 1.0, True), "w": ops.w4a8_repack_weight(codes),
            "s": _uniform(g, (k // 128, n), 0.003, 0.015, torch.float16),
            "in_scale": torch.tensor([0.05], dtype=torch.float32, device="cuda"), "alpha": 0.035}


def _prepare_moe(case, g):
    E, h, i = case["experts"], case["hidden"], case["inter"]
    dt = DTYPES[case["dtype"]]
    state = {"x": _activations(g, case["t"], h, case["dtype"], 1.0, False),
             "logits": torch.randn((case["t"], E), generator=g, device="cuda")}
    if case["op"] == "moe_int4":
        for name, n, k in (("13", 2 * i, h), ("2", h, i)):
            codes = torch.randint(0, 256, (E, n, k // 2), generator=g, device="cuda", dtype=torch.uint8)
            state["w" + name] = ops.repack_weight(codes, L.SRC_MOE_NK, E, k, n)
            state["s" + name] = ops.repack_scales(_uniform(g, (E, n, k // 128), 0.002, 0.01, dt), L.SCALE_NG, E, k, n, 128)
        return state
    for name, n, k in (("13", 2 * i, h), ("2", h, i)):
        q = torch.empty((E, n, k), dtype=torch.uint8, device="cuda")
        s = torch.empty((E, n // 128, k // 128), dtype=torch.float32, device="cuda")
        for e in range(E):
            q[e], s[e] = _fp8_weight(g, n, k)
        state["w" + name], state["s" + name] = ops.fp8_repack_weight(q), s
    return state


def prepare(case, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    make = {"w4a16": _prepare_w4a16, "fp8": _prepare_fp8, "w4a8": _prepare_w4a8}.get(case["op"], _prepare_moe)
    state = make(case, g)
    state["case"] = case
    return state


# ------------------------------------------------------------------------------------------------- one pass
def run(state):
    case, x = state["case"], state["x"]
    op = case["op"]
    if op == "w4a16":
        return ops.w4a16_gemm(x, state["w"], state["s"], state["z"], case["n"], case["k"], case["group"])
    if op == "fp8":
        a_q, a_s = ops.per_token_group_quant_fp8(x, case["k"])
        return ops.fp8_blockwise_gemm(a_q, a_s, state["w"], state["s"], out_dtype=x.dtype)
    if op == "w4a8":
        a_q, xsum = ops.w4a8_static_quant(x, state["in_scale"])
        return ops.w4a8_gemm(a_q, xsum, state["w"], state["s"], state["alpha"], case["n"], out_dtype=x.dtype)
    topk_w, topk_ids = ops.moe_topk_softmax(state["logits"], case["top_k"], norm_topk_prob=True)
    if op == "moe_int4":
        return ops.fused_moe_w4a16(x, state["w13"], state["s13"], state["w2"], state["s2"], topk_ids, topk_w,
                                   case["experts"], case["hidden"], case["inter"], 128)
    return ops.fused_moe_fp8_blockwise(x, state["w13"], state["s13"], state["w2"], state["s2"], topk_ids, topk_w)
