"""Performance cases of the chunked FP16 GEMM: what its users run, through
f16acc_amd.mm and through nn.functional.linear with the patch enabled.

Every case is one call.  "linear" is the patched F.linear of an inference-mode
FP16 layer: x [M, K] ~ N(0, 1), weight [N, K] ~ N(0, 0.02) as stored by
nn.Linear, optional bias ~ N(0, 0.02).  "mm" is f16acc_amd.mm(a, b) on a [M, K]
and b [K, N], both ~ N(0, 1), with the layouts, output type and accumulation
mode its arguments offer.
"""

import torch
import torch.nn.functional as F

import f16acc_amd

CHUNK = 32  # the rounding interval along K


def listed():
    return [
        # The shortest prompt the patch routes (128 rows), on the narrowest
        # projection of Qwen2.5-1.5B (k/v, biased): a call is latency.
        dict(name="linear_kv_128", op="linear", M=128, N=256, K=1536, bias=True),
        # The projections of a Qwen2.5-1.5B prefill of 2048 tokens: k/v and
        # q/o (few output tiles), gate/up (wide), down (long K).
        dict(name="linear_kv_2048", op="linear", M=2048, N=256, K=1536, bias=True),
        dict(name="linear_qo_2048", op="linear", M=2048, N=1536, K=1536, bias=True),
        dict(name="linear_gateup_2048", op="linear", M=2048, N=8960, K=1536, bias=False),
        dict(name="linear_down_2048", op="linear", M=2048, N=1536, K=8960, bias=False),
        # Its lm_head over the whole prompt: the widest output.
        dict(name="linear_lm_head_2048", op="linear", M=2048, N=151936, K=1536, bias=False),
        # Odd extents in every dimension: rows that no 16-byte load fits.
        dict(name="linear_odd", op="linear", M=2049, N=1537, K=8961, bias=True),
        # A small square product with an FP32 result, both operands row-major.
        dict(name="mm_1024_f32", op="mm", M=1024, N=1024, K=1024, a="row", b="row", out="f32", chunked=True,
             overflow=0.0),
        # The headline GEMM: row-major operands, FP16 result.
        dict(name="mm_4096", op="mm", M=4096, N=4096, K=4096, a="row", b="row", out="f16", chunked=True, overflow=0.0),
        # The largest: against a stored weight, FP32 result.
        dict(name="mm_8192_wt_f32", op="mm", M=8192, N=8192, K=8192, a="row", b="wt", out="f32", chunked=True,
             overflow=0.0),
        # Overflow stress: about 5 % of the 128 x 128 blocks of the output
        # have chunks past 65504 and are redone with FP32 accumulation.
        dict(name="mm_4096_overflow", op="mm", M=4096, N=4096, K=4096, a="row", b="row", out="f32", chunked=True,
             overflow=0.22),
        # The plain FP32-accumulating mode (chunked=False) against a weight.
        dict(name="mm_4096_fp32acc", op="mm", M=4096, N=4096, K=4096, a="row", b="wt", out="f16", chunked=False,
             overflow=0.0),
    ]


def _extent(rng, lo, hi):
    """An extent spread over its logarithm: mostly whole tiles' multiples, else
    a multiple of 8, else any number, odd ones among them."""
    v = int(round(lo * (hi / lo) ** rng.random()))
    r = rng.random()
    step = 128 if r < 0.45 else 8 if r < 0.75 else 1
    return max(lo, min(hi, v // step * step))


def draw(rng):
    """Layers of 128 to 4096 tokens and products of 128 to 8192 a side, any
    extents, layouts, types and modes."""
    if rng.random() < 0.5:
        return dict(op="linear", M=_extent(rng, 128, 4096), N=_extent(rng, 128, 16384), K=_extent(rng, 256, 12288),
                    bias=rng.random() < 0.4)
    while True:
        M, N, K = _extent(rng, 128, 8192), _extent(rng, 128, 8192), _extent(rng, 128, 8192)
        a = "row" if rng.random() < 0.85 else "t"  # "t": a transposed view of [K, M]
        b = "row" if rng.random() < 0.5 else "wt"  # "wt": a transposed view of [N, K]
        out = "f16" if rng.random() < 0.6 else "f32"
        chunked = rng.random() < 0.85
        overflow = 0.22 if chunked and rng.random() < 0.12 else 0.0
        out = "f32" if overflow else out  # the redone sums pass the FP16 range
        if M * N * K <= 8192 ** 3 // 2:
            return dict(op="mm", M=M, N=N, K=K, a=a, b=b, out=out, chunked=chunked, overflow=overflow)


def _overflow_blocks(t, dim, share, g):
    """Sets `share` of the 128-wide blocks of t along dim to U(200, 255): where
    such rows of a meet such columns of b, chunk sums pass 65504."""
    blocks = t.shape[dim] // 128
    for i in torch.randperm(blocks, generator=g, device=t.device)[:round(share * blocks)].tolist():
        part = t.narrow(dim, 128 * i, 128)
        part.copy_(200.0 + 55.0 * torch.rand(part.shape, generator=g, device=t.device))


def prepare(case, seed):
    dev = torch.device("cuda")
    g = torch.Generator(device=dev).manual_seed(seed)
    M, N, K = case["M"], case["N"], case["K"]

    def normal(*shape, std=1.0):
        return torch.randn(*shape, generator=g, device=dev).mul_(std).half()

    if case["op"] == "linear":
        f16acc_amd.enable()
        return {"op": "linear", "x": normal(M, K), "w": normal(N, K, std=0.02),
                "bias": normal(N, std=0.02) if case["bias"] else None}
    a = normal(M, K)
    b = normal(K, N)
    if case["overflow"]:
        _overflow_blocks(a, 0, case["overflow"], g)
        _overflow_blocks(b, 1, case["overflow"], g)
    if case["a"] == "t":
        a = a.t().contiguous().t()
    if case["b"] == "wt":
        b = b.t().contiguous().t()
    return {"op": "mm", "a": a, "b": b, "out": torch.float16 if case["out"] == "f16" else torch.float32,
            "chunked": case["chunked"]}


def run(state):
    if state["op"] == "linear":
        with torch.inference_mode():
            return F.linear(state["x"], state["w"], state["bias"])
    return f16acc_amd.mm(state["a"], state["b"], state["out"], state["chunked"])


def work(case):
    M, N, K = case["M"], case["N"], case["K"]
    out = 4 if case.get("out") == "f32" else 2
    bias = 2 * N if case.get("bias") else 0
    return {"bytes": 2 * M * K + 2 * K * N + out * M * N + bias, "flops": 2 * M * N * K}


def tolerance(case):
    # FP16 results: against exact() the path is off by 2.1e-4 (2.9e-4 with a
    # bias, rounded twice) in the 2-norm, and by an ulp of binary16 (1e-3) at
    # most where two sums fall on both sides of a tie.
    if case["op"] == "linear" or case["out"] == "f16":
        return {"rel": 1.2e-3, "max": 4e-3}
    # FP32 sums without chunks.
    if not case["chunked"]:
        return {"rel": 1e-5, "max": 1e-4}
    # FP32 results: 4.3e-6 against exact().  A chunk's partial that another
    # order of its 32 products puts on the other side of a binary16 rounding
    # moves the sum by an ulp of that partial (at most 2^-5 on N(0, 1) data,
    # where short sums have a root mean square of 11).
    return {"rel": 2e-5, "max": 5e-3}


def exact(case, seed):
    """The operation in 64 bits: every 32-long K chunk's dot product rounded
    to binary16 and the chunks added (chunked=False: the plain product).  Where
    chunks overflow, the redone tiles hold the plain product."""
    s = prepare(case, seed)
    linear = s["op"] == "linear"
    a, b = (s["x"], s["w"].t()) if linear else (s["a"], s["b"])
    K = case["K"]
    chunked = linear or (case["chunked"] and not case["overflow"])
    a64, b64 = a.double().contiguous(), b.double().contiguous()
    if not chunked:
        return torch.mm(a64, b64)
    total = torch.zeros(a.shape[0], b.shape[1], dtype=torch.float64, device=a.device)
    for k in range(0, K, CHUNK):
        part = torch.mm(a64[:, k:k + CHUNK].contiguous(), b64[k:k + CHUNK].contiguous())
        total += part.half()
    if linear and s["bias"] is not None:
        total += s["bias"].double()
    return total
