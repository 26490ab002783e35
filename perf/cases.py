"""The work a user of this package has it do, as measurable cases.

Four operations, each through its public entry point:

  swiglu     fused_swiglu on packed weights: Y = SiLU(X Wg) * (X Wu)
  matmul     matmul on packed weights: C = A B, or C += A B with "accumulate"
  mlp        mlp on packed weights: Y = SwiGLU(X), Z = Y Wd
  kernel_fn  the cache's KernelFn(x, wg, wu, init, result): the fused SwiGLU on
             raw row-major weights, read at every call, synchronous

over the sizes of this repository's benchmark workloads: rows M from one
decoded token to a prefill of 4097, model widths K up to 5120, hidden widths N
from 1376 (one of eight shards of 11008) to 14336, and the down projection's
K = 13824.  bf16 operands, fp32 accumulation, results in bf16, fp16 or fp32.
"""
import math

import torch

import dslcompiler_amd as llk

DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def listed():
    return [
        # The smallest call: the validation kernel, a TP-8 slice of a 7B-class
        # MLP's gate and up projections at batch 64, fp32 result.
        dict(name="swiglu m64 tp8 f32", op="swiglu", M=64, K=512, N=1376, out="f32"),
        # One decoded token through an 8B-class MLP's gate and up projections.
        dict(name="swiglu decode m1", op="swiglu", M=1, K=4096, N=14336, out="bf16"),
        # A decode batch of 16 through the same layer.
        dict(name="swiglu decode m16", op="swiglu", M=16, K=4096, N=14336, out="bf16"),
        # The same layer through the JIT-shaped function, as a host program
        # that keeps its weights row-major calls it, batch 8.
        dict(name="kernel_fn decode m8", op="kernel_fn", M=8, K=4096, N=14336, out="bf16"),
        # Sizes that are no multiple of any tile, K = 1000 among them.
        dict(name="swiglu ragged m300", op="swiglu", M=300, K=1000, N=1100, out="bf16"),
        # Prefill of 2048 tokens, 7B-class gate and up projections.
        dict(name="swiglu prefill m2048", op="swiglu", M=2048, K=4096, N=11008, out="bf16"),
        # The plain matrix product.
        dict(name="matmul 4096", op="matmul", M=4096, K=4096, N=4096, out="f32"),
        # The accumulating product (acc += lhs rhs): a down projection added
        # to an fp32 residual stream.
        dict(name="matmul += m1000", op="matmul", M=1000, K=13824, N=5120, out="f32",
             accumulate=True),
        # The whole 13B-class MLP block at ragged token counts: a decode batch,
        # a chunk of prefill, a prompt, and the largest call.
        dict(name="mlp m17", op="mlp", M=17, K=5120, N=13824, out="bf16"),
        dict(name="mlp m255", op="mlp", M=255, K=5120, N=13824, out="bf16"),
        dict(name="mlp m1000", op="mlp", M=1000, K=5120, N=13824, out="bf16"),
        dict(name="mlp m4097", op="mlp", M=4097, K=5120, N=13824, out="bf16"),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def _width(rng, lo, hi, step):
    """A model or hidden width: mostly a multiple of `step`, else any number."""
    n = _log_int(rng, lo, hi)
    return max(step, n // step * step) if rng.random() < 0.75 else n


def draw(rng):
    op = rng.choices(["swiglu", "matmul", "mlp", "kernel_fn"], [35, 25, 25, 15])[0]
    M = _log_int(rng, 1, 4097)
    if op == "matmul":
        # an up projection (K up to 5120) or a down projection (K up to 13824)
        up = rng.random() < 0.5
        K = _width(rng, 512, 5120 if up else 13824, 64)
        N = _width(rng, 1376, 14336, 16) if up else _width(rng, 512, 5120, 64)
        return dict(op=op, M=M, K=K, N=N, out=rng.choice(["f32", "bf16", "f16"]),
                    accumulate=rng.random() < 0.4)
    K = _width(rng, 512, 5120, 64)
    N = _width(rng, 1376, 13824 if op == "mlp" else 14336, 16)
    out = "bf16" if op == "mlp" or rng.random() < 0.75 else "f32"
    return dict(op=op, M=M, K=K, N=N, out=out)


def _inputs(case, seed):
    """X ~ N(0, 1), with 1% of its entries scaled by 20 where the activations
    of a whole MLP are meant; weights ~ N(0, 1/sqrt(fan in)); all bf16."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    M, K, N, op = case["M"], case["K"], case["N"], case["op"]

    def normal(rows, cols, sigma=1.0):
        return torch.randn(rows, cols, generator=g, device="cuda").mul_(sigma).bfloat16()

    x = normal(M, K)
    if op == "mlp":
        big = torch.rand(M, K, generator=g, device="cuda") < 0.01
        x = torch.where(big, x * 20, x)
    w = [normal(K, N, K ** -0.5)]
    if op != "matmul":
        w.append(normal(K, N, K ** -0.5))
    if op == "mlp":
        w.append(normal(N, K, N ** -0.5))
    c = normal(M, N).to(DTYPES[case["out"]]) if case.get("accumulate") else None
    return x, w, c


def prepare(case, seed):
    x, w, c = _inputs(case, seed)
    state = {"op": case["op"], "x": x, "dtype": DTYPES[case["out"]], "c": c}
    if case["op"] == "kernel_fn":
        state["w"] = w
        state["cache"] = llk.JitCache()
        state["fn"] = state["cache"].lookup_or_compile(llk.KernelKey(
            operation=0, isa=7, M_bucket=llk.classify_m(case["M"]), N=case["N"], K=case["K"],
            output_type=2 if case["out"] == "f32" else 0))
        state["y"] = torch.empty(case["M"], case["N"], dtype=state["dtype"], device="cuda")
    else:
        state["w"] = [llk.PackedWeights.from_device(m) for m in w]
    return state


def run(state):
    op, x, w = state["op"], state["x"], state["w"]
    if op == "swiglu":
        return llk.fused_swiglu(x, w[0], w[1], out_dtype=state["dtype"])
    if op == "mlp":
        return llk.mlp(x, w[0], w[1], w[2])
    if op == "kernel_fn":
        state["fn"](x, w[0], w[1], state["y"], state["y"])
        return state["y"]
    if state["c"] is not None:
        return llk.matmul(x, w[0], out=state["c"], accumulate=True)
    return llk.matmul(x, w[0], out_dtype=state["dtype"])


def work(case):
    """Operands read once, results written once; the multiply-adds."""
    M, K, N = case["M"], case["K"], case["N"]
    mats = {"matmul": 1, "mlp": 3}.get(case["op"], 2)
    out = 4 if case["out"] == "f32" else 2
    nbytes = 2 * mats * K * N + 2 * M * K + out * M * N
    if case["op"] == "mlp":
        nbytes += out * M * K
    if case.get("accumulate"):
        nbytes += out * M * N
    return {"bytes": nbytes, "flops": 2 * mats * M * K * N}


def tolerance(case):
    """Two orders of the fp32 sums (1, 3 and the default number of k splits,
    over these ranges) were seen to differ by 5.4e-7 in fp32 results, by
    1.3e-5 (fp16) and 9e-5 (bf16) in the 16-bit ones, whose values differ only
    where they round the other way (by one unit in the last place: the max),
    and by 5e-4 in Z, which carries the flips of Y's rounding through the
    second product; about four times that, and in a small 16-bit result the
    weight of one flip of a large value."""
    if case["op"] == "mlp":
        return {"rel": 2e-3, "max": 2e-2}
    return {"f32": {"rel": 2e-6, "max": 3e-5},
            "f16": {"rel": 1e-4, "max": 2e-3},
            "bf16": {"rel": 8e-4, "max": 1.6e-2}}[case["out"]]


def exact(case, seed):
    x, w, c = _inputs(case, seed)
    a = x.double() @ w[0].double()
    if case["op"] == "matmul":
        return a if c is None else a + c.double()
    y = torch.nn.functional.silu(a) * (x.double() @ w[1].double())
    if case["op"] != "mlp":
        return y
    # Z is the product with the bf16 Y that the call returns.
    return y, y.bfloat16().double() @ w[2].double()
