"""Up to 64 rows with N > 2176: the one-launch plans chosen in place of a k
split (the small-M kernel unsplit at width 1 and 2) and, for K inside one
64-k step, the flex tile kernel's 64-row tiles, against the oracle on both
sides of the rule, with every X alignment and output type; and the rule
itself: the same launch for every result type of the SwiGLU, and for C = A B
and C += A B."""
from __future__ import annotations

import numpy as np
import pytest

from common import assert_parity, assert_parity_bf16, normal_bf16, swiglu_inputs
from gpu_util import from_dev, to_dev

pytestmark = pytest.mark.gpu

# (op, M, N, K, X aligned, the kernel chosen, its k splits)
CASES = [
    ("matmul", 7, 2560, 1280, True, "small_m", 1),
    ("matmul", 64, 2177, 65, False, "small_m", 1),        # the first width of the rule
    ("matmul", 32, 2176, 520, True, "small_m", 1),        # ... and the last one below it
    ("matmul", 40, 2880, 768, True, "small_m", 1),
    ("fused_swiglu", 1, 2305, 520, True, "small_m", 1),
    ("fused_swiglu", 64, 2944, 576, True, "decode_tile", 1),
    ("fused_swiglu", 33, 4097, 1031, False, "small_m", 1),
    ("fused_swiglu", 41, 8496, 2241, False, "small_m", 1),
    ("fused_swiglu", 64, 4096, 63, False, "flex_tile", 1),  # K inside one step
    ("fused_swiglu", 54, 2184, 24, True, "flex_tile", 1),
    ("matmul", 36, 8240, 10, False, "flex_tile", 1),
    ("fused_swiglu", 64, 4096, 65, False, "small_m", 1),    # ... and one past it
]


@pytest.mark.parametrize("op,M,N,K,aligned,kernel,S", CASES,
                         ids=[f"{c[0]}-{c[1]}x{c[2]}x{c[3]}" for c in CASES])
def test_small_routes(llk, gpu, orc, op, M, N, K, aligned, kernel, S):
    print(f"case small routes {op} M={M} N={N} K={K}", flush=True)
    plan = llk.describe_launch(op, M, N, K, x_aligned=aligned)
    if kernel:
        assert (plan["kernel"], plan["splits"]) == (kernel, S), plan
    x, wg, wu = swiglu_inputs(M, K, N, seed=M + N)
    xd, pg = to_dev(gpu, x), llk.PackedWeights.from_host(wg)
    if op == "fused_swiglu":
        pu = llk.PackedWeights.from_host(wu)
        ref = orc.swiglu(x, wg, wu)[0]
        f32 = from_dev(llk.fused_swiglu(xd, pg, pu, out_dtype=gpu.float32))
        b16 = from_dev(llk.fused_swiglu(xd, pg, pu))
    else:
        ref = orc.gemm(x, wg)[0]
        f32 = from_dev(llk.matmul(xd, pg, out_dtype=gpu.float32))
        b16 = from_dev(llk.matmul(xd, pg, out_dtype=gpu.bfloat16))
        f16 = llk.matmul(xd, pg, out_dtype=gpu.float16).cpu().numpy()
        assert np.array_equal(f16, f32.astype(np.float16))
        c = gpu.ones((M, N), dtype=gpu.float32, device="cuda")
        llk.matmul(xd, pg, out=c, accumulate=True)
        assert np.array_equal(from_dev(c), f32 + np.float32(1))  # the same sums, then C
    assert_parity(f32, ref, op)
    assert_parity_bf16(b16, ref, op)


def test_choice_ignores_type_and_accumulation(llk):
    for M in (1, 16, 33, 64):
        for N in (2177, 2560, 4097, 8496, 13824):
            for K in (40, 64, 520, 1031, 2048, 4096):
                al = K % 8 == 0
                p = llk.describe_launch("matmul", M, N, K, x_aligned=al)
                q = llk.describe_launch("matmul", M, N, K, x_aligned=al, accumulate=True)
                r = llk.describe_launch("fused_swiglu", M, N, K, x_aligned=al)
                s = llk.describe_launch("fused_swiglu", M, N, K, x_aligned=al, out_f32=True)
                for k in ("kernel", "splits", "workgroups"):
                    assert p[k] == q[k], (M, N, K, p, q)
                    assert r[k] == s[k], (M, N, K, r, s)


def test_flex_choice_ignores_type(llk):
    """Above 64 rows the other kernels' splits may differ by the SwiGLU's
    result type (the wide tiles give bf16 alone); the flex tile kernel is
    taken for both or neither, with one split."""
    taken = 0
    for M in (65, 128, 191, 300, 512, 1000):
        for N in (544, 1100, 2048, 4432):
            for K in (576, 1000, 1031, 2048, 4096):
                p, q = (llk.describe_launch("fused_swiglu", M, N, K, x_aligned=K % 8 == 0,
                                            out_f32=f32) for f32 in (False, True))
                if "flex_tile" in (p["kernel"], q["kernel"]):
                    taken += 1
                    for k in ("kernel", "splits", "workgroups"):
                        assert p[k] == q[k], (M, N, K, p, q)
    assert taken > 20
