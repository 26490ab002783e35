"""Results wider than bf16: the plan the dispatcher takes sums no more k in one
accumulator than the plan without the flex tile kernel and the one-launch
rule, whose fp32 results it must not be further off than."""
from __future__ import annotations

import random

import pytest

import dslcompiler_amd as llk


def _longest(plan, op, M, K):
    """64-k steps in one accumulator (the small-M kernel's waves share k)."""
    steps = -(-((K + 63) // 64) // plan["splits"])
    if plan["kernel"] != "small_m":
        return steps
    width = plan["group_width"]
    groups = width if width == 1 or (op == "fused_swiglu" and M <= 32) else width // 2
    return -(-steps // (plan["threads_per_workgroup"] // 64 // groups))


@pytest.mark.parametrize("op", ["fused_swiglu", "matmul"])
@pytest.mark.parametrize("rows", [(1, 64), (65, 1000)])
def test_sums_no_longer(op, rows):
    rng = random.Random(rows[1])
    for _ in range(150):
        M, K, N = rng.randint(*rows), rng.randint(512, 6000), rng.randint(1376, 14336)
        if rng.random() < 0.6:
            K -= K % 64
        kw = dict(x_aligned=K % 8 == 0, out_f32=True)
        new = llk.describe_launch(op, M, N, K, **kw)
        llk.set_tunable("flex_tile", 0)
        try:
            old = llk.describe_launch(op, M, N, K, **kw)
        finally:
            llk.set_tunable("flex_tile", 1)
        assert _longest(new, op, M, K) <= _longest(old, op, M, K), (op, M, K, N, new, old)


def test_scratch_size_covers_every_plan():
    """A caller who sizes scratch with the library's own query has room for
    the launch the library takes, for either result type and alignment of X."""
    rng = random.Random(4)
    shapes = [(713, 3384, 1325), (547, 3984, 1330), (265, 3648, 676), (192, 4928, 839)]
    for _ in range(400):
        K, N = rng.randint(512, 6000), rng.randint(512, 3000)
        shapes.append((rng.randint(1, 800), K - K % rng.choice([1, 8, 64]), N))
    for M, K, N in shapes:
        size = llk.swiglu_scratch_size(M, N, K)
        for aligned in (True, False):
            for f32 in (True, False):
                plan = llk.describe_launch("fused_swiglu", M, N, K, x_aligned=aligned, out_f32=f32)
                assert plan["workspace_bytes"] <= size, (M, K, N, aligned, f32, plan, size)


# (op, M, K, N, us with the other kernels, us with the flex tile kernel) on
# MI355X, the weights from HBM at every call
MEASURED = [
    ("matmul", 3501, 640, 12384, 70.5, 95.7), ("matmul", 4061, 9896, 1696, 147.2, 190.4),
    ("fused_swiglu", 110, 11904, 1488, 25.4, 33.8), ("matmul", 299, 3982, 11152, 53.6, 68.3),
    ("fused_swiglu", 74, 896, 11104, 12.5, 15.7), ("matmul", 601, 4048, 5851, 49.0, 61.1),
    ("fused_swiglu", 282, 8640, 976, 30.6, 35.8), ("fused_swiglu", 85, 704, 13280, 11.9, 14.8),
    ("matmul", 4062, 546, 944, 24.4, 12.1), ("fused_swiglu", 860, 576, 2113, 20.3, 10.5),
    ("matmul", 198, 1683, 848, 21.3, 11.5), ("fused_swiglu", 411, 896, 4432, 20.9, 13.6),
    ("matmul", 926, 1946, 960, 30.0, 19.2), ("fused_swiglu", 300, 1000, 1100, 23.6, 15.1),
]


@pytest.mark.parametrize("op,M,K,N,other,flex", MEASURED)
def test_flex_tile_kernel_where_it_is_faster(op, M, K, N, other, flex):
    plan = llk.describe_launch(op, M, N, K, x_aligned=K % 8 == 0)
    assert (plan["kernel"] == "flex_tile") == (flex < other), plan
