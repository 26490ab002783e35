"""Y rows at any element: every kernel's vector stores (and the accumulating
GEMM's loads) of any alignment give what 16-byte aligned rows give, bit for
bit, and leave the elements around the view alone."""
from __future__ import annotations

import numpy as np
import pytest

from common import swiglu_inputs
from gpu_util import to_dev
from test_gpu_any_alignment import _Knobs

pytestmark = pytest.mark.gpu

TILE = dict(flex_tile=0, midm_max_m=64)
# (what, M, N, K, knobs, the bf16 SwiGLU's kernel and k splits, the GEMM's):
# edges of the 256-row and of the 64- to 256-column tiles, N % 4 of 0 to 3,
# columns past the last whole 8- and 16-byte chunk
CASES = [
    ("decode tile", 20, 133, 128, dict(flex_tile=0), ("decode_tile", 1), ("decode_tile", 1)),
    ("decode tile, splits", 64, 131, 640, dict(flex_tile=0, decode_splits=3), ("decode_tile", 3),
     ("decode_tile", 3)),
    ("small-M", 33, 134, 72, dict(flex_tile=0), ("small_m", 1), ("small_m", 1)),
    ("small-M, splits", 5, 9, 1000, dict(flex_tile=0, decode_splits=4), ("small_m", 4),
     ("small_m", 4)),
    ("tile", 257, 515, 64, dict(TILE, tile_wide=0, tile_splits=1), ("tile", 1), ("tile", 1)),
    ("tile, one exact tile", 256, 256, 128, dict(TILE, tile_wide=0, tile_splits=1), ("tile", 1),
     ("tile", 1)),
    ("tile, splits", 300, 254, 640, dict(TILE, tile_wide=0, tile_splits=3), ("tile", 3),
     ("tile", 3)),
    ("wide", 600, 1277, 512, dict(TILE), ("wide_tile", 1), ("tile", 2)),
    ("wide 11", 600, 1277, 512, dict(TILE, tile_wide=11), ("wide_tile", 1), ("tile", 2)),
    ("wide 7, splits", 300, 1277, 1024, dict(TILE, tile_wide=7, tile_splits=2), ("wide_tile", 2),
     ("tile", 2)),
    ("wide 11, splits", 300, 1277, 1024, dict(TILE, tile_wide=11, tile_splits=2),
     ("wide_tile", 2), ("tile", 2)),
]


def _views(gpu, M, N, dt, off, pad):
    """A view at element `off` of rows N + off + pad wide, and its buffer."""
    g = gpu.Generator(device="cuda").manual_seed(M + N)
    c0 = gpu.randn((M, N), generator=g, device="cuda").to(dt)
    buf = gpu.full((M, off + N + pad), -7.0, dtype=dt, device="cuda")
    buf[:, off:off + N] = c0
    return buf[:, off:off + N], buf


@pytest.mark.parametrize("what,M,N,K,knobs,swiglu,gemm", CASES, ids=[c[0] for c in CASES])
def test_any_y(llk, gpu, what, M, N, K, knobs, swiglu, gemm):
    print(f"case any y {what} M={M} N={N} K={K}", flush=True)
    x, wg, wu = swiglu_inputs(M, K, N, seed=M + K)
    xd = to_dev(gpu, x)
    pg, pu = llk.PackedWeights.from_host(wg), llk.PackedWeights.from_host(wu)
    ops = [(lambda y: llk.fused_swiglu(xd, pg, pu, out=y), (gpu.bfloat16, gpu.float32)),
           (lambda y: llk.matmul(xd, pg, out=y), (gpu.bfloat16, gpu.float16, gpu.float32)),
           (lambda y: llk.matmul(xd, pg, out=y, accumulate=True),
            (gpu.bfloat16, gpu.float16, gpu.float32))]
    with _Knobs(llk, **knobs):
        for op_name, want in (("fused_swiglu", swiglu), ("matmul", gemm)):
            plan = llk.describe_launch(op_name, M, N, K)
            assert (plan["kernel"], plan["splits"]) == want, plan
        for i, (op, types) in enumerate(ops):
            for dt in types:
                want = None
                for off, pad in ((0, -N % 8), (0, 1 - N % 2), (1, 0), (2, 1), (4, 4)):
                    y, buf = _views(gpu, M, N, dt, off, pad)
                    op(y)
                    gpu.cuda.synchronize()
                    if want is None:
                        want = y.clone()
                        assert np.isfinite(want.float().cpu().numpy()).all()
                    assert gpu.equal(y, want), (i, dt, off, pad)
                    assert (buf[:, :off] == -7).all() and (buf[:, off + N:] == -7).all(), (i, dt, off)
