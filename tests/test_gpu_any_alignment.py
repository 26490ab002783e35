"""X rows at any element: the small-M kernel's and the padding copy's loads of
any alignment give what the same values in aligned rows give, bit for bit, and
the row after K's last element never reaches a result."""
from __future__ import annotations

import numpy as np
import pytest

from common import swiglu_inputs
from gpu_util import from_dev, to_dev

pytestmark = pytest.mark.gpu


class _Knobs:
    def __init__(self, llk, **kv):
        self.llk, self.kv, self.old = llk, kv, {}

    def __enter__(self):
        for k, v in self.kv.items():
            self.old[k] = self.llk.get_tunable(k)
            self.llk.set_tunable(k, v)

    def __exit__(self, *exc):
        for k, v in self.old.items():
            self.llk.set_tunable(k, v)


def _at(gpu, x, off, pad):
    """x at element `off` of wider rows whose other elements are NaN."""
    M, K = x.shape
    big = np.full((M, off + K + pad), 0x7FC0, np.uint16)
    big[:, off:off + K] = x
    return to_dev(gpu, big)[:, off:off + K]


@pytest.mark.parametrize("K", [8, 64, 200, 1000])
@pytest.mark.parametrize("M,W", [(1, 1), (17, 2), (32, 4), (33, 1), (64, 2)])
def test_small_m_any_alignment(llk, gpu, M, W, K):
    print(f"case any alignment small M={M} W={W} K={K}", flush=True)
    x, wg, wu = swiglu_inputs(M, K, 96, seed=M + K)
    pg, pu = llk.PackedWeights.from_host(wg), llk.PackedWeights.from_host(wu)
    with _Knobs(llk, decode_group_width=W, decode_splits=1):
        want = [from_dev(llk.fused_swiglu(to_dev(gpu, x), pg, pu, out_dtype=gpu.float32)),
                from_dev(llk.matmul(to_dev(gpu, x), pg))]
        for off, pad in ((0, 1), (1, 0), (3, 2), (2, 6)):
            xd = _at(gpu, x, off, pad)
            got = [from_dev(llk.fused_swiglu(xd, pg, pu, out_dtype=gpu.float32)),
                   from_dev(llk.matmul(xd, pg))]
            assert all(np.array_equal(g, w) for g, w in zip(got, want)), (off, pad)


@pytest.mark.parametrize("K", [1, 7, 63, 65, 199, 520])
@pytest.mark.parametrize("M", [5, 40, 70])
def test_ragged_k_any_alignment(llk, gpu, M, K):
    """K that ends inside a 16-byte chunk: as with zero columns up to K + 8."""
    print(f"case any alignment ragged M={M} K={K}", flush=True)
    N = 72
    x, wg, _ = swiglu_inputs(M, K, N, seed=M + K)
    Kp = (K + 63) // 64 * 64
    xp, wp = np.zeros((M, Kp), np.uint16), np.zeros((Kp, N), np.uint16)
    xp[:, :K], wp[:K] = x, wg
    pg, pp = llk.PackedWeights.from_host(wg), llk.PackedWeights.from_host(wp)
    with _Knobs(llk, decode_group_width=1, decode_splits=1, flex_tile=0, tile_splits=1,
                midm_max_m=64):
        want = from_dev(llk.matmul(to_dev(gpu, xp), pp))
        for off, pad in ((0, 0), (0, 1), (1, 3)):
            assert np.array_equal(from_dev(llk.matmul(_at(gpu, x, off, pad), pg)), want), (off, pad)


# The launch depends on the shape and on whether X's rows are 16-byte aligned;
# views of one alignment then take the same sums.
STRIDED = [("matmul", 219, 640, 517), ("fused_swiglu", 101, 2752, 860),
           ("fused_swiglu", 117, 732, 533), ("matmul", 195, 583, 718)]


@pytest.mark.parametrize("op,M,K,N", STRIDED)
def test_row_stride_leaves_the_sums_alone(llk, gpu, op, M, K, N):
    print(f"case row stride {op} M={M} K={K} N={N}", flush=True)
    x, wg, wu = swiglu_inputs(M, K, N, seed=M + K)
    pg, pu = llk.PackedWeights.from_host(wg), llk.PackedWeights.from_host(wu)
    views = ((0, 0), (0, 8), (8, 56)) if K % 8 == 0 else ((0, 0), (0, 1), (1, 0), (1, 2), (2, 0))
    got = []
    for off, pad in views:
        xd = _at(gpu, x, off, pad)
        y = llk.matmul(xd, pg) if op == "matmul" else llk.fused_swiglu(xd, pg, pu,
                                                                      out_dtype=gpu.float32)
        got.append(from_dev(y))
    for g, v in zip(got, views):
        assert np.array_equal(g, got[0]), v
