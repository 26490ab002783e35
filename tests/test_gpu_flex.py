"""The flex tile kernel: against the oracle and, bit for bit, against the
unsplit (or equally split) 128-column tile kernel, whose sums it takes in the
same order -- on M around the 64- and 128-row tiles, N around the 32- to
128-column ones, K that ends inside a 64-k step (at every alignment of X and
of Y), k splits, accumulation, and the row-major weights of the KernelFn."""
from __future__ import annotations

import numpy as np
import pytest

from common import assert_parity, bf16_bits_to_f32, normal_bf16, swiglu_inputs, to_bf16_bits
from gpu_util import from_dev, to_dev

pytestmark = pytest.mark.gpu

TILES = [222, 224, 244]


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


def _tile(llk, S):
    """The 128-column tile kernel with S k splits, for any M."""
    return _Knobs(llk, flex_tile=0, tile_wide=0, tile_splits=S, decode_max_m=0, midm_max_m=64)


# (M, N, K, extra elements per X row, X's first element, S)
SHAPES = [
    (1, 5, 3, 0, 0, 1),           # K below one 16-byte chunk
    (64, 64, 64, 0, 0, 1),        # one exact tile of one step
    (65, 129, 72, 0, 0, 1),       # a row and a column past, K one chunk into a step
    (127, 31, 200, 8, 0, 1),
    (129, 33, 199, 0, 0, 1),      # odd K: odd rows, K inside a chunk
    (190, 257, 641, 3, 1, 1),     # odd base and stride
    (300, 1100, 1000, 0, 0, 1),
    (257, 200, 1343, 0, 0, 4),    # splits, the last one short and ragged
    (130, 96, 520, 2, 0, 3),
]


@pytest.mark.parametrize("cfg", TILES)
@pytest.mark.parametrize("M,N,K,pad,off,S", SHAPES)
def test_flex_matches_tile_kernel_and_oracle(llk, gpu, orc, cfg, M, N, K, pad, off, S):
    print(f"case flex {cfg} M={M} N={N} K={K} pad={pad} off={off} S={S}", flush=True)
    x, wg, wu = swiglu_inputs(M, K, N, seed=M + K)
    big = np.zeros((M, K + pad + off), np.uint16)
    big[:, off:off + K] = x
    xd = to_dev(gpu, big)[:, off:off + K]
    pg, pu = llk.PackedWeights.from_host(wg), llk.PackedWeights.from_host(wu)
    out = {}
    for name, knobs in (("flex", _Knobs(llk, flex_tile=cfg, tile_splits=S)), ("tile", _tile(llk, S))):
        with knobs:
            if name == "flex":
                plan = llk.describe_launch("fused_swiglu", M, N, K)
                assert plan["kernel"] == "flex_tile" and plan["splits"] == S, plan
            out[name] = [from_dev(llk.fused_swiglu(xd, pg, pu, out_dtype=gpu.float32)),
                         from_dev(llk.fused_swiglu(xd, pg, pu)),
                         from_dev(llk.matmul(xd, pg, out_dtype=gpu.float32)),
                         from_dev(llk.matmul(xd, pg, out_dtype=gpu.bfloat16)),
                         llk.matmul(xd, pg, out_dtype=gpu.float16).cpu().numpy().view(np.uint16)]
    for a, b in zip(out["flex"], out["tile"]):
        assert np.array_equal(a, b)
    assert_parity(out["flex"][0], orc.swiglu(x, wg, wu)[0], "swiglu")
    assert_parity(out["flex"][2], orc.gemm(x, wg)[0], "gemm")


@pytest.mark.parametrize("cfg", TILES)
@pytest.mark.parametrize("N,shift", [(96, 0), (100, 4), (77, 1)])
def test_flex_accumulates_into_a_view(llk, gpu, cfg, N, shift):
    """C += A B in every result type, into a view of any alignment: round(P +
    C0) bit for bit, the elements around the view untouched."""
    print(f"case flex accumulate {cfg} N={N} shift={shift}", flush=True)
    M, K = 131, 264
    a, b = normal_bf16(3, 0, (M, K)), normal_bf16(3, 1, (K, N), 1.0 / np.sqrt(K))
    ad, pb = to_dev(gpu, a), llk.PackedWeights.from_host(b)
    with _Knobs(llk, flex_tile=cfg, tile_splits=1):
        p = from_dev(llk.matmul(ad, pb, out_dtype=gpu.float32))
        for dt in (gpu.float32, gpu.bfloat16, gpu.float16):
            buf = gpu.randn((M, N + 2 * shift + 1), device="cuda").to(dt)
            before = buf.clone()
            c = buf[:, shift:shift + N]
            llk.matmul(ad, pb, out=c, accumulate=True)
            want = (gpu.from_numpy(p).cuda() + before[:, shift:shift + N].float()).to(dt)
            assert gpu.equal(c, want), dt
            before[:, shift:shift + N] = c
            assert gpu.equal(buf, before), "wrote outside the view"


@pytest.mark.parametrize("cfg", TILES)
@pytest.mark.parametrize("M,N,K,ldw,S", [(65, 129, 72, 131, 1), (130, 40, 640, 40, 1),
                                        (70, 1, 64, 1, 1), (70, 1, 640, 1, 1), (70, 3, 200, 8, 1),
                                        (129, 300, 1000, 301, 3)])
def test_flex_row_major_weights(llk, gpu, cfg, M, N, K, ldw, S):
    """The KernelFn on device weights of any stride and alignment: the packed
    path's bits; rows of Inf past the last column change nothing."""
    print(f"case flex row-major {cfg} M={M} N={N} K={K} ldw={ldw} S={S}", flush=True)
    x, wg, wu = swiglu_inputs(M, K, N, seed=N)
    xd = to_dev(gpu, x)
    dev = []
    for w in (wg, wu):
        big = np.full((K, ldw), to_bf16_bits(np.array([np.inf], np.float32))[0], np.uint16)
        big[:, :N] = w
        dev.append(to_dev(gpu, big)[:, :N])
    pg, pu = llk.PackedWeights.from_host(wg), llk.PackedWeights.from_host(wu)
    cache = llk.JitCache()
    for out, dt in ((0, gpu.bfloat16), (2, gpu.float32)):
        fn = cache.lookup_or_compile(llk.KernelKey(operation=0, isa=7, N=N, K=K, output_type=out))
        y = gpu.full((M, N), float("nan"), dtype=dt, device="cuda")
        with _Knobs(llk, flex_tile=cfg, tile_splits=S):
            fn(xd, dev[0], dev[1], y, y)
            ref = llk.fused_swiglu(xd, pg, pu, out_dtype=dt)
        assert np.array_equal(from_dev(y), from_dev(ref))
    cache.close()


def test_flex_special_values(llk, gpu):
    """Infinities, NaN and the largest bf16 values of one row of X stay in
    that row, also where K ends inside a step (the next row's elements are
    read beside it) and past the last row."""
    print("case flex special values", flush=True)
    M, N, K = 70, 40, 1003
    x, wg, _ = swiglu_inputs(M, K, N, seed=9)
    f = bf16_bits_to_f32(x)
    f[1, 0], f[33, :2], f[69, 5] = np.inf, np.nan, -3.0e38
    pg = llk.PackedWeights.from_host(wg)
    for cfg in TILES:
        with _Knobs(llk, flex_tile=cfg, tile_splits=1):
            c = from_dev(llk.matmul(to_dev(gpu, to_bf16_bits(f)), pg, out_dtype=gpu.float32))
        with _tile(llk, 1):
            t = from_dev(llk.matmul(to_dev(gpu, to_bf16_bits(f)), pg, out_dtype=gpu.float32))
        assert np.array_equal(c, t, equal_nan=True)
        rows = np.ones(M, bool)
        rows[[1, 33, 69]] = False
        assert np.isfinite(c[rows]).all() and not np.isfinite(c[[1, 33]]).any()
