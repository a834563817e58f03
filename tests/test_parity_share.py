"""GPU parity of the share kernel (DTAS_GEMM_SHARE): every instantiated rows x columns, fp16 and 8-bit weights, at ragged M, N
and K, with every epilogue, against the CPU oracle; and the line that takes it when no config is given."""
import numpy as np
import pytest
import torch

from dtas_amd import _lib, ops
from gpu_util import Guarded, cfg, dev

pytestmark = pytest.mark.gpu

F16_SHAPES = [(r, c) for r in (16, 32, 48, 64) for c in (16, 32, 48, 64, 128) if (r, c) != (16, 48)] + [(96, 16), (96, 32), (96, 48), (128, 48)]
Q8_SHAPES = [(r, c) for r in (16, 32, 48, 64) for c in (16, 32, 48, 64, 128)] + [(80, 16), (96, 32), (96, 48)]


def _inputs(M, N, K, seed):
    rng = np.random.default_rng(seed)
    f16 = lambda *s: rng.standard_normal(s).astype(np.float16)
    return f16(M, K), f16(N), f16(M, N), f16(M, N), rng


def _check(got, want, r1, r2):
    """The oracle's fp16 steps on another summation order of the product: an fp16 ulp of the largest value a step rounds
    (2^-10 of it), twice for the sums on both sides of a rounding boundary, over an fp32 sum's own error (1e-3)."""
    g, w = got.astype(np.float64), want.astype(np.float64)
    big = np.maximum(np.abs(w), np.maximum(np.abs(r1), np.abs(r2)).astype(np.float64)) if r1 is not None else np.abs(w)
    assert np.isfinite(g).all() and (np.abs(g - w) <= 2e-3 + 2.0 ** -9 * big).all(), np.abs(g - w).max()


# columns per workgroup: all of them, one short, a single one; K: one piece, a segment and a piece, whole segments
@pytest.mark.parametrize("rows,cols", F16_SHAPES)
@pytest.mark.parametrize("kind,less,N_of,K", [(0, 0, lambda c: 256 * c, 264), (1, 3, lambda c: 256 * c - 255, 520), (2, 15, lambda c: 1027, 1032),
                                              (3, 1, lambda c: 255 * c + 2, 8), (0, 7, lambda c: 3, 2048)])
def test_share_kernels(oracle, rows, cols, kind, less, N_of, K):
    M, N = rows - less, N_of(cols)
    a, bias, r1, r2, rng = _inputs(M, N, K, rows + cols + kind)
    w = (rng.standard_normal((N, K)) * 0.05).astype(np.float16)
    res = (dev(r1), dev(r2)) if kind in (1, 2) else (None, None)
    out = Guarded((M, N), torch.float32 if kind == 2 else torch.float16)
    ops.gemm(dev(a), dev(w), dev(bias), out.t, cfg(variant=_lib.GEMM_SHARE, tile=[rows, cols, 0]), epilogue=kind, res1=res[0], res2=res[1])
    add2 = kind in (1, 2)
    want = oracle.c.gemm_fused(a, w, bias, r1 if add2 else None, r2 if add2 else None, kind, threads=8)
    _check(out.check(), want, r1 if add2 else None, r2)


@pytest.mark.parametrize("rows,cols", Q8_SHAPES)
@pytest.mark.parametrize("kind,less,N_of,K", [(0, 0, lambda c: 256 * c, 256), (1, 3, lambda c: 256 * c - 255, 512), (2, 15, lambda c: 1027, 1280),
                                              (3, 1, lambda c: 255 * c + 2, 768)])
def test_share_kernels_on_8_bit_weights(oracle, rows, cols, kind, less, N_of, K):
    M, N = rows - less, N_of(cols)
    a, bias, r1, r2, rng = _inputs(M, N, K, rows + cols + kind)
    wq = rng.integers(0, 2 ** 32, (N, K // 4), dtype=np.uint32)
    scale = (rng.random((N, K // 32)) * 4e-4 + 1e-4).astype(np.float16)
    w = oracle.c.decode_q8(wq, scale)
    res = (dev(r1), dev(r2)) if kind in (1, 2) else (None, None)
    out = Guarded((M, N), torch.float32 if kind == 2 else torch.float16)
    ops.gemm_q8(dev(a), dev(wq.view(np.int32)), dev(scale), dev(bias), out.t, cfg(variant=_lib.GEMM_SHARE, tile=[rows, cols, 0]), kind, res[0], res[1])
    add2 = kind in (1, 2)
    _check(out.check(), oracle.c.gemm_fused(a, w, bias, r1 if add2 else None, r2 if add2 else None, kind, threads=8), r1 if add2 else None, r2)


@pytest.mark.parametrize("rows,cols", [(16, 16), (16, 32), (16, 48), (32, 16), (32, 32), (32, 48), (0, 0)])
@pytest.mark.parametrize("K", [256, 768, 1280])
@pytest.mark.parametrize("bad", [600.0, float("inf"), float("nan")])
def test_the_scales_behind_a_row_stay_its_neighbours(oracle, rows, cols, K, bad):
    # K ends inside a segment of 512: the 16 bytes behind a row's scales are the next row's, here too large for fp16 times a byte,
    # infinite or NaN.  Only that row's column may show it (0, 0: what runs without a config)
    M, N = rows or 29, 256 * (cols or 16) - 3
    a, bias, _, _, rng = _inputs(M, N, K, K + rows)
    wq = rng.integers(0, 2 ** 32, (N, K // 4), dtype=np.uint32)
    scale = (rng.random((N, K // 32)) * 4e-4 + 1e-4).astype(np.float16)
    good = np.arange(N) % 3 != 2
    scale[~good] = bad
    out = Guarded((M, N), torch.float16)
    share = cfg(variant=_lib.GEMM_SHARE, tile=[rows, cols, 0]) if rows else None
    ops.gemm_q8(dev(a), dev(wq.view(np.int32)), dev(scale), dev(bias), out.t, share)
    want = oracle.c.gemm_fused(a, oracle.c.decode_q8(wq[good], scale[good]), np.ascontiguousarray(bias[good]), None, None, 0, threads=8)
    _check(out.check()[:, good], want, None, None)


@pytest.mark.parametrize("rows,cols", [(16, 16), (32, 48), (64, 128), (96, 32), (128, 48)])
@pytest.mark.parametrize("bad", [65504.0, float("inf"), float("nan")])
def test_non_finite_rows_and_columns_stay_where_they_are(oracle, rows, cols, bad):
    # the last element of K, the last rows of A and of a workgroup's columns: what lies behind them is read as zero, and zero times
    # any of these would be seen
    M, N, K = rows - 3, 256 * cols - 5, 520
    a, bias, _, _, rng = _inputs(M, N, K, rows + cols)
    w = (rng.standard_normal((N, K)) * 0.05).astype(np.float16)
    a[M - 1, K - 1] = a[0, 0] = a[M // 2, 256] = bad
    w[cols - 1::cols, K - 1] = bad
    w[N - 1, 0] = bad
    r, c = np.isfinite(a).all(1) & (np.abs(a) < 6e4).all(1), np.isfinite(w).all(1) & (np.abs(w) < 6e4).all(1)
    out = Guarded((M, N), torch.float16)
    ops.gemm(dev(a), dev(w), dev(bias), out.t, cfg(variant=_lib.GEMM_SHARE, tile=[rows, cols, 0]))
    want = oracle.c.gemm_fused(a[r], w[c], np.ascontiguousarray(bias[c]), None, None, 0, threads=8)
    _check(np.ascontiguousarray(out.check()[r][:, c]), want, None, None)


# the rows of A up to which the share kernel is chosen
@pytest.mark.parametrize("M", [3, 5, 16, 17, 33, 64, 65, 96, 128])
@pytest.mark.parametrize("N,K,up_to", [(2560, 2560, 65), (7680, 2560, 96), (2560, 10240, 17), (10240, 520, 64), (257, 256, 96), (17000, 2048, 64)])
def test_what_runs_without_a_config_either_side_of_the_line(oracle, M, N, K, up_to):
    assert (_lib.builtin_gemm(M, N, K).config.variant == _lib.GEMM_SHARE) == (M <= up_to)
    a, bias, _, _, rng = _inputs(M, N, K, M + N)
    w = (rng.standard_normal((N, K)) * 0.05).astype(np.float16)
    out = Guarded((M, N), torch.float16)
    ops.gemm(dev(a), dev(w), dev(bias), out.t)
    rows = np.unique(np.linspace(0, M - 1, 6).astype(int))
    _check(out.check()[rows], oracle.c.gemm(np.ascontiguousarray(a[rows]), w, bias, threads=8), None, None)


def test_share_kernel_exact_and_refuses_what_it_cannot_hold():
    rng = np.random.default_rng(6)
    ai, wi = rng.integers(-2, 3, (29, 1032)).astype(np.float16), rng.integers(-2, 3, (700, 1032)).astype(np.float16)
    out = Guarded((29, 700), torch.float16)
    ops.gemm(dev(ai), dev(wi), None, out.t, cfg(variant=_lib.GEMM_SHARE, tile=[32, 16, 0]))
    assert np.array_equal(out.check().astype(np.float64), ai.astype(np.float64) @ wi.astype(np.float64).T)
    for M, tile, block, msg in ((17, [16, 16, 0], 256, "cannot hold M=17"), (8, [16, 48, 0], 256, "no share kernel"), (8, [16, 16, 0], 512, "256 threads")):
        with pytest.raises(_lib.DtasError, match=msg):
            _lib.describe_launch(_lib.OP_GEMM_F16, M, 64, 64, cfg(variant=_lib.GEMM_SHARE, block=block, tile=tile))
