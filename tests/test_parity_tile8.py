"""GPU parity of the 8-wavefront GEMM tiles: every tile and stage count on sizes at its edges, whole and with K in parts, with
every epilogue; and what a call of more than 128 rows without a config runs."""
import numpy as np
import pytest
import torch

from dtas_amd import _lib, ops
from gpu_util import Guarded, assert_bits_equal, cfg, dev

RTOL, ATOL = 1e-2, 2e-3
# (rows, columns, k tiles of W that the LDS holds; 2: the ring of five operand units)
TILES = [(128, 64, 4), (96, 128, 4), (128, 128, 4), (160, 128, 4), (192, 128, 4), (224, 128, 3), (256, 128, 3), (96, 256, 3), (128, 256, 3),
         (160, 256, 3), (192, 256, 3), (192, 256, 2), (224, 256, 3), (256, 256, 2)]


def _check(got, oracle_out, f64):
    got = got.astype(np.float64)
    assert np.isfinite(got).all()
    assert (np.abs(got - f64) <= ATOL + RTOL * np.abs(f64)).all()
    # against the oracle (same fp32 arithmetic, another summation order): about one fp16 ulp
    want = oracle_out.astype(np.float64)
    assert (np.abs(got - want) <= 1e-3 + 2.0 ** -9 * np.abs(want)).all()


def _inputs(M, N, K, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((M, K)).astype(np.float16), (rng.standard_normal((N, K)) * 0.02).astype(np.float16),
            rng.uniform(-1, 1, N).astype(np.float16))


def _cfg(bm, bn, stages, split=1):
    return cfg(variant=_lib.GEMM_MFMA, block=512, vec=8, unroll=2 if stages == 2 else 0, tile=[bm, bn, 64], split_k=split)


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn,stages", TILES)
def test_every_tile_at_its_edges(oracle, bm, bn, stages):
    # one row and column either side of whole tiles; one k tile, as many as there are stages and a chunk more, and one fewer
    for M, N, K, split in ((3, 5, 8, 1), (bm - 1, bn + 1, 64, 1), (bm + 1, 2 * bn - 1, 64 * stages + 8, 1), (2 * bm, bn, 64 * (stages + 1), 1),
                           (bm + 33, bn + 8, 64 * (stages - 1) - 8, 1), (bm + 7, bn + 9, 1096, 3), (2 * bm - 5, bn, 2048, 6)):
        a, w, bias = _inputs(M, N, K, M + N + K)
        out = Guarded((M, N), torch.float16)
        ops.gemm(dev(a), dev(w), dev(bias), out.t, _cfg(bm, bn, stages, split))
        _check(out.check(), oracle.c.gemm(a, w, bias, threads=8), oracle.np64.gemm(a, w, bias))


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn,stages", TILES)
@pytest.mark.parametrize("epilogue", [_lib.EPI_BIAS_ADD2, _lib.EPI_BIAS_ADD2_CAST_F32, _lib.EPI_BIAS_GELU])
def test_every_epilogue_of_every_tile(bm, bn, stages, epilogue):
    # the epilogues act on the product rounded to fp16: the same bits as on 64x64 tiles, whose k order is the same
    M, N, K = bm + 5, bn + 12, 200
    a, w, bias = (dev(x) for x in _inputs(M, N, K, bm + bn))
    g = torch.Generator(device="cuda").manual_seed(1)
    res = [torch.randn(M, N, device="cuda", generator=g).half() for _ in range(2)] if epilogue != _lib.EPI_BIAS_GELU else [None, None]
    plain = cfg(variant=_lib.GEMM_MFMA, block=256, vec=8, unroll=2, tile=[64, 64, 64])
    mm, mm8 = (torch.empty(M, N, dtype=torch.float16, device="cuda") for _ in range(2))
    ops.gemm(a, w, None, mm, plain)
    ops.gemm(a, w, None, mm8, _cfg(bm, bn, stages))
    same = mm == mm8    # (16x16x32 and 32x32x16 products are added in another order: a last bit may differ)
    assert float(same.float().mean()) > 0.98
    outs = []
    for c in (plain, _cfg(bm, bn, stages)):
        out = Guarded((M, N), torch.float32 if epilogue == _lib.EPI_BIAS_ADD2_CAST_F32 else torch.float16)
        ops.gemm(a, w, bias, out.t, c, epilogue=epilogue, res1=res[0], res2=res[1])
        outs.append(out.check())
    keep = same.cpu().numpy()
    assert_bits_equal(outs[0][keep], outs[1][keep])


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(129, 4096, 1024), (203, 2560, 2560), (300, 520, 4096), (385, 7680, 520), (600, 1000, 264), (1025, 2560, 2560),
                                   (1150, 100, 72), (200, 7, 8), (700, 2048, 10240), (897, 2560, 2048)])
def test_what_runs_without_a_config(oracle, M, N, K):
    a, w, bias = _inputs(M, N, K, M + N + K)
    out = Guarded((M, N), torch.float16)
    ops.gemm(dev(a), dev(w), dev(bias), out.t)
    got = out.check()
    named = Guarded((M, N), torch.float16)
    ops.gemm(dev(a), dev(w), dev(bias), named.t, _lib.builtin_gemm(M, N, K).config)
    assert_bits_equal(got, named.check())
    rows = np.linspace(0, M - 1, min(M, 64)).astype(int)
    _check(got[rows], oracle.c.gemm(a[rows], w, bias, threads=8), oracle.np64.gemm(a[rows], w, bias))


Q8_TILES = [(96, 128), (128, 128), (160, 128), (192, 128), (256, 128)]


def _q8(N, K, seed):
    rng = np.random.default_rng(seed)
    return rng.integers(0, 2 ** 32, (N, K // 4), dtype=np.uint32), (rng.random((N, K // 32)) * 0.0008 + 0.0002).astype(np.float16)


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn", Q8_TILES)
def test_every_8_bit_tile_at_its_edges(oracle, bm, bn):
    # k tiles: half of one, fewer than the loads run ahead, a whole number of the loop's three, one and two more; K in parts
    for M, N, K, split in ((3, 5, 32, 1), (bm - 1, bn + 1, 64, 1), (bm + 1, 2 * bn - 1, 224, 1), (2 * bm, bn, 384, 1), (bm + 33, bn + 8, 448, 1),
                           (bm + 7, bn + 9, 1056, 3), (bm - 5, bn, 2080, 6)):
        a, _, bias = _inputs(M, N, K, M + N + K)
        wq, scale = _q8(N, K, M + K)
        w = oracle.c.decode_q8(wq, scale, threads=8)
        out = Guarded((M, N), torch.float16)
        ops.gemm_q8(dev(a), torch.from_numpy(wq.view(np.int32)).cuda(), dev(scale), dev(bias), out.t, _cfg(bm, bn, 0, split))
        _check(out.check(), oracle.c.gemm(a, w, bias, threads=8), oracle.np64.gemm(a, w, bias))


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn", Q8_TILES)
def test_8_bit_tiles_with_the_scales_of_four_k_tiles_in_one_load(oracle, bm, bn):
    # 1 .. 9 k tiles (none to two of the loop's four, none to three behind it), parts of K that begin at odd k tiles; scales off the
    # 4-byte grid and K = 64 k + 32 take the loop that loads them one by one: the same bits from both on the same weights
    for K, split in ((64, 1), (128, 1), (192, 1), (256, 1), (320, 1), (384, 1), (448, 1), (512, 1), (576, 1), (1088, 4), (2112, 7), (640, 2)):
        M, N = bm + 5, bn + 7
        a, _, bias = _inputs(M, N, K, K + bm)
        wq, scale = _q8(N, K, K)
        w = oracle.c.decode_q8(wq, scale, threads=8)
        words = torch.from_numpy(wq.view(np.int32)).cuda()
        out = Guarded((M, N), torch.float16)
        ops.gemm_q8(dev(a), words, dev(scale), dev(bias), out.t, _cfg(bm, bn, 0, split))
        got = out.check()
        _check(got, oracle.c.gemm(a, w, bias, threads=8), oracle.np64.gemm(a, w, bias))
        off = torch.zeros(N * (K // 32) + 1, dtype=torch.float16, device="cuda")
        off[1:] = dev(scale).flatten()
        ops.gemm_q8(dev(a), words, off[1:].view(N, K // 32), dev(bias), out.t, _cfg(bm, bn, 0, split))
        assert_bits_equal(out.check(), got)
        # what lies behind a row's scales is the next row's: infinities there stay with that row
        scale[1::2, :6] = np.inf
        ops.gemm_q8(dev(a), words, dev(scale), dev(bias), out.t, _cfg(bm, bn, 0, split))
        assert_bits_equal(np.ascontiguousarray(out.check()[:, ::2]), np.ascontiguousarray(got[:, ::2]))


@pytest.mark.gpu
@pytest.mark.parametrize("epilogue", [_lib.EPI_BIAS, _lib.EPI_BIAS_ADD2, _lib.EPI_BIAS_ADD2_CAST_F32, _lib.EPI_BIAS_GELU])
@pytest.mark.parametrize("M,N,K", [(97, 2560, 2560), (130, 768, 1024), (203, 520, 2080), (320, 2560, 10240), (450, 7680, 320), (700, 10240, 256), (900, 1000, 4096)])
def test_8_bit_weights_without_a_config(M, N, K, epilogue):
    # against the fp16 GEMM on the dequantised weights, which are the same numbers: another order of the fp32 sums can move the
    # rounding of the product and of the up to three steps behind it by an fp16 ulp each, 2^-10 of what is added up there, S
    # at most -- the result itself may be small where residuals cancel it -- and the GELU's slope stays below 1.13: 2^-8 S
    a, _, bias = (dev(x) for x in _inputs(M, N, K, M + N))
    wq, scale = _q8(N, K, N + K)
    words, scale = torch.from_numpy(wq.view(np.int32)).cuda(), dev(scale)
    w = torch.empty(N, K, dtype=torch.float16, device="cuda")
    ops.decode_q8(words, scale, w)
    g = torch.Generator(device="cuda").manual_seed(1)
    res = [torch.randn(M, N, device="cuda", generator=g).half() for _ in range(2)] if epilogue in (_lib.EPI_BIAS_ADD2, _lib.EPI_BIAS_ADD2_CAST_F32) else [None, None]
    kind = torch.float32 if epilogue == _lib.EPI_BIAS_ADD2_CAST_F32 else torch.float16
    out, want = Guarded((M, N), kind), torch.empty(M, N, dtype=kind, device="cuda")
    ops.gemm_q8(a, words, scale, bias, out.t, None, epilogue, *res)
    ops.gemm(a, w, bias, want, cfg(variant=_lib.GEMM_MFMA, block=256, vec=8, unroll=2, tile=[64, 64, 64]), epilogue, *res)
    mm = torch.empty(M, N, dtype=torch.float16, device="cuda")
    ops.gemm(a, w, None, mm, cfg(variant=_lib.GEMM_MFMA, block=256, vec=8, unroll=2, tile=[64, 64, 64]))
    S = sum(t.double().abs() for t in (mm, bias.expand(M, N), *(r for r in res if r is not None))).cpu().numpy()
    got, want = out.check().astype(np.float64), want.cpu().numpy().astype(np.float64)
    assert (np.abs(got - want) <= 2.0 ** -8 * S).all()


def _among_nans(t):
    """The same elements in a buffer that holds NaN before and behind them (200 rows of them behind)."""
    flat = torch.full((t.numel() + 200 * t.shape[-1] + 512,), float("nan"), dtype=t.dtype, device="cuda")
    flat[512:512 + t.numel()] = t.reshape(-1)
    return flat[512:512 + t.numel()].view(t.shape)


def _check_non_finite(run, a, N):
    """What lies around the operands reaches no result; NaN and infinities in the last rows of A and W reach their row and
    column and no other element: every other one has the bits it has without them."""
    M = a.shape[0]
    clean = run(_among_nans(a))
    assert np.isfinite(clean.astype(np.float64)).all()
    bad = a.clone()
    bad[M - 1, a.shape[1] - 1] = float("nan")
    bad[0, 0] = float("inf")
    got = run(_among_nans(bad), True)
    assert np.isnan(got[M - 1]).all() and np.isnan(got[:, N - 1]).all() and not np.isfinite(got[0].astype(np.float64)).any()
    assert_bits_equal(got[1:M - 1, :N - 1], clean[1:M - 1, :N - 1])


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn,stages", TILES)
def test_non_finite_operands_at_the_edges_of_every_tile(bm, bn, stages):
    # (K = 200: the last k tile is a chunk of 8 wide, the next row's elements and what lies behind the last row follow it)
    for M, N, K, split in ((bm + 3, bn + 5, 200, 1), (bm - 7, 2 * bn - 3, 1096, 2)):
        a, w, _ = (dev(x) for x in _inputs(M, N, K, M))

        def run(a, poison=False):
            wn = w.clone()
            if poison:
                wn[N - 1, K - 1] = float("nan")
            out = Guarded((M, N), torch.float16)
            ops.gemm(a, _among_nans(wn), None, out.t, _cfg(bm, bn, stages, split))
            return out.check()

        _check_non_finite(run, a, N)


@pytest.mark.gpu
@pytest.mark.parametrize("bm,bn", Q8_TILES)
def test_non_finite_operands_at_the_edges_of_every_8_bit_tile(bm, bn):
    # (tiles of 96 and 160 rows load A in whole 64-row steps: the rows in between are past the tile and must not be read)
    for M, N, K, split in ((bm + 3, bn + 5, 224, 1), (2 * bm - 7, bn - 3, 1120, 2)):
        a = dev(_inputs(M, N, K, M)[0])
        wq, scale = _q8(N, K, M)
        words, scale = torch.from_numpy(wq.view(np.int32)).cuda(), dev(scale)

        def run(a, poison=False):
            sn = scale.clone()
            if poison:
                sn[N - 1, K // 32 - 1] = float("nan")
            out = Guarded((M, N), torch.float16)
            ops.gemm_q8(a, words, _among_nans(sn), None, out.t, _cfg(bm, bn, 0, split))
            return out.check()

        _check_non_finite(run, a, N)


@pytest.mark.gpu
@pytest.mark.parametrize("q8,bm,bn,stages", [(False, *t) for t in TILES] + [(True, bm, bn, 0) for bm, bn in Q8_TILES])
def test_a_part_of_k_without_a_k_tile(oracle, q8, bm, bn, stages):
    # 5 k tiles in 4 parts of 2: the last part has none and adds zeros
    M, N, K = bm + 9, bn + 7, 288
    a, w, bias = _inputs(M, N, K, bm * bn)
    out = Guarded((M, N), torch.float16)
    if q8:
        wq, scale = _q8(N, K, bm)
        w = oracle.c.decode_q8(wq, scale, threads=8)
        ops.gemm_q8(dev(a), torch.from_numpy(wq.view(np.int32)).cuda(), dev(scale), dev(bias), out.t, _cfg(bm, bn, 0, 4))
    else:
        ops.gemm(dev(a), dev(w), dev(bias), out.t, _cfg(bm, bn, stages, 4))
    _check(out.check(), oracle.c.gemm(a, w, bias, threads=8), oracle.np64.gemm(a, w, bias))


def test_every_tile_describes_its_launch_and_nothing_else_is_taken():
    for bm, bn, stages in TILES:
        info = _lib.describe_launch(_lib.OP_GEMM_F16, 1000, 3000, 4096, _lib.DtasConfig.from_dict(
            {"variant": _lib.GEMM_MFMA, "block": 512, "vec": 8, "unroll": 2 if stages == 2 else 0, "tile": [bm, bn, 64], "split_k": 1}))
        assert list(info.launch_args)[:4] == [-(-1000 // bm) * -(-3000 // bn), 1, 1, 512] and info.launch_args[4] <= 160 * 1024
    for bm, bn, block, stages in ((96, 128, 256, 4), (160, 256, 256, 3), (64, 128, 512, 2), (64, 64, 512, 2), (96, 64, 512, 4), (320, 128, 512, 2), (96, 128, 512, 5)):
        with pytest.raises(_lib.DtasError):
            _lib.describe_launch(_lib.OP_GEMM_F16, 1000, 3000, 4096, _lib.DtasConfig.from_dict(
                {"variant": _lib.GEMM_MFMA, "block": block, "vec": 8, "unroll": stages, "tile": [bm, bn, 64], "split_k": 1}))


@pytest.mark.parametrize("seed", range(4))
def test_a_call_without_a_config_names_a_launchable_kernel(seed):
    # partial tiles never outgrow the room that a caller who cannot allocate has, as in the rows before
    rng = np.random.default_rng(seed)
    for _ in range(500):
        M, N, K = int(rng.integers(129, 8192)), int(2 ** rng.uniform(0, 17)), 8 * int(2 ** rng.uniform(0, 11))
        info = _lib.builtin_gemm(M, N, K)
        c = info.config
        assert list(_lib.describe_launch(_lib.OP_GEMM_F16, M, N, K, c).launch_args) == list(info.launch_args), (M, N, K)
        if c.split_k > 1:
            assert info.launch_args[0] * c.tile[0] * c.tile[1] * 4 <= 32 << 20 and -(-K // 64) // c.split_k >= 6, (M, N, K)


@pytest.mark.parametrize("M,N,K", [(1960, 611, 6003008), (1358, 500, 7290176), (1424, 426, 9246144), (2203, 257, 11799328), (70, 200, 16777184)])
def test_an_8_bit_call_without_a_config_names_a_tile_that_holds_its_rows(M, N, K):
    # a tile's rows are addressed with 32-bit offsets: from K = 4.2 million the taller tiles no longer hold them, the 64-row one up to 2^24
    info = _lib.builtin_gemm(M, N, K, q8=True)
    if info.name == b"gemm_q8":     # (otherwise the two passes, whose fp16 tile dtas_builtin_gemm describes by itself)
        _lib.describe_launch(_lib.OP_GEMM_F16, M, N, K, info.config)


def test_a_k_that_no_tile_holds_is_refused():
    for K in (1 << 24, 1 << 25):
        with pytest.raises(_lib.DtasError, match="too large"):
            _lib.builtin_gemm(300, 64, K)


@pytest.mark.gpu
@pytest.mark.parametrize("block", [256, 512])
@pytest.mark.parametrize("M,N", [(1, 32), (129, 64), (300, 288), (300, 280), (257, 10240)])
def test_rows_written_through_and_streamed_hold_the_same_bits(block, M, N):
    """C on and off the 64-byte grid, N % 32 = 0 or not: the stores differ, the results do not."""
    gen = torch.Generator(device="cuda").manual_seed(M * 7 + N)
    A = torch.randn(M, 192, device="cuda", generator=gen).half()
    W = (torch.randn(N, 192, device="cuda", generator=gen) * 0.05).half()
    bias = torch.randn(N, device="cuda", generator=gen).half()
    tile = cfg(variant=_lib.GEMM_MFMA, block=block, vec=8, unroll=2 if block == 256 else 0, tile=[128, 128, 64])
    got = []
    for offset in (0, 8, 32, 1):
        raw = torch.full((M * N + 64 + offset,), 1234.5, dtype=torch.float16, device="cuda")
        C = raw[offset:offset + M * N].view(M, N)
        ops.gemm(A, W, bias, C, cfg=tile)
        torch.cuda.synchronize()
        assert bool((raw[:offset] == 1234.5).all()) and bool((raw[offset + M * N:] == 1234.5).all())
        got.append(C.clone())
    assert all(torch.equal(got[0], g) for g in got[1:])
    # (the sum and the result are each rounded to fp16, 2^-11 of at most a few units)
    want = (A.double() @ W.double().t()).half().double() + bias.double()
    assert ((got[0].double() - want).abs() <= 2e-3 + 2e-3 * want.abs()).all()


@pytest.mark.gpu
@pytest.mark.parametrize("block", [256, 512])
@pytest.mark.parametrize("M,N", [(2457, 10240), (2458, 10240), (786432, 32), (786433, 32)])
def test_c_at_the_line_between_written_through_and_streamed(block, M, N):
    """48 MiB and a row more, on the 64-byte grid (by the size) and off it (streamed): the same bits."""
    assert (M * N * 2 <= 48 << 20) == (M in (2457, 786432))
    gen = torch.Generator(device="cuda").manual_seed(M + N)
    A = torch.randn(M, 64, device="cuda", generator=gen).half()
    W = (torch.randn(N, 64, device="cuda", generator=gen) * 0.05).half()
    tile = cfg(variant=_lib.GEMM_MFMA, block=block, vec=8, unroll=2 if block == 256 else 0, tile=[128, 128, 64])
    got = []
    for offset in (0, 8):
        raw = torch.full((M * N + 64,), 1234.5, dtype=torch.float16, device="cuda")
        ops.gemm(A, W, None, raw[offset:offset + M * N].view(M, N), cfg=tile)
        assert bool((raw[:offset] == 1234.5).all()) and bool((raw[offset + M * N:] == 1234.5).all())
        got.append(raw[offset:offset + M * N].view(M, N))
    assert torch.equal(*got)
    want = A.double() @ W.double().t()
    # (fp32 sums of 64 products of magnitude 1e-1 and one rounding to fp16: 2^-11 of the value)
    assert ((got[0].double() - want).abs() <= 1e-5 + 2 ** -11 * 1.01 * want.abs()).all()
