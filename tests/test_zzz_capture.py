"""Calls that use the library's workspaces on streams that are being captured, the first call of a stream among them.  A process
holds 16 sets of workspaces, which these tests use up: last in the order, behind the test that watches the free memory."""
import ctypes

import pytest
import torch

from dtas_amd import _lib, ops
from gpu_util import assert_bits_equal, cfg

pytestmark = pytest.mark.gpu


def new_stream():
    """A stream that no workspace belongs to: torch's own come from a pool, where an earlier test may have had this one."""
    handle = ctypes.c_void_p()
    assert _lib.lib().hipStreamCreateWithFlags(ctypes.byref(handle), 1) == 0   # (found in the runtime that the library is linked to; 1: non-blocking)
    return torch.cuda.ExternalStream(handle.value)


def replays_of(stream, launch, out, replays=3):
    """What three replays of a graph recorded on `stream` leave in `out`, an eager launch on another stream in between."""
    graph, got = torch.cuda.CUDAGraph(), []
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        launch()
    for _ in range(replays):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        got.append(out.cpu().numpy())
        launch()
    return got


def _problem(M, N, K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(M, K, device="cuda", generator=g).half(), (torch.randn(N, K, device="cuda", generator=g) * 0.02).half(),
            (torch.rand(N, device="cuda", generator=g) * 2 - 1).half())


def _pv_problem(heads, n, m, d, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return torch.softmax(torch.randn(heads, n, m, device="cuda", generator=g), -1).half(), torch.randn(heads, m, d, device="cuda", generator=g).half()


def _tile8(bm, bn, stages, split):
    return cfg(variant=_lib.GEMM_MFMA, block=512, unroll=stages, tile=[bm, bn, 64], split_k=split)


def _last_round_split(N, K):
    """The most rows up to 6000 whose call without a config splits only the last round of 256x256 tiles (split_k 0), over
    more partial tiles than the 32 MiB that the first launch of a stream allocates."""
    for M in range(6000, 1000, -1):
        info = _lib.builtin_gemm(M, N, K)
        tiles = -(-M // 256) * -(-N // 256)
        if info.config.split_k == 0 and (info.launch_args[0] - tiles + tiles % 256) * 256 * 256 * 4 > 32 << 20 and info.launch_args[0] > tiles:
            return M
    raise AssertionError("no size splits its last round")


@pytest.mark.parametrize("rows,room", [("few", "none"), ("some", "none"), ("last round", "none"), ("last round", "too small")])
def test_a_first_call_under_capture_gives_the_eager_bits(rows, room):
    # with K in parts, on a stream that has no workspace, or one that has to grow, while it is being captured
    N, K = (4096, 11008) if rows == "last round" else (2560, 10240)
    M = {"few": 100, "some": 200, "last round": _last_round_split(N, K)}[rows]
    c = _lib.builtin_gemm(M, N, K).config
    assert c.split_k > 1 or rows == "last round"
    a, w, _ = _problem(M, N, K, 1)
    out, eager = (torch.zeros(M, N, dtype=torch.float16, device="cuda") for _ in range(2))
    ops.gemm(a, w, None, eager)
    stream = new_stream()
    if room == "too small":
        torch.cuda.synchronize()
        with torch.cuda.stream(stream):
            ops.gemm(a[:200], w, None, out[:200], _tile8(128, 64, 0, 2))
    for got in replays_of(stream, lambda: ops.gemm(a, w, None, out), out):
        assert_bits_equal(got, eager.cpu().numpy())


@pytest.mark.parametrize("M", [203, 1900])
def test_a_first_8_bit_call_under_capture_gives_the_eager_bits(M):
    # tiles with K in parts, and the dequantiser into the stream's buffer
    N, K = 2560, 10240
    info = _lib.builtin_gemm(M, N, K, q8=True)
    assert info.name == (b"decode_q8 + gemm" if M == 1900 else b"gemm_q8")
    a, _, bias = _problem(M, N, K, 2)
    g = torch.Generator(device="cuda").manual_seed(3)
    words = torch.randint(-2 ** 31, 2 ** 31 - 1, (N, K // 4), device="cuda", generator=g, dtype=torch.int32)
    scale = (torch.rand(N, K // 32, device="cuda", generator=g) * 0.0008 + 0.0002).half()
    out, eager = (torch.zeros(M, N, dtype=torch.float16, device="cuda") for _ in range(2))
    ops.gemm_q8(a, words, scale, bias, eager)
    for got in replays_of(new_stream(), lambda: ops.gemm_q8(a, words, scale, bias, out), out):
        assert_bits_equal(got, eager.cpu().numpy())


def test_a_first_call_under_capture_on_more_streams_than_hold_a_workspace():
    # the seventeenth releases the set used longest ago, while a stream is being captured
    M, N, K = 200, 2560, 10240
    a, w, _ = _problem(M, N, K, 1)
    out, eager = (torch.zeros(M, N, dtype=torch.float16, device="cuda") for _ in range(2))
    ops.gemm(a, w, None, eager)
    for _ in range(20):
        for got in replays_of(new_stream(), lambda: ops.gemm(a, w, None, out), out, replays=1):
            assert_bits_equal(got, eager.cpu().numpy())


def test_a_graph_outlives_the_growth_of_its_workspace():
    # the recorded launch keeps the partial tiles it was given when a later one on the stream needs more room
    M, N, K = 200, 2560, 10240
    a, w, _ = _problem(2048, N, K, 1)
    out, eager = (torch.zeros(M, N, dtype=torch.float16, device="cuda") for _ in range(2))
    big = torch.zeros(2048, N, dtype=torch.float16, device="cuda")
    ops.gemm(a[:M], w, None, eager)
    stream, graph = new_stream(), torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        ops.gemm(a[:M], w, None, out)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        ops.gemm(a[:M], w, None, out)
    with torch.cuda.stream(stream):
        ops.gemm(a, w, None, big, _tile8(256, 256, 2, 3))     # 80 tiles in three parts: 60 MiB
    torch.cuda.synchronize()
    taken = [torch.full((4 << 20,), 7.0, device="cuda") for _ in range(8)]   # whatever memory was given back has another owner
    for _ in range(3):
        out.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert_bits_equal(out.cpu().numpy(), eager.cpu().numpy())
        assert all(bool((t == 7.0).all()) for t in taken)
        ops.gemm(a[:M], w, None, eager)


@pytest.mark.parametrize("heads,n,m,d", [(32, 1, 2304, 80), (32, 1, 2400, 80), (32, 1, 3001, 80), (32, 2, 2500, 80), (32, 1, 4096, 80), (40, 1, 3500, 80), (16, 4, 3072, 64), (32, 100, 4096, 80)])
def test_pv_whose_keys_are_shared_gives_the_same_bits_from_a_graph(heads, n, m, d):
    # the parts of the keys meet in the stream's workspace, also when the stream is captured before it has one
    p, v = _pv_problem(heads, n, m, d, heads + m)
    eager, out = (torch.zeros(heads, n, d, dtype=torch.float16, device="cuda") for _ in range(2))
    ops.attn_pv(p, v, eager)
    for got in replays_of(new_stream(), lambda: ops.attn_pv(p, v, out), out):
        assert_bits_equal(got, eager.cpu().numpy())
