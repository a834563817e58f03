"""Calls that use the library's workspaces on streams that are being captured.  A process
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


def _problem(M, N, K, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    return (torch.randn(M, K, device="cuda", generator=g).half(), (torch.randn(N, K, device="cuda", generator=g) * 0.02).half(),
            (torch.rand(N, device="cuda", generator=g) * 2 - 1).half())


def _tile8(bm, bn, stages, split):
    return cfg(variant=_lib.GEMM_MFMA, block=512, unroll=stages, tile=[bm, bn, 64], split_k=split)


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
