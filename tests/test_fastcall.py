"""The natively checked call (csrc/fastcall.cpp) and the Python body behind it are one function: what the first accepts
gives the same bits as the second, and what the second refuses the first leaves to it."""
import ctypes
import os
import subprocess
import sys

import pytest
import torch

from dtas_amd import _fastcall, _lib, ops

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_cpu_tensors_are_refused_by_the_body():
    a = torch.zeros(2, 8, dtype=torch.float16)
    ops.lib()
    assert _fastcall.add(a, a, a) is False
    with pytest.raises(ValueError, match="no CPU path"):
        ops.add(a, a, a)


def test_nothing_is_accepted_before_the_library_is_bound():
    code = "import torch; from dtas_amd import _fastcall as f; assert f.add(1, 2, 3) is False and f.attn_mask() is False; print('ok')"
    assert subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True).stdout.strip() == "ok"


@pytest.mark.parametrize("there", ["None", "types.ModuleType('dtas_amd._fastcall')",
                                   "types.SimpleNamespace(_built_for='1.0 other', add=lambda *a: 1 / 0, bind=lambda *a: 1 / 0)"])
def test_missing_or_built_for_another_torch_the_bodies_serve_every_call(there):
    code = f"""
import sys, types, warnings
import torch
sys.modules["dtas_amd._fastcall"] = {there}
with warnings.catch_warnings(record=True) as w:
    warnings.simplefilter("always")
    from dtas_amd import ops
assert [x.category for x in w if "_fastcall" in str(x.message)] == [RuntimeWarning], w
ops.lib()
a = torch.zeros(2, 8, dtype=torch.float16)
try:
    ops.add(a, a, a)
except ValueError as e:
    print(e)
"""
    done = subprocess.run([sys.executable, "-c", code], cwd=ROOT, capture_output=True, text=True)
    assert "no CPU path" in done.stdout, done.stderr


def test_built_for_this_torch():
    assert ops._fastcall is _fastcall and _fastcall._built_for == f"{torch.__version__} {torch.version.git_version}"


def _calls():
    """(name, positional arguments, index of each output) over forms that the bodies accept."""
    g = torch.Generator(device="cuda").manual_seed(3)
    h = lambda *s: torch.randn(*s, device="cuda", generator=g).half()
    f = lambda *s: torch.randn(*s, device="cuda", generator=g)
    i8 = lambda *s: torch.randint(-128, 128, s, device="cuda", generator=g, dtype=torch.int8)
    words = lambda N, K: torch.randint(0, 255, (N, K), device="cuda", generator=g, dtype=torch.uint8).view(torch.int32)
    scales = lambda N, K: (torch.rand(N, K // 32, device="cuda", generator=g) * 0.01).half()
    z = lambda *s, dtype=torch.float16: torch.zeros(*s, device="cuda", dtype=dtype)
    ids = torch.tensor([3, 0, 99], device="cuda", dtype=torch.int32)
    flat = h(1025)[1:].view(4, 256)  # off every vector width
    yield "add", [h(3, 5, 7), h(3, 5, 7), z(3, 5, 7)], [2]
    yield "add", [h(1).reshape(()), h(1).reshape(()), z(1).reshape(())], [2]
    yield "add", [i8(4, 33), i8(4, 33), z(4, 33, dtype=torch.int8)], [2]
    yield "copy", [flat, z(4, 256)], [1]
    yield "cast", [f(2, 3, 8), z(2, 3, 8)], [1]
    yield "cast", [flat, z(4, 256, dtype=torch.float32)], [1]
    yield "layer_norm", [f(1, 5, 320), f(320), f(1, 320), z(1, 5, 320)], [3]
    yield "layer_norm_f32", [f(5, 320), f(320), f(320), z(5, 320, dtype=torch.float32)], [3]
    yield "rms_norm", [h(5, 264), h(264), z(5, 264)], [2]
    yield "softmax", [f(2, 3, 40), z(2, 3, 40)], [1]
    yield "softmax", [h(7, 33), z(7, 33)], [1]
    yield "gemv", [h(1, 1, 256), h(48, 256), h(48), z(1, 48)], [3]
    yield "gemv", [h(256), h(48, 256), None, z(48), None, _lib.EPI_BIAS_GELU], [3]
    yield "gemv", [h(256), h(48, 256), h(48), z(48, dtype=torch.float32), None, _lib.EPI_BIAS_ADD2_CAST_F32, h(48), h(1, 48)], [3]
    yield "gemv_f32", [f(256), f(48, 256), z(48, dtype=torch.float32)], [2]
    yield "gemm", [h(1, 5, 256), h(48, 256), None, z(1, 5, 48)], [3]
    yield "gemm", [h(5, 256), h(48, 256), h(48), z(5, 48), None, _lib.EPI_BIAS_ADD2, h(5, 48), h(1, 5, 48)], [3]
    yield "attn_scores", [h(2, 3, 16), h(1, 2, 9, 16), h(1, 1, 3, 9), z(2, 3, 9, dtype=torch.float32), 0.25], [3]
    yield "attn_pv", [h(2, 3, 16), h(2, 16, 24), z(1, 2, 3, 24)], [2]
    yield "decode_q8", [words(6, 64), scales(6, 64), z(6, 64)], [2]
    yield "attn_mask", [z(1, 1, 5, 9)], [0]
    yield "softmax_temperature", [f(2, 50), f(1).abs() + 0.5, z(2, 50, dtype=torch.float32)], [2]
    yield "split3", [h(5, 4, 48), z(5, 4, 16), z(5, 64).view(5, 4, 16), z(20, 16)], [1, 2, 3]
    yield "swap_axes", [h(1, 5, 3, 16), z(3, 5, 16)], [1]
    yield "rotary", [h(1, 3, 2, 16), f(8, 4).cos().half(), f(8, 4).sin().half(), z(1, 3, 2, 16), 7], [3]
    yield "take", [h(100, 64), ids, z(3, 64)], [2]
    yield "take_q8", [words(100, 64), scales(100, 64), ids, z(1, 3, 64)], [3]
    yield "gemv_q8_f32", [f(64), words(6, 64).view(torch.uint32), scales(6, 64).float(), z(6, dtype=torch.float32)], [3]
    yield "gemv_q8", [h(64), words(6, 64), scales(6, 64), h(6), z(6)], [4]
    yield "gemm_q8", [h(5, 256), words(48, 256), scales(48, 256), h(48), z(5, 48), None, _lib.EPI_BIAS_GELU], [4]


class _Subclass(torch.Tensor):
    """An object that only the Python body takes."""


@pytest.mark.gpu
def test_same_results_as_the_body(monkeypatch):
    ops.lib()
    names = [n for n in dir(_fastcall) if not n.startswith("_") and n != "bind"]
    seen = set()
    for name, args, outs in _calls():
        print(name, [tuple(a.shape) if isinstance(a, torch.Tensor) else a for a in args], flush=True)
        took = []
        fast = getattr(_fastcall, name)
        with monkeypatch.context() as m:
            m.setattr(ops._fastcall, name, lambda *a: took.append(fast(*a)) or took[-1])
            getattr(ops, name)(*args)
        got = [args[i].clone() for i in outs]
        for i in outs:
            args[i].zero_()
        slow = [a.as_subclass(_Subclass) if isinstance(a, torch.Tensor) else a for a in args]
        with monkeypatch.context() as m:
            m.setattr(ops._fastcall, name, lambda *a: took.append(fast(*a)) or took[-1])
            getattr(ops, name)(*slow)
        assert took == [True, False], name   # (the second time the body computed it)
        for i, g in zip(outs, got):
            assert g.count_nonzero() > 0 and torch.equal(args[i].contiguous().view(torch.uint8) if args[i].dim() else args[i], g.view(torch.uint8) if g.dim() else g), name
        seen.add(name)
    assert seen == set(names)


@pytest.mark.gpu
def test_refusals_stay_the_bodys():
    ops.lib()
    h = lambda *s: torch.zeros(*s, device="cuda", dtype=torch.float16)
    with pytest.raises(ValueError, match="compact row-major"):
        ops.copy(h(8, 6).t(), h(6, 8))
    with pytest.raises(ValueError, match="agree in dtype and shape"):
        ops.add(h(2, 8), h(2, 8), h(16))
    with pytest.raises(ValueError, match="shape mismatch"):
        ops.gemm(h(4, 64), h(32, 64), h(31), h(4, 32))
    with pytest.raises(ValueError, match="shape mismatch"):
        ops.attn_scores(h(2, 3, 16), h(2, 9, 16), h(9, 3), torch.zeros(2, 3, 9, device="cuda"))
    with pytest.raises(_lib.DtasError, match="gemv"):
        ops.gemv(h(64), h(32, 64), h(32), h(32), epilogue=9)
    ops.copy(h(0, 8), h(0, 8))  # empty: no launch, no error


@pytest.mark.gpu
def test_an_exception_of_the_library_comes_back_with_the_gil(tmp_path):
    ops.lib()
    (tmp_path / "throws.cpp").write_text('extern "C" int throws(const void*, void*, long, long, const void*, void*) { throw 1; }')
    subprocess.run(["g++", "-shared", "-fPIC", "-o", str(tmp_path / "throws.so"), str(tmp_path / "throws.cpp")], check=True)
    throws = ctypes.CDLL(str(tmp_path / "throws.so")).throws
    a = torch.ones(4, 8, device="cuda", dtype=torch.float16)
    addresses = _lib.entry_addresses()
    try:
        _fastcall.bind({**addresses, "dtas_copy_f16": ctypes.cast(throws, ctypes.c_void_p).value}, _lib.DtasError)
        for _ in range(3):
            with pytest.raises(_lib.DtasError, match="dtas_copy_f16: a C\\+\\+ exception"):
                ops.copy(a, a.clone())
    finally:
        _fastcall.bind(addresses, _lib.DtasError)
    b = torch.zeros_like(a)
    ops.copy(a, b)
    assert torch.equal(a, b)
