// The ordinary case of every entry point of dtas_amd.ops, checked and launched natively: tensors in, one library call out.
// A call of three rows of 4096 costs the host 2.9 .. 3.7 us here (copy, RMSNorm; which of the two goes with the core that the
// process got), no more than the launch (the library's entry point through ctypes, pointers at hand: 3.1 .. 3.8), and 5.3 .. 6.4
// us through the checks, pointers and extents in Python; a decode layer of 19 launches is bound by just that (one layer at
// 127 keys 110 -> 72 .. 75 us).
// Each function takes the arguments of the `ops` function of its name (without `cfg`) and returns True after the launch.
// For whatever is not the ordinary case -- another type of object, a tensor that is not a plain contiguous one on the
// device, any check that does not hold, an extent of zero, a torch-function mode -- it does nothing and returns False:
// the Python body behind it then decides and words the error.  A call that the library refuses raises DtasError.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <pthread.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/dtas_abi.h"

namespace {

// the entry points of the library that dtas_amd._lib has loaded (bind()); null: not bound, and every call returns False
#define DTAS_ENTRIES(X)                                                                                                  \
  X(dtas_add_f16) X(dtas_add_f32) X(dtas_add_i8) X(dtas_copy_f16) X(dtas_copy_f32) X(dtas_copy_i8) X(dtas_cast_f16_f32)  \
  X(dtas_cast_f32_f16) X(dtas_layer_norm_f32_f16) X(dtas_layer_norm_f32) X(dtas_rms_norm_f16) X(dtas_softmax_f32_f16)    \
  X(dtas_softmax_f16) X(dtas_gemv_f16) X(dtas_gemv_f16_fused) X(dtas_gemv_f32) X(dtas_gemm_f16) X(dtas_gemm_f16_fused)   \
  X(dtas_attn_scores_f16_f32) X(dtas_attn_pv_f16) X(dtas_decode_q8_f16) X(dtas_attn_mask_f16)                            \
  X(dtas_softmax_temperature_f32) X(dtas_split3_f16) X(dtas_swap_axes_f16) X(dtas_rotary_f16) X(dtas_take_f16)           \
  X(dtas_take_q8_f16) X(dtas_gemv_q8_f32) X(dtas_gemv_q8_f16) X(dtas_gemm_q8_f16_fused) X(dtas_last_error)
#define DTAS_DECLARE(name) decltype(&::name) p_##name = nullptr;
DTAS_ENTRIES(DTAS_DECLARE)
#undef DTAS_DECLARE
PyObject* g_error = nullptr;  // dtas_amd._lib.DtasError
bool g_bound = false;

// An argument: a plain contiguous device tensor.  `ok` turns false, for good, with the first one that is not.
struct Args {
  PyObject* const* at;
  bool ok;
  Args(PyObject* const* args, Py_ssize_t given, Py_ssize_t wanted)
      : at(args), ok(g_bound && given == wanted && !at::impl::torch_function_mode_enabled()) {}

  const at::Tensor* tensor(int i) {
    if (!ok) return nullptr;
    if (!THPVariable_CheckExact(at[i])) return bad();
    const at::Tensor& t = THPVariable_Unpack(at[i]);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() ||
        t.key_set().has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                                 c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize})) ||
        !t.is_contiguous() || t.numel() == 0)
      return bad();
    return &t;
  }
  const at::Tensor* tensor(int i, at::ScalarType type) {
    const at::Tensor* t = tensor(i);
    return t && t->scalar_type() != type ? bad() : t;
  }
  // None: nullptr; a tensor of `type` with `count` elements (a check that fails leaves `ok` false)
  const at::Tensor* optional(int i, at::ScalarType type, int64_t count) {
    if (!ok || at[i] == Py_None) return nullptr;
    const at::Tensor* t = tensor(i, type);
    return t && t->numel() != count ? bad() : t;
  }
  int64_t integer(int i) {
    if (!ok || !PyLong_CheckExact(at[i])) return ok = false, 0;
    int overflow = 0;
    const long long v = PyLong_AsLongLongAndOverflow(at[i], &overflow);
    ok = overflow == 0;
    return v;
  }
  float number(int i) {
    if (!ok || !PyFloat_CheckExact(at[i])) return ok = false, 0.f;
    return static_cast<float>(PyFloat_AS_DOUBLE(at[i]));
  }
  bool require(bool condition) { return ok = ok && condition; }
  const at::Tensor* bad() { return ok = false, nullptr; }
};

void* ptr(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }
int64_t last(const at::Tensor* t) { return t->dim() > 0 ? t->size(-1) : 1; }

constexpr auto F16 = at::kHalf;
constexpr auto F32 = at::kFloat;

// The library call on torch's current stream, without the GIL (a launch waits when the queue is full).
template <class F, class... A>
PyObject* launch(const char* name, F fn, A... args) {
  void* stream = c10::hip::getCurrentHIPStream().stream();
  int rc;
  bool thrown = false;
  Py_BEGIN_ALLOW_THREADS
  try {  // (nothing may leave this block but through its end, which takes the GIL again)
    rc = fn(args..., stream);
  } catch (...) {
    rc = -1;
    thrown = true;
  }
  Py_END_ALLOW_THREADS
  if (rc == 0) Py_RETURN_TRUE;
  PyErr_Format(g_error, "%s: %s", name, thrown ? "a C++ exception left the library" : p_dtas_last_error());
  return nullptr;
}
#define DTAS_CALL(name, ...) launch(#name, p_##name, __VA_ARGS__)
constexpr const dtas_config* kBuiltIn = nullptr;

#define DTAS_FUNCTION(name, wanted, ...)                                              \
  PyObject* name(PyObject*, PyObject* const* argv, Py_ssize_t argc) {                 \
    try {                                                                             \
      Args a(argv, argc, wanted);                                                     \
      __VA_ARGS__                                                                     \
    } catch (...) { /* torch refused something: the Python body meets it again */     \
    }                                                                                 \
    Py_RETURN_FALSE;                                                                  \
  }

DTAS_FUNCTION(add, 3, {
  auto *A = a.tensor(0), *B = a.tensor(1), *out = a.tensor(2);
  if (a.ok && A->scalar_type() == B->scalar_type() && A->scalar_type() == out->scalar_type() && A->sizes() == B->sizes() && A->sizes() == out->sizes()) {
    const int64_t H = last(A), n = A->numel() / H;
    switch (A->scalar_type()) {
      case at::kHalf: return DTAS_CALL(dtas_add_f16, ptr(A), ptr(B), ptr(out), n, H, kBuiltIn);
      case at::kFloat: return DTAS_CALL(dtas_add_f32, ptr(A), ptr(B), ptr(out), n, H, kBuiltIn);
      case at::kChar: return DTAS_CALL(dtas_add_i8, ptr(A), ptr(B), ptr(out), n, H, kBuiltIn);
      default: break;
    }
  }
})

DTAS_FUNCTION(copy, 2, {
  auto *A = a.tensor(0), *B = a.tensor(1);
  if (a.ok && A->scalar_type() == B->scalar_type() && A->sizes() == B->sizes()) {
    const int64_t H = last(A), n = A->numel() / H;
    switch (A->scalar_type()) {
      case at::kHalf: return DTAS_CALL(dtas_copy_f16, ptr(A), ptr(B), n, H, kBuiltIn);
      case at::kFloat: return DTAS_CALL(dtas_copy_f32, ptr(A), ptr(B), n, H, kBuiltIn);
      case at::kChar: return DTAS_CALL(dtas_copy_i8, ptr(A), ptr(B), n, H, kBuiltIn);
      default: break;
    }
  }
})

DTAS_FUNCTION(cast, 2, {
  auto *A = a.tensor(0), *out = a.tensor(1);
  if (a.ok && A->sizes() == out->sizes()) {
    const int64_t H = last(A), n = A->numel() / H;
    if (A->scalar_type() == F16 && out->scalar_type() == F32) return DTAS_CALL(dtas_cast_f16_f32, ptr(A), ptr(out), n, H, kBuiltIn);
    if (A->scalar_type() == F32 && out->scalar_type() == F16) return DTAS_CALL(dtas_cast_f32_f16, ptr(A), ptr(out), n, H, kBuiltIn);
  }
})

DTAS_FUNCTION(layer_norm, 5, {
  auto *x = a.tensor(0, F32), *gamma = a.tensor(1, F32), *beta = a.tensor(2, F32), *out = a.tensor(3, F16);
  const float eps = a.number(4);
  if (a.ok && out->sizes() == x->sizes() && gamma->numel() == last(x) && beta->numel() == last(x))
    return DTAS_CALL(dtas_layer_norm_f32_f16, ptr(x), ptr(gamma), ptr(beta), ptr(out), x->numel() / last(x), last(x), eps, kBuiltIn);
})

DTAS_FUNCTION(layer_norm_f32, 5, {
  auto *x = a.tensor(0, F32), *gamma = a.tensor(1, F32), *beta = a.tensor(2, F32), *out = a.tensor(3, F32);
  const float eps = a.number(4);
  if (a.ok && out->sizes() == x->sizes() && gamma->numel() == last(x) && beta->numel() == last(x))
    return DTAS_CALL(dtas_layer_norm_f32, ptr(x), ptr(gamma), ptr(beta), ptr(out), x->numel() / last(x), last(x), eps);
})

DTAS_FUNCTION(rms_norm, 4, {
  auto *x = a.tensor(0, F16), *w = a.tensor(1, F16), *out = a.tensor(2, F16);
  const float eps = a.number(3);
  if (a.ok && out->sizes() == x->sizes() && w->numel() == last(x))
    return DTAS_CALL(dtas_rms_norm_f16, ptr(x), ptr(w), ptr(out), x->numel() / last(x), last(x), eps, kBuiltIn);
})

DTAS_FUNCTION(softmax, 2, {
  auto *A = a.tensor(0), *out = a.tensor(1, F16);
  if (a.ok && out->sizes() == A->sizes()) {
    const int64_t cols = last(A), rows = A->numel() / cols;
    if (A->scalar_type() == F32) return DTAS_CALL(dtas_softmax_f32_f16, ptr(A), ptr(out), rows, cols, kBuiltIn);
    if (A->scalar_type() == F16) return DTAS_CALL(dtas_softmax_f16, ptr(A), ptr(out), rows, cols, kBuiltIn);
  }
})

// x, W, bias, y, epilogue, res1, res2
DTAS_FUNCTION(gemv, 7, {
  const int64_t epilogue = a.integer(4);
  auto *x = a.tensor(0, F16), *W = a.tensor(1, F16), *y = a.tensor(3, epilogue == DTAS_EPI_BIAS_ADD2_CAST_F32 ? F32 : F16);
  if (a.ok && W->dim() == 2) {
    const int64_t N = W->size(0), K = W->size(1);
    auto *bias = a.optional(2, F16, N), *res1 = a.optional(5, F16, N), *res2 = a.optional(6, F16, N);
    if (a.require(x->numel() == K && y->numel() == N && epilogue == static_cast<int32_t>(epilogue))) {
      if (epilogue == DTAS_EPI_BIAS && !res1 && !res2) return DTAS_CALL(dtas_gemv_f16, ptr(x), ptr(W), ptr(bias), ptr(y), N, K, kBuiltIn);
      return DTAS_CALL(dtas_gemv_f16_fused, ptr(x), ptr(W), ptr(bias), ptr(res1), ptr(res2), ptr(y), N, K, static_cast<int32_t>(epilogue), kBuiltIn);
    }
  }
})

DTAS_FUNCTION(gemv_f32, 3, {
  auto *x = a.tensor(0, F32), *W = a.tensor(1, F32), *y = a.tensor(2, F32);
  if (a.ok && W->dim() == 2 && x->numel() == W->size(1) && y->numel() == W->size(0))
    return DTAS_CALL(dtas_gemv_f32, ptr(x), ptr(W), ptr(y), W->size(0), W->size(1), kBuiltIn);
})

// A, W, bias, C, epilogue, res1, res2
DTAS_FUNCTION(gemm, 7, {
  const int64_t epilogue = a.integer(4);
  auto *A = a.tensor(0, F16), *W = a.tensor(1, F16), *C = a.tensor(3, epilogue == DTAS_EPI_BIAS_ADD2_CAST_F32 ? F32 : F16);
  if (a.ok && W->dim() == 2 && A->dim() > 0 && C->dim() > 0) {
    const int64_t N = W->size(0), K = W->size(1), M = A->numel() / K;
    auto *bias = a.optional(2, F16, N), *res1 = a.optional(5, F16, M * N), *res2 = a.optional(6, F16, M * N);
    if (a.require(A->size(-1) == K && C->size(-1) == N && C->numel() == M * N && epilogue == static_cast<int32_t>(epilogue))) {
      if (epilogue == DTAS_EPI_BIAS && !res1 && !res2) return DTAS_CALL(dtas_gemm_f16, ptr(A), ptr(W), ptr(bias), ptr(C), M, N, K, kBuiltIn);
      return DTAS_CALL(dtas_gemm_f16_fused, ptr(A), ptr(W), ptr(bias), ptr(res1), ptr(res2), ptr(C), M, N, K, static_cast<int32_t>(epilogue), kBuiltIn);
    }
  }
})

DTAS_FUNCTION(attn_scores, 5, {
  auto *Q = a.tensor(0, F16), *K = a.tensor(1, F16), *mask = a.tensor(2, F16), *out = a.tensor(3, F32);
  const float scale = a.number(4);
  if (a.ok && Q->dim() >= 3 && K->dim() >= 3 && mask->dim() >= 2 && out->dim() >= 3) {
    const int64_t heads = Q->size(-3), n = Q->size(-2), d = Q->size(-1), m = K->size(-2);
    if (K->size(-3) == heads && K->size(-1) == d && mask->size(-2) == n && mask->size(-1) == m && out->size(-3) == heads && out->size(-2) == n &&
        out->size(-1) == m && Q->numel() == heads * n * d && K->numel() == heads * m * d && mask->numel() == n * m && out->numel() == heads * n * m)
      return DTAS_CALL(dtas_attn_scores_f16_f32, ptr(Q), ptr(K), ptr(mask), ptr(out), heads, n, m, d, scale, kBuiltIn);
  }
})

DTAS_FUNCTION(attn_pv, 3, {
  auto *P = a.tensor(0, F16), *V = a.tensor(1, F16), *out = a.tensor(2, F16);
  if (a.ok && P->dim() >= 3 && V->dim() >= 3 && out->dim() >= 3) {
    const int64_t heads = P->size(-3), n = P->size(-2), m = P->size(-1), d = V->size(-1);
    if (V->size(-3) == heads && V->size(-2) == m && out->size(-3) == heads && out->size(-2) == n && out->size(-1) == d &&
        P->numel() == heads * n * m && V->numel() == heads * m * d && out->numel() == heads * n * d)
      return DTAS_CALL(dtas_attn_pv_f16, ptr(P), ptr(V), ptr(out), heads, n, m, d, kBuiltIn);
  }
})

// 8-bit weights: 32-bit words [N, K/4] and scales [N, K/32]
bool q8_shape(const at::Tensor* Wq, const at::Tensor* scale, int64_t* N, int64_t* K) {
  if (Wq->dim() != 2 || scale->dim() != 2 || (Wq->scalar_type() != at::kInt && Wq->scalar_type() != at::kUInt32)) return false;
  *N = Wq->size(0);
  *K = Wq->size(1) * 4;
  return *K % 32 == 0 && scale->size(0) == *N && scale->size(1) == *K / 32;
}

DTAS_FUNCTION(decode_q8, 3, {
  auto *Wq = a.tensor(0), *scale = a.tensor(1, F16), *W = a.tensor(2, F16);
  int64_t N, K;
  if (a.ok && q8_shape(Wq, scale, &N, &K) && W->numel() == N * K) return DTAS_CALL(dtas_decode_q8_f16, ptr(Wq), ptr(scale), ptr(W), N, K, kBuiltIn);
})

DTAS_FUNCTION(attn_mask, 1, {
  auto* out = a.tensor(0, F16);
  if (a.ok && out->dim() >= 2 && out->numel() == out->size(-2) * out->size(-1)) return DTAS_CALL(dtas_attn_mask_f16, ptr(out), out->size(-2), out->size(-1));
})

DTAS_FUNCTION(softmax_temperature, 3, {
  auto *logits = a.tensor(0, F32), *temperature = a.tensor(1, F32), *out = a.tensor(2, F32);
  if (a.ok && out->sizes() == logits->sizes() && temperature->numel() == 1)
    return DTAS_CALL(dtas_softmax_temperature_f32, ptr(logits), ptr(temperature), ptr(out), logits->numel() / last(logits), last(logits));
})

DTAS_FUNCTION(split3, 4, {
  auto *A = a.tensor(0, F16), *out0 = a.tensor(1, F16), *out1 = a.tensor(2, F16), *out2 = a.tensor(3, F16);
  if (a.ok && A->dim() > 0 && A->size(-1) % 3 == 0) {
    const int64_t d = A->size(-1) / 3, rows = A->numel() / A->size(-1);
    for (auto* o : {out0, out1, out2}) a.require(o->dim() > 0 && o->size(-1) == d && o->numel() == rows * d);
    if (a.ok) return DTAS_CALL(dtas_split3_f16, ptr(A), ptr(out0), ptr(out1), ptr(out2), rows, d);
  }
})

DTAS_FUNCTION(swap_axes, 2, {
  auto *A = a.tensor(0, F16), *out = a.tensor(1, F16);
  if (a.ok && A->dim() >= 3 && out->dim() >= 3) {
    const int64_t n0 = A->size(-3), n1 = A->size(-2), d = A->size(-1);
    if (A->numel() == n0 * n1 * d && out->size(-3) == n1 && out->size(-2) == n0 && out->size(-1) == d && out->numel() == n0 * n1 * d)
      return DTAS_CALL(dtas_swap_axes_f16, ptr(A), ptr(out), n0, n1, d);
  }
})

DTAS_FUNCTION(rotary, 5, {
  auto *A = a.tensor(0, F16), *cos = a.tensor(1, F16), *sin = a.tensor(2, F16), *out = a.tensor(3, F16);
  const int64_t m = a.integer(4);
  if (a.ok && cos->dim() == 2 && cos->sizes() == sin->sizes() && A->dim() >= 3 && out->sizes() == A->sizes()) {
    const int64_t n = A->size(-3), heads = A->size(-2), d = A->size(-1);
    if (A->numel() == n * heads * d)
      return DTAS_CALL(dtas_rotary_f16, ptr(A), ptr(cos), ptr(sin), ptr(out), n, m, heads, d, cos->size(1), cos->size(0), kBuiltIn);
  }
})

DTAS_FUNCTION(take, 3, {
  auto *A = a.tensor(0, F16), *ids = a.tensor(1, at::kInt), *out = a.tensor(2, F16);
  if (a.ok && A->dim() == 2 && out->numel() == ids->numel() * A->size(1))
    return DTAS_CALL(dtas_take_f16, ptr(A), ptr(ids), ptr(out), ids->numel(), A->size(0), A->size(1), kBuiltIn);
})

DTAS_FUNCTION(take_q8, 4, {
  auto *Wq = a.tensor(0), *scale = a.tensor(1, F16), *ids = a.tensor(2, at::kInt), *out = a.tensor(3, F16);
  int64_t V, K;
  if (a.ok && q8_shape(Wq, scale, &V, &K) && out->numel() == ids->numel() * K)
    return DTAS_CALL(dtas_take_q8_f16, ptr(Wq), ptr(scale), ptr(ids), ptr(out), ids->numel(), V, K, kBuiltIn);
})

DTAS_FUNCTION(gemv_q8_f32, 4, {
  auto *x = a.tensor(0, F32), *Wq = a.tensor(1), *scale = a.tensor(2, F32), *y = a.tensor(3, F32);
  int64_t N, K;
  if (a.ok && q8_shape(Wq, scale, &N, &K) && x->numel() == K && y->numel() == N)
    return DTAS_CALL(dtas_gemv_q8_f32, ptr(x), ptr(Wq), ptr(scale), ptr(y), N, K, kBuiltIn);
})

// x, Wq, scale, bias, y, epilogue
DTAS_FUNCTION(gemv_q8, 6, {
  auto *x = a.tensor(0, F16), *Wq = a.tensor(1), *scale = a.tensor(2, F16), *y = a.tensor(4, F16);
  const int64_t epilogue = a.integer(5);
  int64_t N, K;
  if (a.ok && q8_shape(Wq, scale, &N, &K)) {
    auto* bias = a.optional(3, F16, N);
    if (a.require(x->numel() == K && y->numel() == N && epilogue == static_cast<int32_t>(epilogue)))
      return DTAS_CALL(dtas_gemv_q8_f16, ptr(x), ptr(Wq), ptr(scale), ptr(bias), ptr(y), N, K, static_cast<int32_t>(epilogue), kBuiltIn);
  }
})

// A, Wq, scale, bias, C, epilogue, res1, res2
DTAS_FUNCTION(gemm_q8, 8, {
  const int64_t epilogue = a.integer(5);
  auto *A = a.tensor(0, F16), *Wq = a.tensor(1), *scale = a.tensor(2, F16), *C = a.tensor(4, epilogue == DTAS_EPI_BIAS_ADD2_CAST_F32 ? F32 : F16);
  int64_t N, K;
  if (a.ok && q8_shape(Wq, scale, &N, &K) && A->dim() > 0 && C->dim() > 0) {
    const int64_t M = A->numel() / K;
    auto *bias = a.optional(3, F16, N), *res1 = a.optional(6, F16, M * N), *res2 = a.optional(7, F16, M * N);
    if (a.require(A->size(-1) == K && C->size(-1) == N && C->numel() == M * N && epilogue == static_cast<int32_t>(epilogue)))
      return DTAS_CALL(dtas_gemm_q8_f16_fused, ptr(A), ptr(Wq), ptr(scale), ptr(bias), ptr(res1), ptr(res2), ptr(C), M, N, K,
                       static_cast<int32_t>(epilogue), kBuiltIn);
  }
})

// bind({entry point: address}, DtasError)
PyObject* bind(PyObject*, PyObject* args) {
  PyObject *addresses, *error;
  if (!PyArg_ParseTuple(args, "O!O", &PyDict_Type, &addresses, &error)) return nullptr;
#define DTAS_BIND(name)                                                                                       \
  {                                                                                                           \
    PyObject* v = PyDict_GetItemString(addresses, #name);                                                     \
    void* p = v ? PyLong_AsVoidPtr(v) : nullptr;                                                              \
    if (!p) return PyErr_Occurred() ? nullptr : PyErr_Format(PyExc_KeyError, "no address for %s", #name);     \
    p_##name = reinterpret_cast<decltype(p_##name)>(p);                                                       \
  }
  DTAS_ENTRIES(DTAS_BIND)
#undef DTAS_BIND
  Py_INCREF(error);
  Py_XDECREF(g_error);
  g_error = error;
  g_bound = true;
  Py_RETURN_NONE;
}

#define DTAS_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {DTAS_METHOD(add), DTAS_METHOD(copy), DTAS_METHOD(cast), DTAS_METHOD(layer_norm), DTAS_METHOD(layer_norm_f32),
                         DTAS_METHOD(rms_norm), DTAS_METHOD(softmax), DTAS_METHOD(gemv), DTAS_METHOD(gemv_f32), DTAS_METHOD(gemm),
                         DTAS_METHOD(attn_scores), DTAS_METHOD(attn_pv), DTAS_METHOD(decode_q8), DTAS_METHOD(attn_mask),
                         DTAS_METHOD(softmax_temperature), DTAS_METHOD(split3), DTAS_METHOD(swap_axes), DTAS_METHOD(rotary),
                         DTAS_METHOD(take), DTAS_METHOD(take_q8), DTAS_METHOD(gemv_q8_f32), DTAS_METHOD(gemv_q8), DTAS_METHOD(gemm_q8),
                         {"bind", bind, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fastcall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fastcall() {
  // a forked child has no GPU: torch's own check, behind the Python body, says so
  pthread_atfork(nullptr, nullptr, [] { g_bound = false; });
  PyObject* m = PyModule_Create(&module);
  // the torch whose headers this was compiled against: dtas_amd.ops uses it with no other (tensors are read in place)
  if (m && PyModule_AddStringConstant(m, "_built_for", DTAS_BUILT_FOR) != 0) Py_CLEAR(m);
  return m;
}
