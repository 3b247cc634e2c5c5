// Native side of the per-call wrappers of _lib.py: argument checks, output and workspace allocation (torch's caching
// allocator) and the foreign call of the entry points that a quantized linear's forward and backward go through.
//
// A small call is bound by the host: a tensor allocated from Python costs 1.6 us, a ctypes call with 20 arguments 4 us,
// the checks of one operand 1 us, and a training pass through one linear makes 16 allocations and 5 calls.  Here they
// cost 0.6 us, nothing measurable and 0.1 us.
//
// Every function returns its tensors; None when an argument is not what the kernels take, or its device has not been
// checked yet (the Python wrapper then runs the full checks, which name the argument, and calls again); or the entry
// point's status as an int when it refuses the call.  Nothing is kept between calls but the entry points' addresses
// and which devices are gfx950.  The GIL is released around the foreign calls.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>

#include "../../include/k2q.h"

namespace {

// Entry points of libk2q.so, bound by _lib.load().
struct Api {
  decltype(&k2q_linear_fwd) linear_fwd;
  decltype(&k2q_linear_fwd_ws_bytes) linear_fwd_ws_bytes;
  decltype(&k2q_linear_fwd_fuses_down) linear_fwd_fuses_down;
  decltype(&k2q_lora_grads) lora_grads;
  decltype(&k2q_lora_grads_ws_bytes) lora_grads_ws_bytes;
  decltype(&k2q_lora_down) lora_down;
  decltype(&k2q_lora_down_ws_bytes) lora_down_ws_bytes;
  decltype(&k2q_pad_factors) pad_factors;
  decltype(&k2q_dx_prep_eff) dx_prep_eff;
  decltype(&k2q_gemm_dx_lin) gemm_dx_lin;
  decltype(&k2q_dequant_fp8) dequant_fp8;
  decltype(&k2q_gemm_bf16) gemm_bf16;
  decltype(&k2q_gemm_plan_ws_bytes) gemm_plan_ws_bytes;
} api{};

PyObject* raw_stream_of = nullptr;   // torch._C._cuda_getCurrentRawStream
constexpr int MAX_DEVICES = 64;
bool device_ok[MAX_DEVICES] = {};

using at::Tensor;

// The argument as a tensor, or null for None; `bad` is set for anything else.
const Tensor* tensor_of(PyObject* o, bool& bad) {
  if (o == Py_None) return nullptr;
  if (!THPVariable_Check(o)) {
    bad = true;
    return nullptr;
  }
  return &THPVariable_Unpack(o);
}

bool aligned(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// A contiguous, 16-byte aligned operand of this type and shape rank on device d.
bool operand(const Tensor* t, at::ScalarType ty, int64_t ndim, c10::Device d) {
  return t && t->scalar_type() == ty && t->dim() == ndim && t->is_contiguous() && t->device() == d && aligned(*t);
}

bool ready(c10::Device d) { return d.is_cuda() && d.index() >= 0 && d.index() < MAX_DEVICES && device_ok[d.index()]; }

Tensor alloc(at::IntArrayRef shape, at::ScalarType ty, c10::Device d) {
  return at::empty(shape, at::TensorOptions().dtype(ty).device(d));
}

Tensor workspace(int64_t bytes, c10::Device d) { return bytes > 0 ? alloc({bytes}, at::kByte, d) : Tensor(); }

void* ptr(const Tensor* t) { return t ? t->data_ptr() : nullptr; }
void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
template <class T>
T* as(void* p) { return static_cast<T*>(p); }

bool stream_of(c10::Device d, void*& st) {
  PyObject* i = PyLong_FromLong(d.index());
  PyObject* r = i ? PyObject_CallOneArg(raw_stream_of, i) : nullptr;
  Py_XDECREF(i);
  if (!r) return false;
  st = PyLong_AsVoidPtr(r);
  Py_DECREF(r);
  return !PyErr_Occurred();
}

PyObject* wrap(const Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}

PyObject* pack(std::initializer_list<Tensor> ts) {
  PyObject* r = PyTuple_New((Py_ssize_t)ts.size());
  if (!r) return nullptr;
  Py_ssize_t i = 0;
  for (const Tensor& t : ts) {
    PyObject* o = wrap(t);
    if (!o) {
      Py_DECREF(r);
      return nullptr;
    }
    PyTuple_SET_ITEM(r, i++, o);
  }
  return r;
}

bool rank_ok(int64_t r) { return r >= 16 && r <= K2Q_MAX_RANK && r % 16 == 0; }
bool width_ok(int64_t k) { return k >= 128 && k % 128 == 0 && k <= 16384; }

// Runs f with C++ exceptions turned into the Python ones that torch's own bindings give (an allocation that fails is
// torch.OutOfMemoryError, which callers catch by that name).
template <class F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (const std::exception&) {
    torch::translate_exception_to_python(std::current_exception());
  }
  return nullptr;
}

template <class T>
struct Plain {
  using type = T;   // an argument of this type is converted to it, not deduced from
};

// Calls an entry point with the GIL released.  The arguments are values made before that: reading a tensor's pointer can
// throw (a functorch wrapper has none), and nothing may throw without the GIL.
template <class... P>
int foreign(int (*fn)(P...), typename Plain<P>::type... args) {
  struct Released {
    PyThreadState* state = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(state); }
  } released;
  return fn(args...);
}

#define K2Q_ARGS(N)                                                       \
  if (n != N) {                                                           \
    PyErr_SetString(PyExc_TypeError, "wrong number of arguments");        \
    return nullptr;                                                       \
  }                                                                       \
  bool bad = false;
#define K2Q_REFUSE Py_RETURN_NONE

// alloc_codes(x2): the int8 code and f32 scale buffers of a forward over x2 (M, K).
PyObject* py_alloc_codes(PyObject*, PyObject* const* a, Py_ssize_t n) {
  K2Q_ARGS(1)
  return guarded([&]() -> PyObject* {
    const Tensor* x = tensor_of(a[0], bad);
    if (!x || x->dim() != 2) {
      PyErr_SetString(PyExc_ValueError, "x must be a 2-D tensor");
      return nullptr;
    }
    return pack({alloc({x->size(0), x->size(1)}, at::kChar, x->device()), alloc({x->size(0)}, at::kFloat, x->device())});
  });
}

// linear_fwd(x2, qx, sx, codes_ready, A, B, lora_scale, qw, sw, bias, w4, need_u) -> (y, u | None)
PyObject* py_linear_fwd(PyObject*, PyObject* const* a, Py_ssize_t n) {
  K2Q_ARGS(12)
  return guarded([&]() -> PyObject* {
    const Tensor *x = tensor_of(a[0], bad), *qx = tensor_of(a[1], bad), *sx = tensor_of(a[2], bad),
                 *A = tensor_of(a[4], bad), *B = tensor_of(a[5], bad), *qw = tensor_of(a[7], bad),
                 *sw = tensor_of(a[8], bad), *bias = tensor_of(a[9], bad);
    const int ready_codes = PyObject_IsTrue(a[3]), w4 = PyObject_IsTrue(a[10]), need_u = PyObject_IsTrue(a[11]);
    const double scale = PyFloat_AsDouble(a[6]);
    if (PyErr_Occurred()) return nullptr;
    if (bad || !x || !qx || !sx || !qw || !sw || x->dim() != 2 || qw->dim() != 2) K2Q_REFUSE;
    const int64_t M = x->size(0), K = x->size(1), N = qw->size(0);
    const c10::Device d = x->device();
    if (!ready(d) || x->scalar_type() != at::kBFloat16 || x->stride(1) != 1 || qw->device() != d || qx->dim() != 2 ||
        qx->size(0) != M || qx->size(1) != K || sx->dim() != 1 || sx->size(0) != M)
      K2Q_REFUSE;
    int64_t r = 0;
    if (A) {
      if (!B || A->dim() != 2 || B->dim() != 2) K2Q_REFUSE;
      r = A->size(0);
      if (A->size(1) != K || B->size(0) != N || B->size(1) != r || A->scalar_type() != at::kFloat ||
          B->scalar_type() != at::kFloat || A->device() != d || !A->is_contiguous() || !B->is_contiguous() || !rank_ok(r))
        K2Q_REFUSE;
    }
    if (bias && (bias->dim() != 1 || bias->size(0) != N || bias->scalar_type() != at::kFloat || bias->device() != d)) K2Q_REFUSE;
    void* st;
    if (!stream_of(d, st)) return nullptr;
    const int wmode = w4 ? K2Q_WMODE_W4 : K2Q_WMODE_W8;
    Tensor y = alloc({M, N}, at::kBFloat16, d);
    Tensor u = r && (need_u || M <= 8) ? alloc({M, r}, at::kFloat, d) : Tensor();
    // with u given, a call that takes u from the rotate/quant pass and whose GEMM does not split uses no workspace
    int64_t nws = api.linear_fwd_ws_bytes(wmode, M, N, K, r);
    if (nws > 0 && u.defined() && !ready_codes && M > 8 && api.linear_fwd_fuses_down(M, K, r) &&
        api.linear_fwd_ws_bytes(wmode, M, N, K, 0) == 0)
      nws = 0;
    Tensor ws = workspace(nws, d);
    const int rc = foreign(api.linear_fwd, as<uint16_t>(ptr(x)), x->stride(0), M, K, as<int8_t>(ptr(qx)),
                           as<float>(ptr(sx)), ready_codes, as<float>(ptr(A)), as<float>(A ? ptr(B) : nullptr), r,
                           (float)scale, as<float>(ptr(u)), wmode, ptr(qw), ptr(sw), as<float>(ptr(bias)), N,
                           as<uint16_t>(ptr(y)), ptr(ws), nws, st);
    if (rc) return PyLong_FromLong(rc);
    return pack({y, need_u ? u : Tensor()});
  });
}

// lora_grads(dy, x | None, u | None, B, lora_scale) -> (g, dA | None, dB | None)
PyObject* py_lora_grads(PyObject*, PyObject* const* a, Py_ssize_t n) {
  K2Q_ARGS(5)
  return guarded([&]() -> PyObject* {
    const Tensor *dy = tensor_of(a[0], bad), *x = tensor_of(a[1], bad), *u = tensor_of(a[2], bad),
                 *B = tensor_of(a[3], bad);
    const double scale = PyFloat_AsDouble(a[4]);
    if (PyErr_Occurred()) return nullptr;
    if (bad || !dy || !B) K2Q_REFUSE;
    const c10::Device d = dy->device();
    if (!ready(d) || !operand(dy, at::kBFloat16, 2, d) || !operand(B, at::kFloat, 2, d)) K2Q_REFUSE;
    const int64_t M = dy->size(0), N = dy->size(1), r = B->size(1);
    if (B->size(0) != N || !rank_ok(r) || N % 128) K2Q_REFUSE;
    int64_t K = 128;
    if (x) {
      if (!operand(x, at::kBFloat16, 2, d) || x->size(0) != M || !width_ok(x->size(1))) K2Q_REFUSE;
      K = x->size(1);
    }
    if (u && (!operand(u, at::kFloat, 2, d) || u->size(0) != M || u->size(1) != r)) K2Q_REFUSE;
    void* st;
    if (!stream_of(d, st)) return nullptr;
    const int64_t nws = api.lora_grads_ws_bytes(M, N, K, r);
    Tensor ws = workspace(nws, d);
    Tensor g = alloc({M, r}, at::kFloat, d);
    Tensor dA = x ? alloc({r, K}, at::kFloat, d) : Tensor(), dB = u ? alloc({N, r}, at::kFloat, d) : Tensor();
    const int rc = foreign(api.lora_grads, as<uint16_t>(ptr(dy)), as<uint16_t>(ptr(x)), as<float>(ptr(u)),
                           as<float>(ptr(B)), r, (float)scale, M, N, K, as<float>(ptr(g)), as<float>(ptr(dA)),
                           as<float>(ptr(dB)), ptr(ws), nws, st);
    if (rc) return PyLong_FromLong(rc);
    return pack({g, dA, dB});
  });
}

// lora_down(x, A) -> u
PyObject* py_lora_down(PyObject*, PyObject* const* a, Py_ssize_t n) {
  K2Q_ARGS(2)
  return guarded([&]() -> PyObject* {
    const Tensor *x = tensor_of(a[0], bad), *A = tensor_of(a[1], bad);
    if (bad || !x || !A) K2Q_REFUSE;
    const c10::Device d = x->device();
    if (!ready(d) || !operand(x, at::kBFloat16, 2, d) || !operand(A, at::kFloat, 2, d)) K2Q_REFUSE;
    const int64_t M = x->size(0), K = x->size(1), r = A->size(0);
    if (A->size(1) != K || !rank_ok(r)) K2Q_REFUSE;
    void* st;
    if (!stream_of(d, st)) return nullptr;
    const int64_t nws = api.lora_down_ws_bytes(M, K, r);
    Tensor ws = workspace(nws, d), u = alloc({M, r}, at::kFloat, d);
    const int rc = foreign(api.lora_down, as<uint16_t>(ptr(x)), M, K, K, as<float>(ptr(A)), r, ptr(ws), nws,
                           as<float>(ptr(u)), st);
    return rc ? PyLong_FromLong(rc) : wrap(u);
  });
}

// pad_factors(A, B, rp) -> (rp, K) and (N, rp) with zero ranks behind A's and B's
PyObject* py_pad_factors(PyObject*, PyObject* const* a, Py_ssize_t n) {
  K2Q_ARGS(3)
  return guarded([&]() -> PyObject* {
    const Tensor *A = tensor_of(a[0], bad), *B = tensor_of(a[1], bad);
    const int64_t rp = PyLong_AsLongLong(a[2]);
    if (PyErr_Occurred()) return nullptr;
    if (bad || !A || !B) K2Q_REFUSE;
    const c10::Device d = A->device();
    if (!ready(d) || !operand(A, at::kFloat, 2, d) || !operand(B, at::kFloat, 2, d)) K2Q_REFUSE;
    const int64_t r = A->size(0), K = A->size(1), N = B->size(0);
    if (B->size(1) != r || r < 1 || rp < r || !rank_ok(rp) || K % 4 || K < 4 || N < 1) K2Q_REFUSE;
    void* st;
    if (!stream_of(d, st)) return nullptr;
    Tensor ap = alloc({rp, K}, at::kFloat, d), bp = alloc({N, rp}, at::kFloat, d);
    const int rc = foreign(api.pad_factors, as<float>(ptr(A)), as<float>(ptr(B)), r, rp, K, N, as<float>(ptr(ap)),
                           as<float>(ptr(bp)), st);
    if (rc) return PyLong_FromLong(rc);
    return pack({ap, bp});
  });
}

// A ConvRot layer's codes and scales on device d; N, K its widths.
bool convrot_ok(const Tensor* q, const Tensor* s, bool w4, c10::Device d, int64_t& N, int64_t& K) {
  if (!operand(q, w4 ? at::kByte : at::kChar, 2, d) || !operand(s, w4 ? at::kBFloat16 : at::kFloat, w4 ? 2 : 1, d))
    return false;
  N = q->size(0);
  K = w4 ? 2 * q->size(1) : q->size(1);
  if (w4 ? (s->size(0) != K / 64 || s->size(1) != N) : s->size(0) != N) return false;
  return width_ok(K) && N % 64 == 0;
}

// dx_weight(qw, sw, w4) -> wt (K, N)
PyObject* py_dx_weight(PyObject*, PyObject* const* a, Py_ssize_t n) {
  K2Q_ARGS(3)
  return guarded([&]() -> PyObject* {
    const Tensor *q = tensor_of(a[0], bad), *s = tensor_of(a[1], bad);
    const int w4 = PyObject_IsTrue(a[2]);
    if (bad || !q || !s) K2Q_REFUSE;
    const c10::Device d = q->device();
    int64_t N, K;
    if (!ready(d) || !convrot_ok(q, s, w4, d, N, K)) K2Q_REFUSE;
    void* st;
    if (!stream_of(d, st)) return nullptr;
    Tensor wt = alloc({K, N}, at::kBFloat16, d);
    const int rc = foreign(api.dx_prep_eff, w4 ? nullptr : as<int8_t>(ptr(q)), w4 ? nullptr : as<float>(ptr(s)),
                           w4 ? as<uint8_t>(ptr(q)) : nullptr, w4 ? as<uint16_t>(ptr(s)) : nullptr, N, K,
                           as<uint16_t>(ptr(wt)), st);
    return rc ? PyLong_FromLong(rc) : wrap(wt);
  });
}

// dx = bf16(dy wt^T + g A) over wt (K, N) with the split schedule's workspace; the operands are checked.
PyObject* dx_lin(const Tensor& dy, const Tensor& wt, const Tensor* g, const Tensor* A, void* st) {
  const int64_t M = dy.size(0), N = dy.size(1), K = wt.size(0), r = g ? g->size(1) : 0;
  const c10::Device d = dy.device();
  Tensor dx = alloc({M, K}, at::kBFloat16, d);
  const int64_t nws = api.gemm_plan_ws_bytes(K2Q_GEMM_DX_LIN, M, N, K);
  Tensor ws = workspace(nws, d);
  const int rc = foreign(api.gemm_dx_lin, as<uint16_t>(dy.data_ptr()), as<uint16_t>(wt.data_ptr()), M, N, K,
                         as<float>(ptr(g)), r ? as<float>(ptr(A)) : nullptr, r, as<uint16_t>(dx.data_ptr()), ptr(ws),
                         nws, st);
  return rc ? PyLong_FromLong(rc) : wrap(dx);
}

bool lora_terms_ok(const Tensor* g, const Tensor* A, int64_t M, int64_t K, c10::Device d) {
  if (!g) return true;
  return operand(g, at::kFloat, 2, d) && operand(A, at::kFloat, 2, d) && g->size(0) == M && rank_ok(g->size(1)) &&
         A->size(0) == g->size(1) && A->size(1) == K;
}

// gemm_dx(dy, wt, g | None, A | None, qw | None, sw | None, w4) -> dx: the input gradient through a prebuilt
// effective weight (of the ConvRot layer qw / sw; None for an fp8 base's)
PyObject* py_gemm_dx(PyObject*, PyObject* const* a, Py_ssize_t n) {
  K2Q_ARGS(7)
  return guarded([&]() -> PyObject* {
    const Tensor *dy = tensor_of(a[0], bad), *wt = tensor_of(a[1], bad), *g = tensor_of(a[2], bad),
                 *A = tensor_of(a[3], bad), *q = tensor_of(a[4], bad), *s = tensor_of(a[5], bad);
    const int w4 = PyObject_IsTrue(a[6]);
    if (bad || !dy || !wt) K2Q_REFUSE;
    const c10::Device d = dy->device();
    if (!ready(d) || !operand(dy, at::kBFloat16, 2, d) || !operand(wt, at::kBFloat16, 2, d)) K2Q_REFUSE;
    if (wt->size(1) != dy->size(1) || dy->size(1) % 64 || !width_ok(wt->size(0)) ||
        !lora_terms_ok(g, A, dy->size(0), wt->size(0), d))
      K2Q_REFUSE;
    int64_t N, K;
    if (q && (!convrot_ok(q, s, w4, d, N, K) || N != dy->size(1) || K != wt->size(0))) K2Q_REFUSE;
    void* st;
    if (!stream_of(d, st)) return nullptr;
    return dx_lin(*dy, *wt, g, A, st);
  });
}

// The fp8 base's codes (N, K) and bf16 row scales.
bool fp8_ok(const Tensor* q, const Tensor* s, c10::Device d) {
  return operand(q, at::kFloat8_e4m3fn, 2, d) && s && s->scalar_type() == at::kBFloat16 && s->numel() == q->size(0) &&
         s->is_contiguous() && s->device() == d && q->size(1) % 64 == 0;
}

// dequant_fp8(q, s, transpose) -> bf16 (N, K), or (K, N)
PyObject* py_dequant_fp8(PyObject*, PyObject* const* a, Py_ssize_t n) {
  K2Q_ARGS(3)
  return guarded([&]() -> PyObject* {
    const Tensor *q = tensor_of(a[0], bad), *s = tensor_of(a[1], bad);
    const int tr = PyObject_IsTrue(a[2]);
    if (bad || !q || !s) K2Q_REFUSE;
    const c10::Device d = q->device();
    if (!ready(d) || !fp8_ok(q, s, d)) K2Q_REFUSE;
    const int64_t N = q->size(0), K = q->size(1);
    if (tr && N % 8) K2Q_REFUSE;
    void* st;
    if (!stream_of(d, st)) return nullptr;
    Tensor w = tr ? alloc({K, N}, at::kBFloat16, d) : alloc({N, K}, at::kBFloat16, d);
    const int rc = foreign(api.dequant_fp8, as<uint8_t>(ptr(q)), as<uint16_t>(ptr(s)), N, K, tr, as<uint16_t>(ptr(w)),
                           st);
    return rc ? PyLong_FromLong(rc) : wrap(w);
  });
}

// gemm_bf16(x, w, bias | None, u | None, B | None, lora_scale) -> y
PyObject* py_gemm_bf16(PyObject*, PyObject* const* a, Py_ssize_t n) {
  K2Q_ARGS(6)
  return guarded([&]() -> PyObject* {
    const Tensor *x = tensor_of(a[0], bad), *w = tensor_of(a[1], bad), *bias = tensor_of(a[2], bad),
                 *u = tensor_of(a[3], bad), *B = tensor_of(a[4], bad);
    const double scale = PyFloat_AsDouble(a[5]);
    if (PyErr_Occurred()) return nullptr;
    if (bad || !x || !w) K2Q_REFUSE;
    const c10::Device d = x->device();
    if (!ready(d) || !operand(x, at::kBFloat16, 2, d) || !operand(w, at::kBFloat16, 2, d)) K2Q_REFUSE;
    const int64_t M = x->size(0), K = x->size(1), N = w->size(0);
    if (w->size(1) != K || K % 64 || N % 4) K2Q_REFUSE;
    if (bias && (!operand(bias, at::kFloat, 1, d) || bias->size(0) != N)) K2Q_REFUSE;
    int64_t r = 0;
    if (u) {
      if (!operand(u, at::kFloat, 2, d) || !operand(B, at::kFloat, 2, d)) K2Q_REFUSE;
      r = u->size(1);
      if (u->size(0) != M || B->size(0) != N || B->size(1) != r || !rank_ok(r)) K2Q_REFUSE;
    }
    void* st;
    if (!stream_of(d, st)) return nullptr;
    Tensor y = alloc({M, N}, at::kBFloat16, d);
    const int64_t nws = api.gemm_plan_ws_bytes(K2Q_GEMM_BF16, M, N, K);
    Tensor ws = workspace(nws, d);
    const int rc = foreign(api.gemm_bf16, as<uint16_t>(ptr(x)), as<uint16_t>(ptr(w)), as<float>(ptr(bias)),
                           as<float>(ptr(u)), u ? as<float>(ptr(B)) : nullptr, r, (float)scale, M, N, K,
                           as<uint16_t>(ptr(y)), ptr(ws), nws, st);
    return rc ? PyLong_FromLong(rc) : wrap(y);
  });
}

// bind(dict of entry point addresses, raw stream getter)
PyObject* py_bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  K2Q_ARGS(2)
  (void)bad;
  auto get = [&](const char* name, auto& fn) {
    PyObject* v = PyDict_GetItemString(a[0], name);
    if (!v) {
      PyErr_Format(PyExc_KeyError, "no address for %s", name);
      return false;
    }
    fn = reinterpret_cast<std::decay_t<decltype(fn)>>(PyLong_AsVoidPtr(v));
    return !PyErr_Occurred();
  };
  if (!get("k2q_linear_fwd", api.linear_fwd) || !get("k2q_linear_fwd_ws_bytes", api.linear_fwd_ws_bytes) ||
      !get("k2q_linear_fwd_fuses_down", api.linear_fwd_fuses_down) || !get("k2q_lora_grads", api.lora_grads) ||
      !get("k2q_lora_grads_ws_bytes", api.lora_grads_ws_bytes) || !get("k2q_lora_down", api.lora_down) ||
      !get("k2q_lora_down_ws_bytes", api.lora_down_ws_bytes) || !get("k2q_pad_factors", api.pad_factors) ||
      !get("k2q_dx_prep_eff", api.dx_prep_eff) || !get("k2q_gemm_dx_lin", api.gemm_dx_lin) ||
      !get("k2q_dequant_fp8", api.dequant_fp8) || !get("k2q_gemm_bf16", api.gemm_bf16) ||
      !get("k2q_gemm_plan_ws_bytes", api.gemm_plan_ws_bytes))
    return nullptr;
  Py_INCREF(a[1]);
  Py_XSETREF(raw_stream_of, a[1]);
  Py_RETURN_NONE;
}

// device_checked(index): the device is gfx950
PyObject* py_device_checked(PyObject*, PyObject* const* a, Py_ssize_t n) {
  K2Q_ARGS(1)
  (void)bad;
  const long i = PyLong_AsLong(a[0]);
  if (PyErr_Occurred()) return nullptr;
  if (i >= 0 && i < MAX_DEVICES) device_ok[i] = true;
  Py_RETURN_NONE;
}

#define K2Q_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {K2Q_METHOD(bind),        K2Q_METHOD(device_checked), K2Q_METHOD(alloc_codes),
                         K2Q_METHOD(linear_fwd),  K2Q_METHOD(lora_grads),     K2Q_METHOD(lora_down),
                         K2Q_METHOD(dx_weight),   K2Q_METHOD(gemm_dx),        K2Q_METHOD(dequant_fp8),
                         K2Q_METHOD(gemm_bf16),   K2Q_METHOD(pad_factors),    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_k2q_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__k2q_native() {
  PyObject* m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "built_for", K2Q_BUILT_FOR) < 0) Py_CLEAR(m);
  return m;
}
