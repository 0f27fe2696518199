// The tensor operators of hpfp8/ops.py that a linear layer's step is made of, from Python straight to the C ABI of libhpfp8.so.
//
// A small layer's step is bound by the host: through Python a launch costs 10 to 24 us (outputs allocated one by one and turned
// into views, arguments checked, a ctypes call), of which the launch itself is 3.  Each function here does the same for the
// plain case -- ordinary tensors of the types and layouts that the kernels take -- and returns None for everything else,
// refused calls among them: the Python form of the operator then runs as if this one were not there, and copies, pads or raises.
// Host time of a call, us, Python form / here: quantize_1x128 10.5 / 5.3, both forms 15.9 / 7.8, with the bias gradient 24.4 / 12.1,
// 128 x 128 with the transposed codes 12.7 / 6.4, gemm_blockwise 12.2 / 4.9.
#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include <map>
#include <mutex>

#include "../../include/hpfp8.h"

namespace {

constexpr int64_t kBlock = 128;

// the library's functions, by the names of the header (bound at run time: HPFP8_LIBRARY may name another build)
#define HPFP8_FUNCTIONS(X) \
  X(hpfp8_quantize_1x128_kmajor_bf16) X(hpfp8_quantize_1x128_kmajor_pow2_bf16) X(hpfp8_quantize_1x128_and_128x1_t_bf16) \
  X(hpfp8_quantize_1x128_and_128x1_t_pow2_bf16) X(hpfp8_quantize_128x1_t_colsum_bf16) X(hpfp8_quantize_rows_128x1_t_bf16) \
  X(hpfp8_column_sum_finish) X(hpfp8_quantize_128x128_bf16) X(hpfp8_quantize_128x128_pow2_bf16) \
  X(hpfp8_quantize_per_tensor_t_bf16) X(hpfp8_transpose_codes) X(hpfp8_gemm_blockwise) X(hpfp8_gemm_blockwise_pow2) X(hpfp8_gemm_per_tensor)
struct Library {
#define HPFP8_POINTER(name) decltype(&::name) name = nullptr;
  HPFP8_FUNCTIONS(HPFP8_POINTER)
#undef HPFP8_POINTER
} lib;
PyObject* fail_function = nullptr;       // fail_function(name, status) raises
PyObject* backward_function = nullptr;   // backward_function(grad_out, saved tensors, ..., as LinearNode has them) -> (dx, dw, db)
PyObject* parameter_class = nullptr;

// A tensor without wrappers or modes around it, on the device that kernels are launched on.
bool plain(PyObject* o, int64_t device, const at::Tensor*& t) {
  if (o != Py_None && (Py_TYPE(o) == (PyTypeObject*)THPVariableClass || Py_TYPE(o) == (PyTypeObject*)parameter_class)) {
    t = &THPVariable_Unpack(o);
    return t->defined() && t->is_cuda() && t->get_device() == device && t->layout() == at::kStrided && !at::isTensorSubclassLike(*t);
  }
  return false;
}
bool no_modes() { return !c10::impl::TorchDispatchModeTLS::any_modes_set(); }

bool source_2d(PyObject* o, int64_t device, const at::Tensor*& t) {      // bf16 [M > 0, C > 0, a multiple of 128], contiguous
  return plain(o, device, t) && t->scalar_type() == at::kBFloat16 && t->dim() == 2 && t->size(0) > 0 && t->size(1) > 0 &&
         t->size(1) % kBlock == 0 && t->is_contiguous();
}
bool codes_2d(PyObject* o, int64_t device, const at::Tensor*& t) {
  return plain(o, device, t) && t->scalar_type() == at::kFloat8_e4m3fn && t->dim() == 2 && t->size(0) > 0 && t->size(1) > 0 &&
         t->size(1) % kBlock == 0 && t->stride(1) == 1 && (t->size(0) == 1 || t->stride(0) % 16 == 0);
}
bool floats(PyObject* o, int64_t device, const at::Tensor*& t) { return plain(o, device, t) && t->scalar_type() == at::kFloat; }
bool bias_of(PyObject* o, int64_t device, int64_t n, const at::Tensor*& t) {
  t = nullptr;
  return o == Py_None || (plain(o, device, t) && t->scalar_type() == at::kBFloat16 && t->dim() == 1 && t->size(0) == n && t->is_contiguous());
}

// per-row b scales [rows, k-blocks] as the kernel reads them: k-block-major, rows of whole vectors
bool row_scales_fit(const at::Tensor& s) {
  return s.stride(0) == 1 && (s.size(1) == 1 || (s.stride(1) >= s.size(0) && s.stride(1) % 4 == 0)) && (uintptr_t)s.data_ptr() % 16 == 0;
}
int64_t row_stride(const at::Tensor& t) { return t.size(0) > 1 ? t.stride(0) : std::max<int64_t>(t.size(1), 16); }
int64_t rows_up(int64_t m) { return (m + kBlock - 1) / kBlock * kBlock; }
int64_t padded_ld(int64_t n) { return n / kBlock % 2 == 1 ? n : n + kBlock; }       // (ops._padded_ld has the reason)

at::Tensor new_codes(const at::Tensor& like, int64_t r, int64_t c) { return at::empty({r, c}, like.options().dtype(at::kFloat8_e4m3fn)); }
at::Tensor new_codes_t(const at::Tensor& like, int64_t r, int64_t c) {
  return at::empty_strided({r, c}, {padded_ld(c), 1}, like.options().dtype(at::kFloat8_e4m3fn));
}
at::Tensor new_floats(const at::Tensor& like, int64_t r, int64_t c) { return at::empty({r, c}, like.options().dtype(at::kFloat)); }
// [r, c] stored column by column: k-block-major scales
at::Tensor new_floats_t(const at::Tensor& like, int64_t r, int64_t c) {
  return at::empty_strided({r, c}, {1, r}, like.options().dtype(at::kFloat));
}
float* f32(const at::Tensor& t) { return t.data_ptr<float>(); }

// The status of the last C call of an operator and its name; what the operator returns once the interpreter's lock is held again.
struct Call {
  const char* name = nullptr;
  int status = 0;
  bool ok() const { return status == 0; }
};
#define HPFP8_CALL(call, function, ...) ((call).name = #function, (call).status = lib.function(__VA_ARGS__))

PyObject* failed(const Call& call) {
  PyObject* r = PyObject_CallFunction(fail_function, "si", call.name, call.status);
  Py_XDECREF(r);
  if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "%s failed (%d)", call.name, call.status);
  return nullptr;
}
template <class... T>
PyObject* tuple_of(T&&... tensors) {
  PyObject* out = PyTuple_New(sizeof...(T));
  if (!out) return nullptr;
  Py_ssize_t i = 0;
  (PyTuple_SET_ITEM(out, i++, THPVariable_Wrap(std::forward<T>(tensors))), ...);
  return out;
}

struct Where {
  int64_t device;
  void* stream;
};
// the last two arguments: device index and stream handle
Where where(PyObject* const* args, Py_ssize_t n) {
  const int64_t device = PyLong_AsLongLong(args[n - 2]);
  void* const stream = PyLong_AsVoidPtr(args[n - 1]);
  if (PyErr_Occurred()) throw python_error();
  return {device, stream};
}
bool truth(PyObject* o) {
  const int r = PyObject_IsTrue(o);
  if (r < 0) throw python_error();
  return r != 0;
}
void expect(Py_ssize_t got, Py_ssize_t want) {
  TORCH_CHECK_TYPE(got == want, "expected ", want, " arguments, got ", got);
}

// (x, pow2, device, stream) -> (codes, scale_inv), k-block-major scales
PyObject* quantize_1x128(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 4);
  const Where w = where(args, n);
  const bool pow2 = truth(args[1]);
  const at::Tensor* x;
  if (!source_2d(args[0], w.device, x) || !no_modes()) Py_RETURN_NONE;
  at::Tensor q, s;
  Call call;
  {
    pybind11::gil_scoped_release free;
    const int64_t m = x->size(0), k = x->size(1);
    q = new_codes(*x, m, k);
    s = new_floats_t(*x, m, k / kBlock);
    if (pow2) HPFP8_CALL(call, hpfp8_quantize_1x128_kmajor_pow2_bf16, x->data_ptr(), m, k, q.data_ptr(), nullptr, f32(s), w.stream);
    else HPFP8_CALL(call, hpfp8_quantize_1x128_kmajor_bf16, x->data_ptr(), m, k, q.data_ptr(), nullptr, f32(s), w.stream);
  }
  return call.ok() ? tuple_of(std::move(q), std::move(s)) : failed(call);
  END_HANDLE_TH_ERRORS
}

// Both operand forms of x from one read of it, and the sum over its rows; any number of rows.
struct Forms {
  at::Tensor q, s, qt, st, total;        // (per tensor: s is the one scale, st undefined)
};
Forms make_both(const at::Tensor& x, bool pow2, bool column_sum, void* stream, Call& call) {
  const int64_t m = x.size(0), k = x.size(1), mp = rows_up(m);
  Forms f;
  f.q = new_codes(x, m, k);
  f.qt = new_codes_t(x, k, mp);
  f.s = new_floats_t(x, m, k / kBlock);
  f.st = new_floats_t(x, k, mp / kBlock);
  at::Tensor part;
  if (column_sum) part = new_floats(x, mp / kBlock, k);
  void *const src = x.data_ptr(), *const q = f.q.data_ptr(), *const qt = f.qt.data_ptr();
  const int64_t ld = f.qt.stride(0);
  if (m != mp)
    HPFP8_CALL(call, hpfp8_quantize_rows_128x1_t_bf16, src, m, k, q, f32(f.s), qt, ld, f32(f.st), pow2, column_sum ? f32(part) : nullptr, stream);
  else if (column_sum)
    HPFP8_CALL(call, hpfp8_quantize_128x1_t_colsum_bf16, src, m, k, q, nullptr, f32(f.s), qt, ld, nullptr, f32(f.st), pow2, f32(part), stream);
  else if (pow2)
    HPFP8_CALL(call, hpfp8_quantize_1x128_and_128x1_t_pow2_bf16, src, m, k, 1, q, nullptr, f32(f.s), qt, ld, nullptr, f32(f.st), stream);
  else
    HPFP8_CALL(call, hpfp8_quantize_1x128_and_128x1_t_bf16, src, m, k, 1, q, nullptr, f32(f.s), qt, ld, nullptr, f32(f.st), stream);
  if (column_sum && call.ok()) {
    f.total = at::empty({k}, x.options());
    HPFP8_CALL(call, hpfp8_column_sum_finish, f32(part), mp / kBlock, k, f.total.data_ptr(), nullptr, stream);
  }
  return f;
}

// The same with one scale; sync: the block through which the one-launch form's grid agrees on the maximum, or null.
Forms make_per_tensor(const at::Tensor& x, bool column_sum, uint32_t* sync, void* stream, Call& call) {
  const int64_t m = x.size(0), k = x.size(1), mp = rows_up(m);
  Forms f;
  f.q = new_codes(x, m, k);
  f.qt = new_codes_t(x, k, mp);
  f.s = at::empty({}, x.options().dtype(at::kFloat));
  at::Tensor part, amax;
  if (column_sum) part = new_floats(x, mp / kBlock, k);
  if (!sync) amax = at::empty({}, x.options().dtype(at::kFloat));
  HPFP8_CALL(call, hpfp8_quantize_per_tensor_t_bf16, x.data_ptr(), m, k, f.q.data_ptr(), f.qt.data_ptr(), f.qt.stride(0),
             sync ? nullptr : f32(amax), nullptr, f32(f.s), sync, column_sum ? f32(part) : nullptr, stream);
  if (column_sum && call.ok()) {
    f.total = at::empty({k}, x.options());
    HPFP8_CALL(call, hpfp8_column_sum_finish, f32(part), mp / kBlock, k, f.total.data_ptr(), nullptr, stream);
  }
  return f;
}

void multiply_blockwise(const at::Tensor& a, const at::Tensor& sa, const at::Tensor& b, const at::Tensor& sb, int64_t sb_sn, int64_t sb_sk,
                        const void* bias, const at::Tensor& c, int64_t gran, bool accumulate, bool pow2, void* stream, Call& call) {
  const int64_t m = a.size(0), k = a.size(1), n = b.size(0), ldc = m > 1 ? c.stride(0) : n;
  const int out_type = c.scalar_type() == at::kFloat ? HPFP8_OUT_F32 : HPFP8_OUT_BF16;
  if (pow2)
    HPFP8_CALL(call, hpfp8_gemm_blockwise_pow2, a.data_ptr(), row_stride(a), f32(sa), sa.stride(0), sa.stride(1), b.data_ptr(), row_stride(b),
               f32(sb), sb_sn, sb_sk, (int)gran, m, n, k, bias, c.data_ptr(), ldc, out_type, accumulate, stream);
  else
    HPFP8_CALL(call, hpfp8_gemm_blockwise, a.data_ptr(), row_stride(a), f32(sa), sa.stride(0), sa.stride(1), b.data_ptr(), row_stride(b),
               f32(sb), sb_sn, sb_sk, (int)gran, m, n, k, bias, c.data_ptr(), ldc, out_type, accumulate, stream);
}

at::Tensor multiply_per_tensor(const at::Tensor& a, const at::Tensor& sa, const at::Tensor& b, const at::Tensor& sb, const void* bias,
                               void* stream, Call& call) {
  at::Tensor c = at::empty({a.size(0), b.size(0)}, a.options().dtype(at::kBFloat16));
  HPFP8_CALL(call, hpfp8_gemm_per_tensor, a.data_ptr(), row_stride(a), f32(sa), b.data_ptr(), row_stride(b), f32(sb), a.size(0), b.size(0),
             a.size(1), bias, c.data_ptr(), b.size(0), HPFP8_OUT_BF16, stream);
  return c;
}

// (x, pow2, column_sum, device, stream) -> (codes, scale_inv, codes_t, scale_inv_t[, sum over rows])
PyObject* both_forms(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 5);
  const Where w = where(args, n);
  const bool pow2 = truth(args[1]), column_sum = truth(args[2]);
  const at::Tensor* x;
  if (!source_2d(args[0], w.device, x) || !no_modes()) Py_RETURN_NONE;
  Forms f;
  Call call;
  {
    pybind11::gil_scoped_release free;
    f = make_both(*x, pow2, column_sum, w.stream, call);
  }
  if (!call.ok()) return failed(call);
  if (column_sum) return tuple_of(std::move(f.q), std::move(f.s), std::move(f.qt), std::move(f.st), std::move(f.total));
  return tuple_of(std::move(f.q), std::move(f.s), std::move(f.qt), std::move(f.st));
  END_HANDLE_TH_ERRORS
}

// (w, with_transpose, pow2, device, stream) -> (codes, scale_inv[, codes_t])
PyObject* quantize_128x128(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 5);
  const Where w = where(args, n);
  const bool with_t = truth(args[1]), pow2 = truth(args[2]);
  const at::Tensor* x;
  if (!source_2d(args[0], w.device, x) || x->size(0) % kBlock || !no_modes()) Py_RETURN_NONE;
  at::Tensor q, s, qt;
  Call call;
  {
    pybind11::gil_scoped_release free;
    const int64_t r = x->size(0), c = x->size(1);
    q = new_codes(*x, r, c);
    if (with_t) qt = new_codes_t(*x, c, r);
    s = new_floats(*x, r / kBlock, c / kBlock);
    void* const t = with_t ? qt.data_ptr() : nullptr;
    const int64_t ld = with_t ? qt.stride(0) : 0;
    if (pow2) HPFP8_CALL(call, hpfp8_quantize_128x128_pow2_bf16, x->data_ptr(), r, c, q.data_ptr(), t, ld, nullptr, f32(s), w.stream);
    else HPFP8_CALL(call, hpfp8_quantize_128x128_bf16, x->data_ptr(), r, c, q.data_ptr(), t, ld, nullptr, f32(s), w.stream);
  }
  if (!call.ok()) return failed(call);
  return with_t ? tuple_of(std::move(q), std::move(s), std::move(qt)) : tuple_of(std::move(q), std::move(s));
  END_HANDLE_TH_ERRORS
}

// (x, column_sum, sync block or None, device, stream) -> (codes, scale_inv, codes_t[, sum over rows])
PyObject* quantize_per_tensor_t(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 5);
  const Where w = where(args, n);
  const bool column_sum = truth(args[1]);
  const at::Tensor *x, *sync = nullptr;
  if (!source_2d(args[0], w.device, x) || (args[2] != Py_None && !plain(args[2], w.device, sync)) || !no_modes()) Py_RETURN_NONE;
  Forms f;
  Call call;
  {
    pybind11::gil_scoped_release free;
    f = make_per_tensor(*x, column_sum, sync ? (uint32_t*)sync->data_ptr() : nullptr, w.stream, call);
  }
  if (!call.ok()) return failed(call);
  if (column_sum) return tuple_of(std::move(f.q), std::move(f.s), std::move(f.qt), std::move(f.total));
  return tuple_of(std::move(f.q), std::move(f.s), std::move(f.qt));
  END_HANDLE_TH_ERRORS
}

// (a, sa, b, sb, bias or None, out or None, sb_gran, accumulate, pow2, device, stream) -> c; out: float32 or bfloat16 [M, N]
PyObject* gemm_blockwise(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  expect(n_args, 11);
  const Where w = where(args, n_args);
  const int64_t gran = PyLong_AsLongLong(args[6]);
  if (PyErr_Occurred()) throw python_error();
  const bool accumulate = truth(args[7]), pow2 = truth(args[8]);
  const at::Tensor *a, *sa, *b, *sb, *bias, *given = nullptr;
  if (!codes_2d(args[0], w.device, a) || !codes_2d(args[2], w.device, b) || !floats(args[1], w.device, sa) || !floats(args[3], w.device, sb))
    Py_RETURN_NONE;
  const int64_t m = a->size(0), k = a->size(1), n = b->size(0), kb = k / kBlock;
  if (b->size(1) != k || n % kBlock || (gran != 1 && gran != kBlock) || sa->dim() != 2 || sa->size(0) != m || sa->size(1) != kb ||
      sb->dim() != 2 || sb->size(0) != n / gran || sb->size(1) != kb || !bias_of(args[4], w.device, n, bias) || !no_modes())
    Py_RETURN_NONE;
  // (per-row scales in another layout than the kernel's are copied by the Python form)
  if (gran == 1 && !row_scales_fit(*sb)) Py_RETURN_NONE;
  if (args[5] == Py_None) {
    if (accumulate) Py_RETURN_NONE;
  } else if (!plain(args[5], w.device, given) || given->dim() != 2 || given->size(0) != m || given->size(1) != n || given->stride(1) != 1 ||
             (given->scalar_type() != at::kFloat && (accumulate || given->scalar_type() != at::kBFloat16))) {
    Py_RETURN_NONE;
  }
  at::Tensor c;
  Call call;
  {
    pybind11::gil_scoped_release free;
    c = given ? *given : at::empty({m, n}, a->options().dtype(at::kBFloat16));
    multiply_blockwise(*a, *sa, *b, *sb, sb->stride(0), sb->stride(1), bias ? bias->data_ptr() : nullptr, c, gran, accumulate, pow2, w.stream,
                       call);
  }
  if (!call.ok()) return failed(call);
  if (!given) return THPVariable_Wrap(std::move(c));
  Py_INCREF(args[5]);
  return args[5];
  END_HANDLE_TH_ERRORS
}

// (a, sa, b, sb, bias or None, device, stream) -> c, bf16
PyObject* gemm_per_tensor(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  expect(n_args, 7);
  const Where w = where(args, n_args);
  const at::Tensor *a, *sa, *b, *sb, *bias;
  if (!codes_2d(args[0], w.device, a) || !codes_2d(args[2], w.device, b) || !floats(args[1], w.device, sa) || !floats(args[3], w.device, sb))
    Py_RETURN_NONE;
  const int64_t k = a->size(1), n = b->size(0);
  if (b->size(1) != k || n % kBlock || sa->numel() != 1 || sb->numel() != 1 || !bias_of(args[4], w.device, n, bias) || !no_modes()) Py_RETURN_NONE;
  at::Tensor c;
  Call call;
  {
    pybind11::gil_scoped_release free;
    c = multiply_per_tensor(*a, *sa, *b, *sb, bias ? bias->data_ptr() : nullptr, w.stream, call);
  }
  return call.ok() ? THPVariable_Wrap(std::move(c)) : failed(call);
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------
// backward of the linear in training
// ------------------------------------------------------------------------------------------------
// One block per device and stream for the one-launch per-tensor quantizer, as ops._sync_words keeps (which has the rule: zero
// between calls, never two launches at once, none while a graph is captured).
uint32_t* sync_block(const at::Tensor& x, int64_t tiles, hipStream_t stream) {
  constexpr int64_t kOnePassTiles = 256;
  if (tiles > kOnePassTiles || c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return nullptr;
  static std::mutex lock;
  static auto* const blocks = new std::map<std::pair<int64_t, hipStream_t>, at::Tensor>;      // (never destroyed: the device may go first)
  std::lock_guard<std::mutex> guard(lock);
  at::Tensor& t = (*blocks)[{x.get_device(), stream}];
  if (!t.defined()) t = at::zeros({128}, x.options().dtype(at::kInt));
  return (uint32_t*)t.data_ptr();
}

[[noreturn]] void raise_python_error() {       // (with the interpreter's lock held)
  python_error e;
  e.persist();
  throw e;
}
[[noreturn]] void raise(const Call& call) {
  pybind11::gil_scoped_acquire held;
  failed(call);
  raise_python_error();
}

// Saved tensors come back through whatever hooks the program has set, so they are looked at again before a kernel reads them.
bool codes_again(const at::Tensor& t, const at::Tensor& go, int64_t r, int64_t c) {
  return t.defined() && t.device() == go.device() && t.layout() == at::kStrided && !at::isTensorSubclassLike(t) &&
         (t.scalar_type() == at::kFloat8_e4m3fn || t.scalar_type() == at::kByte) && t.dim() == 2 && t.size(0) == r && t.size(1) == c &&
         t.stride(1) == 1 && (r == 1 || t.stride(0) % 16 == 0);
}
bool floats_again(const at::Tensor& t, const at::Tensor& go, at::IntArrayRef sizes) {
  return t.defined() && t.device() == go.device() && t.layout() == at::kStrided && !at::isTensorSubclassLike(t) && t.scalar_type() == at::kFloat &&
         t.sizes() == sizes;
}

// What forward has made, in Python, for y = x W^T + b with gradients of x and W to come: y, and for backward xt, sxt (per
// tensor: the one scale), the weight's transposed codes (per tensor with a cached weight: its codes), sw.
struct Made {
  at::Tensor y, xt, sxt, w, sw;
  bool per_tensor, pow2, has_bias, w_transposed;
};

// The graph's node.  A step of a small layer, forward and backward, with the Python function's backward 175 us, 114 with this one: on
// the autograd engine's own thread the interpreter runs cold.  (An empty Python node's step takes 55.)
struct LinearNode : torch::autograd::Function<LinearNode> {
  static at::Tensor forward(torch::autograd::AutogradContext* ctx, const at::Tensor& x, const at::Tensor& weight,
                            const std::optional<at::Tensor>& bias, const Made& made) {
    (void)weight;
    (void)bias;
    ctx->save_for_backward({made.xt, made.sxt, made.w, made.sw});
    ctx->saved_data["shape"] = x.sizes().vec();
    ctx->saved_data["flags"] = (int64_t)(made.per_tensor | made.pow2 << 1 | made.has_bias << 2 | made.w_transposed << 3);
    return made.y;
  }

  static torch::autograd::variable_list in_python(const at::Tensor& go, const torch::autograd::variable_list& saved,
                                                  const std::vector<int64_t>& shape, int64_t flags) {
    pybind11::gil_scoped_acquire held;
    pybind11::tuple size(shape.size());
    for (size_t i = 0; i < shape.size(); ++i) size[i] = shape[i];
    const pybind11::tuple args = pybind11::make_tuple(go, saved[0], saved[1], saved[2], saved[3], size, bool(flags & 1), bool(flags & 2),
                                                      bool(flags & 4), bool(flags & 8));
    const auto grads = pybind11::reinterpret_steal<pybind11::object>(PyObject_CallObject(backward_function, args.ptr()));
    if (!grads) raise_python_error();
    torch::autograd::variable_list out(4);
    for (int i = 0; i < 3; ++i) {
      const pybind11::object g = pybind11::tuple(grads)[i];
      if (!g.is_none()) out[i] = g.cast<at::Tensor>();
    }
    return out;
  }

  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const at::Tensor &xt = saved[0], &sxt = saved[1], &w = saved[2], &sw = saved[3];
    const int64_t flags = ctx->saved_data["flags"].toInt();
    const bool per_tensor = flags & 1, pow2 = flags & 2, has_bias = flags & 4, w_transposed = flags & 8;
    const std::vector<int64_t> shape = ctx->saved_data["shape"].toIntVector();
    // Under a dispatch mode (the engine carries the program's into its threads), and for anything but ordinary tensors where the kernels
    // read them, the Python function answers.
    if (!no_modes() || at::isTensorSubclassLike(grads[0])) return in_python(grads[0], saved, shape, flags);
    at::Tensor go = grads[0];
    if (go.dim() != 2) go = go.reshape({-1, go.size(-1)});
    if (go.scalar_type() != at::kBFloat16) go = go.to(at::kBFloat16);
    go = go.contiguous();
    const int64_t m = go.size(0), mp = rows_up(m), out = go.size(1), in = shape.back();
    bool as_made = go.is_cuda() && go.layout() == at::kStrided;
    if (per_tensor)
      as_made = as_made && codes_again(xt, go, in, mp) && codes_again(w, go, w_transposed ? in : out, w_transposed ? out : in) &&
                sxt.numel() == 1 && floats_again(sxt, go, sxt.sizes()) && sw.numel() == 1 && floats_again(sw, go, sw.sizes());
    else
      as_made = as_made && codes_again(xt, go, in, mp) && codes_again(w, go, in, out) && floats_again(sxt, go, {in, mp / kBlock}) &&
                floats_again(sw, go, {out / kBlock, in / kBlock});
    if (!as_made) return in_python(grads[0], saved, shape, flags);
    const c10::hip::HIPStream current = c10::hip::getCurrentHIPStream(go.get_device());
    void* const stream = current.stream();
    Call call;
    at::Tensor dx, dw, db;
    if (per_tensor) {
      Forms f = make_per_tensor(go, has_bias, sync_block(go, mp / kBlock * (out / kBlock), current.stream()), stream, call);
      if (!call.ok()) raise(call);
      at::Tensor wt = w;
      if (!w_transposed) {
        wt = new_codes_t(w, w.size(1), w.size(0));
        HPFP8_CALL(call, hpfp8_transpose_codes, w.data_ptr(), w.size(0), w.size(1), row_stride(w), wt.data_ptr(), wt.stride(0), stream);
        if (!call.ok()) raise(call);
      }
      dx = multiply_per_tensor(f.q, f.s, wt, sw, nullptr, stream, call);
      if (!call.ok()) raise(call);
      dw = multiply_per_tensor(f.qt, f.s, xt, sxt, nullptr, stream, call);
      db = std::move(f.total);
    } else {
      Forms f = make_both(go, pow2, has_bias, stream, call);
      if (!call.ok()) raise(call);
      // dx[M, K] = go[M, N] . W[N, K]: b operand = W^T codes [K, N], its 128x128 scales W's with the two strides swapped
      dx = at::empty({m, in}, go.options());
      multiply_blockwise(f.q, f.s, w, sw, sw.stride(1), sw.stride(0), nullptr, dx, kBlock, false, pow2, stream, call);
      if (!call.ok()) raise(call);
      // dW[N, K] = go^T[N, M] . x[M, K]: contraction over the tokens
      dw = at::empty({out, in}, go.options());
      at::Tensor scales = sxt;           // per row, in the kernel's layout
      if (!row_scales_fit(scales)) scales = scales.t().contiguous().t();
      multiply_blockwise(f.qt, f.st, xt, scales, scales.stride(0), scales.stride(1), nullptr, dw, 1, false, pow2, stream, call);
      db = std::move(f.total);
    }
    if (!call.ok()) raise(call);
    if (shape.size() != 2) dx = dx.view(shape);
    return {dx, dw, db, at::Tensor()};
  }
};

// (x, weight, bias, codes, scale_inv, codes_t of the weight; None from the bias on) -> whether linear_node takes them: ordinary tensors,
// x and weight trained, no mode, trace or transform under way that a Python autograd function would answer in its own way (or refuse).
PyObject* trains(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 6);
  const at::Tensor *x, *weight, *bias = nullptr, *form;
  if (!c10::GradMode::is_enabled() || !THPVariable_Check(args[0]) || !THPVariable_Unpack(args[0]).is_cuda()) Py_RETURN_FALSE;
  const int64_t device = THPVariable_Unpack(args[0]).get_device();
  if (!plain(args[0], device, x) || !plain(args[1], device, weight) || (args[2] != Py_None && !plain(args[2], device, bias))) Py_RETURN_FALSE;
  for (int i = 3; i < 6; ++i)
    if (args[i] != Py_None && !plain(args[i], device, form)) Py_RETURN_FALSE;
  const bool ok = x->requires_grad() && weight->requires_grad() && x->dim() >= 2 && x->numel() > 0 && weight->numel() > 0 && no_modes() &&
                  !torch::jit::tracer::isTracing() && !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
                  !x->_fw_grad(0).defined() && !weight->_fw_grad(0).defined() && !(bias && bias->_fw_grad(0).defined());
  return PyBool_FromLong(ok);
  END_HANDLE_TH_ERRORS
}

// (x, weight, bias or None, y, xt, sxt, w, sw, per_tensor, pow2, w_transposed) -> y with its place in the graph
PyObject* linear_node(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 11);
  TORCH_CHECK_TYPE(THPVariable_Check(args[0]) && THPVariable_Check(args[1]), "tensors expected");
  const at::Tensor &x = THPVariable_Unpack(args[0]), &weight = THPVariable_Unpack(args[1]);
  const at::Tensor* const bias = args[2] == Py_None ? nullptr : &THPVariable_Unpack(args[2]);
  const at::Tensor* t[5];
  for (int i = 0; i < 5; ++i) TORCH_CHECK_TYPE(plain(args[3 + i], x.get_device(), t[i]), "tensors on ", x.device(), " expected");
  const Made made{*t[0], *t[1], *t[2], *t[3], *t[4], truth(args[8]), truth(args[9]), bias != nullptr, truth(args[10])};
  return THPVariable_Wrap(LinearNode::apply(x, weight, bias ? std::optional<at::Tensor>(*bias) : std::nullopt, made));
  END_HANDLE_TH_ERRORS
}

// (handle of the loaded library, function that raises for a name and a status, torch.nn.Parameter)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 3);
  void* const handle = PyLong_AsVoidPtr(args[0]);
  if (PyErr_Occurred()) throw python_error();
#define HPFP8_LOOK_UP(function) \
  lib.function = (decltype(lib.function))dlsym(handle, #function); \
  TORCH_CHECK(lib.function, "the library has no " #function);
  HPFP8_FUNCTIONS(HPFP8_LOOK_UP)
#undef HPFP8_LOOK_UP
  Py_INCREF(args[1]);
  fail_function = args[1];
  Py_INCREF(args[2]);
  parameter_class = args[2];
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// -> the torch, C++ ABI and interpreter that this module was built for (hpfp8/_lib.py native_tag)
PyObject* built_for(PyObject*, PyObject* const*, Py_ssize_t) { return PyUnicode_FromString(HPFP8_BUILT_FOR); }

// (the Python function that LinearNode's backward calls where it does not apply itself)
PyObject* bind_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 1);
  Py_INCREF(args[0]);
  backward_function = args[0];
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

#define HPFP8_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {HPFP8_METHOD(built_for), HPFP8_METHOD(bind), HPFP8_METHOD(bind_backward), HPFP8_METHOD(quantize_1x128), HPFP8_METHOD(both_forms),
                         HPFP8_METHOD(quantize_128x128), HPFP8_METHOD(quantize_per_tensor_t), HPFP8_METHOD(gemm_blockwise),
                         HPFP8_METHOD(gemm_per_tensor), HPFP8_METHOD(trains), HPFP8_METHOD(linear_node),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
