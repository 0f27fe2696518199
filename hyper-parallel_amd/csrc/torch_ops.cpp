// The tensor operators of hpfp8/ops.py that a linear layer's step is made of, from Python straight to the C ABI of libhpfp8.so.
//
// A small layer's step is bound by the host: through Python a launch costs 10 to 24 us (outputs allocated one by one and turned
// into views, arguments checked, a ctypes call), of which the launch itself is 3.  Each function here does the same for the
// plain case -- ordinary tensors of the types and layouts that the kernels take -- and returns None for everything else,
// refused calls among them: the Python form of the operator then runs as if this one were not there, and copies, pads or raises.
// Host time of a call, us, Python form / here: quantize_1x128 10.5 / 5.3, both forms 15.9 / 7.8, with the bias gradient 24.4 / 12.1,
// 128 x 128 with the transposed codes 12.7 / 6.4, gemm_blockwise 12.2 / 4.9.
// What a program calls many times for little work goes in one call: a layer in inference, operators one by one / here, linear 16 / 11,
// per tensor 23 / 11.5, the MLP block 30 to 35 / 16 to 20, the grouped linear 23 / 12; the forward of a training step, per tensor 26 / 18;
// the gradient bucket there and back, 72 gradients, 67 / 15.
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
  X(hpfp8_quantize_per_tensor_t_bf16) X(hpfp8_transpose_codes) X(hpfp8_gemm_blockwise) X(hpfp8_gemm_blockwise_pow2) X(hpfp8_gemm_per_tensor) \
  X(hpfp8_quantize_per_tensor_sync_bf16) X(hpfp8_gemm_few_rows) X(hpfp8_linear_few_rows) X(hpfp8_linear_few_rows_bf16) X(hpfp8_linear_backward) X(hpfp8_quantize_two_per_tensor_t_bf16) X(hpfp8_gemm_blockwise_swiglu_quantize) X(hpfp8_swiglu_quantize_1x128_bf16) \
  X(hpfp8_swiglu_quantize_1x128_pow2_bf16) X(hpfp8_swiglu_quantize_1x128_fast_bf16) X(hpfp8_gemm_grouped_blockwise) \
  X(hpfp8_bucket_pack_quantize_bf16) X(hpfp8_bucket_unpack_dequantize_bf16)
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

struct Rows {
  at::Tensor q, s;        // codes, scale_inv stored k-block-major
};
// the 1x128 form of m rows of k values
Rows make_rows(const at::Tensor& x, int64_t m, int64_t k, bool pow2, void* stream, Call& call) {
  Rows r{new_codes(x, m, k), new_floats_t(x, m, k / kBlock)};
  if (pow2) HPFP8_CALL(call, hpfp8_quantize_1x128_kmajor_pow2_bf16, x.data_ptr(), m, k, r.q.data_ptr(), nullptr, f32(r.s), stream);
  else HPFP8_CALL(call, hpfp8_quantize_1x128_kmajor_bf16, x.data_ptr(), m, k, r.q.data_ptr(), nullptr, f32(r.s), stream);
  return r;
}

// (x, pow2, device, stream) -> (codes, scale_inv), k-block-major scales
PyObject* quantize_1x128(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  expect(n, 4);
  const Where w = where(args, n);
  const bool pow2 = truth(args[1]);
  const at::Tensor* x;
  if (!source_2d(args[0], w.device, x) || !no_modes()) Py_RETURN_NONE;
  Rows r;
  Call call;
  {
    pybind11::gil_scoped_release free;
    r = make_rows(*x, x->size(0), x->size(1), pow2, w.stream, call);
  }
  return call.ok() ? tuple_of(std::move(r.q), std::move(r.s)) : failed(call);
  END_HANDLE_TH_ERRORS
}

// Both operand forms of x from one read of it, and the sum over its rows; any number of rows.
struct Forms {
  at::Tensor q, s, qt, st, total;        // (per tensor: s is the one scale, st undefined)
  at::Tensor part;                       // the sum's parts, where it is left to linear_backward
};
Forms make_both(const at::Tensor& x, bool pow2, bool column_sum, void* stream, Call& call, bool finish = true) {
  const int64_t m = x.size(0), k = x.size(1), mp = rows_up(m);
  Forms f;
  f.q = new_codes(x, m, k);
  f.qt = new_codes_t(x, k, mp);
  f.s = new_floats_t(x, m, k / kBlock);
  f.st = new_floats_t(x, k, mp / kBlock);
  at::Tensor& part = f.part;
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
  if (column_sum) f.total = at::empty({k}, x.options());
  if (column_sum && finish && call.ok()) {
    HPFP8_CALL(call, hpfp8_column_sum_finish, f32(part), mp / kBlock, k, f.total.data_ptr(), nullptr, stream);
  }
  return f;
}

// The same with one scale; sync: the block through which the one-launch form's grid agrees on the maximum, or null.
Forms make_per_tensor(const at::Tensor& x, bool column_sum, uint32_t* sync, void* stream, Call& call, bool finish = true) {
  const int64_t m = x.size(0), k = x.size(1), mp = rows_up(m);
  Forms f;
  f.q = new_codes(x, m, k);
  f.qt = new_codes_t(x, k, mp);
  f.s = at::empty({}, x.options().dtype(at::kFloat));
  at::Tensor &part = f.part, amax;
  if (column_sum) part = new_floats(x, mp / kBlock, k);
  if (!sync) amax = at::empty({}, x.options().dtype(at::kFloat));
  HPFP8_CALL(call, hpfp8_quantize_per_tensor_t_bf16, x.data_ptr(), m, k, f.q.data_ptr(), f.qt.data_ptr(), f.qt.stride(0),
             sync ? nullptr : f32(amax), nullptr, f32(f.s), sync, column_sum ? f32(part) : nullptr, stream);
  if (column_sum) f.total = at::empty({k}, x.options());
  if (column_sum && finish && call.ok()) {
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
constexpr int64_t kOnePassTiles = 256, kOnePassValues = (int64_t)1 << 22;
uint32_t* sync_block(const at::Tensor& x, bool one_pass, hipStream_t stream) {
  if (!one_pass || c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return nullptr;
  static std::mutex lock;
  static auto* const blocks = new std::map<std::pair<int64_t, hipStream_t>, at::Tensor>;      // (never destroyed: the device may go first)
  std::lock_guard<std::mutex> guard(lock);
  at::Tensor& t = (*blocks)[{x.get_device(), stream}];
  if (!t.defined()) t = at::zeros({256}, x.options().dtype(at::kInt));       // (512 bytes; two tensors at once: the other 512 too)
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

hpfp8_operand operand(const at::Tensor& codes, const at::Tensor& scale_inv) {
  const bool one = scale_inv.dim() != 2;
  return {codes.data_ptr(), row_stride(codes), f32(scale_inv), one ? 0 : scale_inv.stride(0), one ? 0 : scale_inv.stride(1)};
}

// (go, sgo, wt, swt, go_t, sgo_t, xt, sxt, main gradient or None, pow2, device, stream) -> (dx, dw): both products of a blockwise backward;
// swt the weight's scales [K / 128, N / 128], main gradient: fp32 [N, K] that dw is added onto (and is then the same tensor).
PyObject* linear_backward(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  expect(n_args, 12);
  const Where at_ = where(args, n_args);
  const bool pow2 = truth(args[9]);
  const at::Tensor *q[4], *s[4], *given = nullptr;
  for (int i = 0; i < 4; ++i)
    if (!codes_2d(args[2 * i], at_.device, q[i]) || !floats(args[2 * i + 1], at_.device, s[i]) || s[i]->dim() != 2) Py_RETURN_NONE;
  const int64_t m = q[0]->size(0), n = q[0]->size(1), k = q[1]->size(0), mp = rows_up(m);
  const int64_t rows[] = {m, k / kBlock, n, k}, blocks[] = {n / kBlock, n / kBlock, mp / kBlock, mp / kBlock};
  for (int i = 0; i < 4; ++i)
    if (s[i]->size(0) != rows[i] || s[i]->size(1) != blocks[i]) Py_RETURN_NONE;
  if (k % kBlock || q[1]->size(1) != n || q[2]->size(0) != n || q[2]->size(1) != mp || q[3]->size(0) != k || q[3]->size(1) != mp || !row_scales_fit(*s[3]) ||
      !no_modes())
    Py_RETURN_NONE;
  if (args[8] != Py_None && (!plain(args[8], at_.device, given) || given->scalar_type() != at::kFloat || given->dim() != 2 || given->size(0) != n ||
                             given->size(1) != k || !given->is_contiguous()))
    Py_RETURN_NONE;
  at::Tensor dx, dw;
  Call call;
  {
    pybind11::gil_scoped_release free;
    dx = at::empty({m, k}, q[0]->options().dtype(at::kBFloat16));
    dw = given ? *given : at::empty({n, k}, dx.options());
    const hpfp8_operand a = operand(*q[0], *s[0]), b = operand(*q[1], *s[1]), at = operand(*q[2], *s[2]), bt = operand(*q[3], *s[3]);
    HPFP8_CALL(call, hpfp8_linear_backward, &a, &b, &at, &bt, m, n, k, dx.data_ptr(), dw.data_ptr(), given != nullptr, nullptr, nullptr,
               pow2 ? HPFP8_BLOCKWISE_POW2 : HPFP8_BLOCKWISE, at_.stream);
  }
  return call.ok() ? tuple_of(std::move(dx), std::move(dw)) : failed(call);
  END_HANDLE_TH_ERRORS
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
      Forms f = make_per_tensor(go, has_bias, sync_block(go, mp / kBlock * (out / kBlock) <= kOnePassTiles, current.stream()), stream, call, false);
      if (!call.ok()) raise(call);
      at::Tensor wt = w;
      if (!w_transposed) {
        wt = new_codes_t(w, w.size(1), w.size(0));
        HPFP8_CALL(call, hpfp8_transpose_codes, w.data_ptr(), w.size(0), w.size(1), row_stride(w), wt.data_ptr(), wt.stride(0), stream);
        if (!call.ok()) raise(call);
      }
      dx = at::empty({m, in}, go.options());
      dw = at::empty({out, in}, go.options());
      const hpfp8_operand a = operand(f.q, f.s), b = operand(wt, sw), at = operand(f.qt, f.s), bt = operand(xt, sxt);
      HPFP8_CALL(call, hpfp8_linear_backward, &a, &b, &at, &bt, m, out, in, dx.data_ptr(), dw.data_ptr(), 0, has_bias ? f32(f.part) : nullptr,
                 has_bias ? f.total.data_ptr() : nullptr, HPFP8_PER_TENSOR, stream);
      db = std::move(f.total);
    } else {
      Forms f = make_both(go, pow2, has_bias, stream, call, false);
      if (!call.ok()) raise(call);
      // dx[M, K] = go[M, N] . W[N, K]: b operand = W^T codes [K, N], its 128x128 scales W's with the two strides swapped
      dx = at::empty({m, in}, go.options());
      // dW[N, K] = go^T[N, M] . x[M, K]: contraction over the tokens
      dw = at::empty({out, in}, go.options());
      at::Tensor scales = sxt;           // per row, in the kernel's layout
      if (!row_scales_fit(scales)) scales = scales.t().contiguous().t();
      const hpfp8_operand a = operand(f.q, f.s), b{w.data_ptr(), row_stride(w), f32(sw), sw.stride(1), sw.stride(0)};
      const hpfp8_operand at = operand(f.qt, f.st), bt = operand(xt, scales);
      HPFP8_CALL(call, hpfp8_linear_backward, &a, &b, &at, &bt, m, out, in, dx.data_ptr(), dw.data_ptr(), 0, has_bias ? f32(f.part) : nullptr,
                 has_bias ? f.total.data_ptr() : nullptr, pow2 ? HPFP8_BLOCKWISE_POW2 : HPFP8_BLOCKWISE, stream);
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

// ------------------------------------------------------------------------------------------------
// inference: a layer's steps in one call
// ------------------------------------------------------------------------------------------------
// A layer's input: bf16 [..., K > 0, a multiple of 128], contiguous, with rows.
bool layer_input(PyObject* o, int64_t device, const at::Tensor*& t) {
  return plain(o, device, t) && t->scalar_type() == at::kBFloat16 && t->dim() >= 1 && t->numel() > 0 && t->size(-1) % kBlock == 0 &&
         t->is_contiguous();
}
// Whether a call on these (None among them) is one without a graph, trace or transform, which a Python autograd function would answer
// in its own way.
bool without_graph(PyObject* const* tensors, int n) {
  if (!no_modes() || torch::jit::tracer::isTracing() || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode))
    return false;
  const bool grad = c10::GradMode::is_enabled();
  for (int i = 0; i < n; ++i) {
    if (tensors[i] == Py_None) continue;
    if (!THPVariable_Check(tensors[i])) return false;
    const at::Tensor& t = THPVariable_Unpack(tensors[i]);
    if (at::isTensorSubclassLike(t) || (grad && t.requires_grad()) || t._fw_grad(0).defined()) return false;
  }
  return true;
}
at::Tensor new_rows_like(const at::Tensor& x, int64_t n) {
  std::vector<int64_t> shape = x.sizes().vec();
  shape.back() = n;
  return at::empty(shape, x.options().requires_grad(false));
}
bool weight_form(PyObject* codes, PyObject* scale_inv, int64_t device, const at::Tensor*& q, const at::Tensor*& s) {
  return codes_2d(codes, device, q) && floats(scale_inv, device, s) && q->size(0) % kBlock == 0 && s->dim() == 2 &&
         s->size(0) == q->size(0) / kBlock && s->size(1) == q->size(1) / kBlock;
}
// c[m rows, n] = rows . weight^T (+ bias); c of any shape with n as its last, contiguous
void multiply_rows(const Rows& r, const at::Tensor& w, const at::Tensor& sw, const void* bias, const at::Tensor& c, bool pow2, void* stream, Call& call) {
  const int64_t m = r.q.size(0), k = r.q.size(1), n = w.size(0);
  if (pow2)
    HPFP8_CALL(call, hpfp8_gemm_blockwise_pow2, r.q.data_ptr(), k, f32(r.s), r.s.stride(0), r.s.stride(1), w.data_ptr(), row_stride(w), f32(sw),
               sw.stride(0), sw.stride(1), (int)kBlock, m, n, k, bias, c.data_ptr(), n, HPFP8_OUT_BF16, 0, stream);
  else
    HPFP8_CALL(call, hpfp8_gemm_blockwise, r.q.data_ptr(), k, f32(r.s), r.s.stride(0), r.s.stride(1), w.data_ptr(), row_stride(w), f32(sw),
               sw.stride(0), sw.stride(1), (int)kBlock, m, n, k, bias, c.data_ptr(), n, HPFP8_OUT_BF16, 0, stream);
}

// c = x . weight^T (+ bias) of m rows of bf16, quantized here or, where that is the better form, inside the product.
void multiply_source(const at::Tensor& x, int64_t m, int64_t k, const at::Tensor& w, const at::Tensor& sw, const void* bias, const at::Tensor& c, bool pow2,
                     void* stream, Call& call) {
  if (m <= lib.hpfp8_linear_few_rows(w.size(0), k) && (uintptr_t)x.data_ptr() % 16 == 0) {
    HPFP8_CALL(call, hpfp8_linear_few_rows_bf16, x.data_ptr(), w.data_ptr(), row_stride(w), f32(sw), sw.stride(0), sw.stride(1), m, w.size(0), k, pow2,
               bias, c.data_ptr(), w.size(0), HPFP8_OUT_BF16, stream);
    return;
  }
  const Rows r = make_rows(x, m, k, pow2, stream, call);
  if (call.ok()) multiply_rows(r, w, sw, bias, c, pow2, stream, call);
}

// (x, weight, bias or None, the weight's codes, scale_inv, codes_t or None each, per_tensor, pow2, device, stream) -> y with its place in
// the graph: forward of what `trains` has taken (hpfp8/linear.py _trained) in one call.  A blockwise weight that has no FP8 form yet is
// left to the operators one by one (quantizing it dominates such a step).
PyObject* linear_train(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  expect(n_args, 10);
  const Where at_ = where(args, n_args);
  const bool per_tensor = truth(args[6]), pow2 = truth(args[7]);
  const at::Tensor *x, *weight, *bias, *wq = nullptr, *sw = nullptr, *wqt = nullptr;
  if (!layer_input(args[0], at_.device, x) || x->dim() < 2 || !source_2d(args[1], at_.device, weight)) Py_RETURN_NONE;
  const int64_t k = x->size(-1), m = x->numel() / k, n = weight->size(0);
  if (weight->size(1) != k || n % kBlock || !bias_of(args[2], at_.device, n, bias) || (args[3] == Py_None && !per_tensor)) Py_RETURN_NONE;
  if (args[3] != Py_None) {
    if (!codes_2d(args[3], at_.device, wq) || wq->size(0) != n || wq->size(1) != k || !floats(args[4], at_.device, sw)) Py_RETURN_NONE;
    if (per_tensor ? sw->numel() != 1 : (sw->dim() != 2 || sw->size(0) != n / kBlock || sw->size(1) != k / kBlock)) Py_RETURN_NONE;
    if (!per_tensor && args[5] != Py_None && (!codes_2d(args[5], at_.device, wqt) || wqt->size(0) != k || wqt->size(1) != n)) Py_RETURN_NONE;
  }
  Made made{{}, {}, {}, {}, {}, per_tensor, pow2, bias != nullptr, true};
  Call call;
  {
    pybind11::gil_scoped_release free;
    at::NoGradGuard no_grad;
    void* const stream = at_.stream;
    const at::Tensor x2 = x->dim() == 2 ? *x : x->view({m, k});
    auto transposed = [&](const at::Tensor& codes) {
      at::Tensor t = new_codes_t(codes, k, n);
      HPFP8_CALL(call, hpfp8_transpose_codes, codes.data_ptr(), n, k, row_stride(codes), t.data_ptr(), t.stride(0), stream);
      return t;
    };
    Forms fx, fw;
    if (per_tensor) {
      const int64_t tiles = rows_up(m) / kBlock * (k / kBlock);
      const int64_t w_tiles = n / kBlock * (k / kBlock);
      uint32_t* const sync = sync_block(x2, tiles <= kOnePassTiles, (hipStream_t)stream);
      if (sync && !wq && w_tiles <= kOnePassTiles) {
        for (Forms* f : {&fx, &fw}) {
          const int64_t rows = f == &fx ? m : n;
          f->q = new_codes(x2, rows, k);
          f->qt = new_codes_t(x2, k, rows_up(rows));
          f->s = at::empty({}, x2.options().dtype(at::kFloat).requires_grad(false));
        }
        HPFP8_CALL(call, hpfp8_quantize_two_per_tensor_t_bf16, x2.data_ptr(), m, k, fx.q.data_ptr(), fx.qt.data_ptr(), fx.qt.stride(0), f32(fx.s),
                   weight->data_ptr(), n, fw.q.data_ptr(), fw.qt.data_ptr(), fw.qt.stride(0), f32(fw.s), sync, stream);
      } else {
        fx = make_per_tensor(x2, false, sync, stream, call);
      }
      if (call.ok() && !wq && !fw.q.defined()) fw = make_per_tensor(*weight, false, sync_block(*weight, w_tiles <= kOnePassTiles, (hipStream_t)stream), stream, call);
      made.w_transposed = !wq;
      made.w = wq ? *wq : fw.qt;
      made.sw = wq ? *sw : fw.s;
      made.xt = fx.qt;
      made.sxt = fx.s;
      if (call.ok()) made.y = multiply_per_tensor(fx.q, fx.s, wq ? *wq : fw.q, made.sw, bias ? bias->data_ptr() : nullptr, stream, call);
    } else {
      fx = make_both(x2, pow2, false, stream, call);
      if (call.ok()) {
        made.w = wqt ? *wqt : transposed(*wq);
        made.sw = *sw;
      }
      made.xt = fx.qt;
      made.sxt = fx.st;
      if (call.ok()) {
        made.y = at::empty({m, n}, x->options().requires_grad(false));
        multiply_blockwise(fx.q, fx.s, *wq, made.sw, made.sw.stride(0), made.sw.stride(1), bias ? bias->data_ptr() : nullptr, made.y, kBlock,
                           false, pow2, stream, call);
      }
    }
    if (call.ok() && x->dim() != 2) {
      std::vector<int64_t> shape = x->sizes().vec();
      shape.back() = n;
      made.y = made.y.view(shape);
    }
  }
  if (!call.ok()) return failed(call);
  return THPVariable_Wrap(LinearNode::apply(*x, *weight, bias ? std::optional<at::Tensor>(*bias) : std::nullopt, made));
  END_HANDLE_TH_ERRORS
}

// (x, weight, bias or None, codes, scale_inv, per_tensor, pow2, device, stream) -> y
PyObject* linear_infer(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  expect(n_args, 9);
  const Where at_ = where(args, n_args);
  const bool per_tensor = truth(args[5]), pow2 = truth(args[6]);
  const at::Tensor *x, *w, *sw, *bias;
  if (!without_graph(args, 3) || !layer_input(args[0], at_.device, x) || !codes_2d(args[3], at_.device, w) || !floats(args[4], at_.device, sw))
    Py_RETURN_NONE;
  const int64_t k = x->size(-1), m = x->numel() / k, n = w->size(0);
  if (w->size(1) != k || n % kBlock || !bias_of(args[2], at_.device, n, bias)) Py_RETURN_NONE;
  if (per_tensor ? sw->numel() != 1 : !weight_form(args[3], args[4], at_.device, w, sw)) Py_RETURN_NONE;
  at::Tensor y;
  Call call;
  bool taken = true;
  {
    pybind11::gil_scoped_release free;
    const void* const b = bias ? bias->data_ptr() : nullptr;
    if (per_tensor) {
      uint32_t* const sync = sync_block(*x, x->numel() <= kOnePassValues, (hipStream_t)at_.stream);
      taken = sync != nullptr;       // (larger ones, and all under capture, take two launches: the Python form)
      if (taken) {
        const at::Tensor q = new_codes(*x, m, k), s = at::empty({}, x->options().dtype(at::kFloat).requires_grad(false));
        HPFP8_CALL(call, hpfp8_quantize_per_tensor_sync_bf16, x->data_ptr(), x->numel(), q.data_ptr(), nullptr, nullptr, f32(s), sync, at_.stream);
        if (call.ok()) {
          y = new_rows_like(*x, n);
          HPFP8_CALL(call, hpfp8_gemm_per_tensor, q.data_ptr(), k, f32(s), w->data_ptr(), row_stride(*w), f32(*sw), m, n, k, b, y.data_ptr(), n,
                     HPFP8_OUT_BF16, at_.stream);
        }
      }
    } else {
      y = new_rows_like(*x, n);
      multiply_source(*x, m, k, *w, *sw, b, y, pow2, at_.stream, call);
    }
  }
  if (!taken) Py_RETURN_NONE;
  return call.ok() ? THPVariable_Wrap(std::move(y)) : failed(call);
  END_HANDLE_TH_ERRORS
}

// (x, gate/up codes, scale_inv, pow2, down codes, scale_inv, pow2, fast, device, stream) -> y
PyObject* swiglu_mlp_infer(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  expect(n_args, 10);
  const Where at_ = where(args, n_args);
  const bool pow2 = truth(args[3]), pow2_down = truth(args[6]), fast = truth(args[7]);
  const at::Tensor *x, *gu, *sgu, *dn, *sdn;
  if (!no_modes() || !layer_input(args[0], at_.device, x) || !weight_form(args[1], args[2], at_.device, gu, sgu) ||
      !weight_form(args[4], args[5], at_.device, dn, sdn))
    Py_RETURN_NONE;
  const int64_t k = x->size(-1), m = x->numel() / k, n = gu->size(0), inter = n / 2;
  if (gu->size(1) != k || n % (2 * kBlock) || dn->size(1) != inter) Py_RETURN_NONE;
  at::Tensor y;
  Call call;
  {
    pybind11::gil_scoped_release free;
    // (ops.gemm_blockwise_swiglu_quantize has the reason for the two forms)
    const bool two_steps = m <= lib.hpfp8_gemm_few_rows(k) && n * row_stride(*gu) < 0x7FFFF000;
    Rows r, a;
    if (!two_steps) r = make_rows(*x, m, k, pow2, at_.stream, call);
    if (call.ok()) {
      a = Rows{new_codes(*x, m, inter), new_floats_t(*x, m, inter / kBlock)};
      if (two_steps) {
        const at::Tensor h = at::empty({m, n}, x->options().requires_grad(false));
        multiply_source(*x, m, k, *gu, *sgu, nullptr, h, pow2, at_.stream, call);
        if (call.ok()) {
          if (fast)
            HPFP8_CALL(call, hpfp8_swiglu_quantize_1x128_fast_bf16, h.data_ptr(), m, inter, n, 1, pow2_down, a.q.data_ptr(), nullptr, f32(a.s), nullptr, at_.stream);
          else if (pow2_down)
            HPFP8_CALL(call, hpfp8_swiglu_quantize_1x128_pow2_bf16, h.data_ptr(), m, inter, n, 1, a.q.data_ptr(), nullptr, f32(a.s), nullptr, at_.stream);
          else
            HPFP8_CALL(call, hpfp8_swiglu_quantize_1x128_bf16, h.data_ptr(), m, inter, n, 1, a.q.data_ptr(), nullptr, f32(a.s), nullptr, at_.stream);
        }
      } else {
        HPFP8_CALL(call, hpfp8_gemm_blockwise_swiglu_quantize, r.q.data_ptr(), k, f32(r.s), r.s.stride(0), r.s.stride(1), gu->data_ptr(), row_stride(*gu),
                   f32(*sgu), sgu->stride(0), sgu->stride(1), m, inter, k, fast, pow2, pow2_down, a.q.data_ptr(), inter, nullptr, f32(a.s), at_.stream);
      }
    }
    if (call.ok()) {
      y = new_rows_like(*x, dn->size(0));
      multiply_rows(a, *dn, *sdn, nullptr, y, pow2_down, at_.stream, call);
    }
  }
  return call.ok() ? THPVariable_Wrap(std::move(y)) : failed(call);
  END_HANDLE_TH_ERRORS
}

// (x, weight, offs, codes, scale_inv, device, stream) -> y
PyObject* grouped_infer(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  expect(n_args, 7);
  const Where at_ = where(args, n_args);
  const at::Tensor *x, *offs, *w, *sw;
  if (!without_graph(args, 3) || !layer_input(args[0], at_.device, x) || x->dim() != 2 || !plain(args[2], at_.device, offs) || !plain(args[3], at_.device, w) ||
      !floats(args[4], at_.device, sw))
    Py_RETURN_NONE;
  const int64_t m = x->size(0), k = x->size(1);
  if (w->dim() != 3 || w->scalar_type() != at::kFloat8_e4m3fn || !w->is_contiguous() || w->size(2) != k || w->size(1) % kBlock || w->numel() == 0 ||
      offs->scalar_type() != at::kInt || offs->dim() != 1 || !offs->is_contiguous() || offs->size(0) != w->size(0) || !sw->is_contiguous() ||
      sw->sizes() != at::IntArrayRef({w->size(0), w->size(1) / kBlock, k / kBlock}))
    Py_RETURN_NONE;
  at::Tensor y;
  Call call;
  {
    pybind11::gil_scoped_release free;
    const Rows r = make_rows(*x, m, k, false, at_.stream, call);
    if (call.ok()) {
      const int64_t n = w->size(1);
      y = new_rows_like(*x, n);
      HPFP8_CALL(call, hpfp8_gemm_grouped_blockwise, r.q.data_ptr(), k, f32(r.s), r.s.stride(0), r.s.stride(1), w->data_ptr(), f32(*sw),
                 offs->data_ptr<int32_t>(), (int)w->size(0), m, n, k, y.data_ptr(), n, HPFP8_OUT_BF16, at_.stream);
    }
  }
  return call.ok() ? THPVariable_Wrap(std::move(y)) : failed(call);
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------------------------------------
// the gradient bucket
// ------------------------------------------------------------------------------------------------
// A table of int64 (an array of ctypes, held by the bucket) while a call lasts.
struct Table {
  Py_buffer view{};
  bool held;
  Table(PyObject* o, int64_t count) : held(PyObject_GetBuffer(o, &view, PyBUF_SIMPLE) == 0) {
    if (!held) throw python_error();
    TORCH_CHECK_TYPE(view.len >= count * 8, "a table of ", count, " entries expected");
  }
  ~Table() {
    if (held) PyBuffer_Release(&view);
  }
  Table(const Table&) = delete;
  const int64_t* data() const { return (const int64_t*)view.buf; }
};
// The addresses of a list or tuple of contiguous bf16 tensors of numels[i] * times elements; nothing where one is anything else.
bool gradients(PyObject* o, int64_t device, const int64_t* numels, int64_t count, int64_t times, std::vector<void*>& ptrs) {
  if (!(PyList_CheckExact(o) || PyTuple_CheckExact(o)) || PySequence_Fast_GET_SIZE(o) != count) return false;
  ptrs.resize(count);
  for (int64_t i = 0; i < count; ++i) {
    const at::Tensor* t;
    if (!plain(PySequence_Fast_GET_ITEM(o, i), device, t) || t->scalar_type() != at::kBFloat16 || !t->is_contiguous() || t->numel() != numels[i] * times)
      return false;
    ptrs[i] = t->data_ptr();
  }
  return true;
}

// (gradients, numels, offsets, count, shards, row_elems, device, stream) -> (codes, scale_inv)
PyObject* bucket_pack(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  expect(n_args, 8);
  const Where at_ = where(args, n_args);
  const int64_t count = PyLong_AsLongLong(args[3]), shards = PyLong_AsLongLong(args[4]), row = PyLong_AsLongLong(args[5]);
  if (PyErr_Occurred()) throw python_error();
  if (count <= 0 || !no_modes()) Py_RETURN_NONE;
  const Table numels(args[1], count), offsets(args[2], count);
  std::vector<void*> ptrs;
  if (!gradients(args[0], at_.device, numels.data(), count, shards, ptrs)) Py_RETURN_NONE;
  const at::TensorOptions options = THPVariable_Unpack(PySequence_Fast_GET_ITEM(args[0], 0)).options().requires_grad(false);
  const at::Tensor q = at::empty({shards, row}, options.dtype(at::kFloat8_e4m3fn)), s = at::empty({shards, row / kBlock}, options.dtype(at::kFloat));
  Call call;
  {
    pybind11::gil_scoped_release free;
    HPFP8_CALL(call, hpfp8_bucket_pack_quantize_bf16, ptrs.data(), numels.data(), offsets.data(), (int)count, (int)shards, row, q.data_ptr(), nullptr,
               f32(s), at_.stream);
  }
  return call.ok() ? tuple_of(q, s) : failed(call);
  END_HANDLE_TH_ERRORS
}

// (codes_row, scale_inv_row, outs, numels, offsets, count, row_elems, grad_scale, device, stream) -> whether it was done
PyObject* bucket_unpack(PyObject*, PyObject* const* args, Py_ssize_t n_args) {
  HANDLE_TH_ERRORS
  expect(n_args, 10);
  const Where at_ = where(args, n_args);
  const int64_t count = PyLong_AsLongLong(args[5]), row = PyLong_AsLongLong(args[6]);
  const double grad_scale = PyFloat_AsDouble(args[7]);
  if (PyErr_Occurred()) throw python_error();
  const at::Tensor *q, *s;
  if (count <= 0 || !no_modes() || !plain(args[0], at_.device, q) || !floats(args[1], at_.device, s) || q->scalar_type() != at::kFloat8_e4m3fn ||
      q->numel() != row || s->numel() != row / kBlock || !q->is_contiguous() || !s->is_contiguous())
    Py_RETURN_FALSE;
  const Table numels(args[3], count), offsets(args[4], count);
  std::vector<void*> ptrs;
  if (!gradients(args[2], at_.device, numels.data(), count, 1, ptrs)) Py_RETURN_FALSE;
  Call call;
  {
    pybind11::gil_scoped_release free;
    HPFP8_CALL(call, hpfp8_bucket_unpack_dequantize_bf16, ptrs.data(), numels.data(), offsets.data(), (int)count, row, q->data_ptr(), f32(*s),
               (float)grad_scale, at_.stream);
  }
  if (!call.ok()) return failed(call);
  Py_RETURN_TRUE;
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
                         HPFP8_METHOD(gemm_per_tensor), HPFP8_METHOD(trains), HPFP8_METHOD(linear_node), HPFP8_METHOD(linear_train), HPFP8_METHOD(linear_infer), HPFP8_METHOD(linear_backward),
                         HPFP8_METHOD(swiglu_mlp_infer), HPFP8_METHOD(grouped_infer), HPFP8_METHOD(bucket_pack), HPFP8_METHOD(bucket_unpack),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
