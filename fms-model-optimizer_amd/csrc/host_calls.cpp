// The host side of the hot calls: argument checks, output allocation and the launch of one or several entry
// points of libfmsmo_hip.so, from torch tensors, in one call out of Python.
//
// An eager call of a 5 us kernel is bound by what the host does for it: checks and allocations written in
// Python took 13 us around the 4.6 us of the launch (4096 x 4096, one token: 18.8 us a call; with these 5.8 over and over
// on one input, 7.6 ... 8.1 on new ones).
//
// Every function takes the common case only -- plain, well-formed tensors on the current GPU, outside dispatch
// modes and transforms -- and returns None for anything else, which then takes the general path in Python (and
// gets its error messages there).  Nothing is kept from one call to the next.
#include <ATen/ATen.h>
#include <cmath>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include "../../include/fmsmo_hip.h"

namespace {

// ------------------------------------------------------------------ the library's entry points
#define ENTRIES(X)                                                                                       \
  X(fmsmo_quant_act_i8_pertoken) X(fmsmo_quant_act_i8_static) X(fmsmo_quant_act_i8_static_t)             \
  X(fmsmo_quant_act_fp8_pertoken) X(fmsmo_quant_act_fp8_dynamic) X(fmsmo_quant_act_fp8_tensor)           \
  X(fmsmo_quant_act_i8_static_scale) X(fmsmo_quant_act_i8_pertoken_clips) X(fmsmo_gemm_i8_dq_ws) X(fmsmo_gemm_fp8_dq_ws) X(fmsmo_gemm_workspace_bytes)      \
  X(fmsmo_gemm_fp8_workspace_bytes) X(fmsmo_decode_linear_i8) X(fmsmo_decode_linear_fp8)                 \
  X(fmsmo_decode_linear_ok) X(fmsmo_decode_linear_f32s_ok) X(fmsmo_small_linear_better) X(fmsmo_small_linear_i8) X(fmsmo_small_linear_fp8) X(fmsmo_small_linear_static_ok) X(fmsmo_small_linear_i8_static_scale) X(fmsmo_grouped_gemm_i8_dq)                   \
  X(fmsmo_matmul_chunk_i8_dq_ws) X(fmsmo_matmul_chunk_fp_dq) X(fmsmo_matmul_chunk_workspace_bytes)    \
  X(fmsmo_quant_i8_affine_sums) X(fmsmo_quant_i8_affine_pair) X(fmsmo_affine_sum_parts) X(fmsmo_affine_parts_first) X(fmsmo_affine_add_parts) X(fmsmo_bmm_qa_ok)   \
  X(fmsmo_bmm_qa_i8) X(fmsmo_bmm_i8_zp)
#define DECLARE(f) decltype(&::f) p_##f = nullptr;
ENTRIES(DECLARE)
#undef DECLARE
PyObject* g_raise_status = nullptr;  // raise_status(name, code)

PyObject* none() { Py_RETURN_NONE; }

// Calls an entry point without the interpreter lock; a non-zero status leaves the binding's exception set.
template <class F, class... A>
bool launch(const char* name, F f, A... a) {
  PyThreadState* ts = PyEval_SaveThread();
  const int rc = f(a...);
  PyEval_RestoreThread(ts);
  if (rc == 0) return true;
  PyObject* r = PyObject_CallFunction(g_raise_status, "si", name, rc);
  Py_XDECREF(r);
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, name);
  return false;
}
#define LAUNCH(f, ...) launch(#f, p_##f, __VA_ARGS__)

// ------------------------------------------------------------------ what a well-formed argument is
int code_of(at::ScalarType t) {
  return t == at::kHalf ? FMSMO_F16 : t == at::kBFloat16 ? FMSMO_BF16 : t == at::kFloat ? FMSMO_F32 : -1;
}
at::ScalarType promoted(at::ScalarType a, at::ScalarType b) { return a == b ? a : at::kFloat; }

// the tensor of a plain torch.Tensor / Parameter that owns memory on a GPU, else null (subclasses and the
// wrappers of transforms are none)
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || !t.unsafeGetTensorImpl()->has_storage()) return nullptr;
  return &t;
}
struct Mat {
  const at::Tensor* t = nullptr;
  int64_t rows = 0, cols = 0, ld = 0;
  char* p = nullptr;
  explicit operator bool() const { return t != nullptr; }
};
// a 2-D tensor with unit inner stride
Mat mat(PyObject* o) {
  Mat m;
  const at::Tensor* t = plain(o);
  if (!t || t->dim() != 2) return m;
  const int64_t r = t->size(0), c = t->size(1), s0 = t->stride(0);
  if (t->stride(1) != 1 || (r > 1 && s0 < c)) return m;
  return Mat{t, r, c, r > 1 ? s0 : std::max(c, s0), (char*)t->data_ptr()};
}
// [.., K] as rows of K: contiguous, or a matrix as above
Mat rows_of(PyObject* o) {
  const at::Tensor* t = plain(o);
  if (!t || t->dim() == 0) return Mat{};
  if (t->dim() == 2) return mat(o);
  const int64_t K = t->size(-1);
  if (K == 0 || !t->is_contiguous()) return Mat{};
  return Mat{t, t->numel() / K, K, K, (char*)t->data_ptr()};
}
// fp32 vector of n elements or one
const at::Tensor* vec32(PyObject* o, int64_t n) {
  const at::Tensor* t = plain(o);
  if (!t || t->scalar_type() != at::kFloat || t->dim() != 1 || !t->is_contiguous() || t->requires_grad() ||
      (t->numel() != n && t->numel() != 1))
    return nullptr;
  return t;
}
// an optional vector of n 16-bit or fp32 elements
struct Opt {
  bool ok = false;
  void* p = nullptr;
  int dt = 0;
  at::ScalarType st = at::kFloat;
  const at::Tensor* t = nullptr;
};
Opt opt_vec(PyObject* o, int64_t n, int align = 1) {
  Opt r;
  if (o == Py_None) {
    r.ok = true;
    return r;
  }
  const at::Tensor* t = plain(o);
  if (!t || t->dim() != 1 || t->numel() != n || !t->is_contiguous() || code_of(t->scalar_type()) < 0 ||
      (uintptr_t)t->data_ptr() % align)
    return r;
  return Opt{true, t->data_ptr(), code_of(t->scalar_type()), t->scalar_type(), t};
}
bool dtype_arg(PyObject* o, at::ScalarType* st) {
  if (!THPDtype_Check(o)) return false;
  *st = ((THPDtype*)o)->scalar_type;
  return code_of(*st) >= 0;
}
// the call can be made here: every tensor of it (null: an operand left out) on the current device -- a scale on another
// one is the general path's to move -- and no mode that wants to see the allocations
template <class... T>
bool here(const T*... t) {
  const auto d = c10::hip::current_device();
  return !c10::impl::TorchDispatchModeTLS::any_modes_set() && ((!t || t->get_device() == d) && ...);
}
void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
// part of a graph: its launches cost the host nothing when it is replayed
bool capturing(const at::Tensor& t) {
  hipStreamCaptureStatus s = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing((hipStream_t)stream_of(t), &s) == hipSuccess) return s == hipStreamCaptureStatusActive;
  (void)hipGetLastError();
  return false;
}
at::Tensor empty(at::IntArrayRef sizes, at::ScalarType st, const at::Tensor& like) {
  return at::empty(sizes, like.options().dtype(st).requires_grad(false));
}
at::Tensor workspace(int64_t bytes, const at::Tensor& like) {
  return bytes > 0 ? empty({bytes}, at::kByte, like) : at::Tensor();
}
PyObject* wrap(at::Tensor t) { return THPVariable_Wrap(std::move(t)); }
PyObject* wrap2(at::Tensor a, at::Tensor b) {
  PyObject* t = PyTuple_New(2);
  PyTuple_SET_ITEM(t, 0, wrap(std::move(a)));
  PyTuple_SET_ITEM(t, 1, wrap(std::move(b)));
  return t;
}
at::Tensor out_like(const at::Tensor& x, int64_t N, at::ScalarType st) {
  if (x.dim() == 2) return empty({x.size(0), N}, st, x);
  std::vector<int64_t> s(x.sizes().begin(), x.sizes().end());
  s.back() = N;
  return empty(s, st, x);
}
#define WANT(n) \
  if (nargs != (n)) return PyErr_Format(PyExc_TypeError, "%s takes %d arguments", __func__, (int)(n))
#define REAL(i) PyFloat_AsDouble(args[i])
#define WHOLE(i) PyLong_AsLong(args[i])
#define NUMBERS_OK \
  if (PyErr_Occurred()) return PyErr_Clear(), none()

// ------------------------------------------------------------------ quantizers
// (x, smooth | None, compute dtype | None, saturate) -> (q int8 [M,K], scale fp32 [M])
PyObject* quant_i8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(4);
  const Mat x = mat(args[0]);
  if (!x || code_of(x.t->scalar_type()) < 0) return none();
  const Opt sm = opt_vec(args[1], x.cols, 16);
  if (!sm.ok || !here(x.t, sm.t)) return none();
  at::ScalarType ct = sm.p ? promoted(x.t->scalar_type(), sm.st) : x.t->scalar_type();
  if (args[2] != Py_None && !dtype_arg(args[2], &ct)) return none();
  const int sat = PyObject_IsTrue(args[3]);
  at::Tensor q = empty({x.rows, x.cols}, at::kChar, *x.t), s = empty({x.rows}, at::kFloat, *x.t);
  if (!LAUNCH(fmsmo_quant_act_i8_pertoken, x.p, code_of(x.t->scalar_type()), x.ld, sm.p, sm.dt, code_of(ct), sat,
              (int8_t*)q.data_ptr(), x.cols, (float*)s.data_ptr(), x.rows, x.cols, stream_of(*x.t)))
    return nullptr;
  return wrap2(q, s);
  END_HANDLE_TH_ERRORS
}
// int8 codes per token without divisors, scale [M,1] and the clip values [2,M,1]
bool codes_and_clips(const Mat& x, at::Tensor* q, at::Tensor* s, at::Tensor* c) {
  const int dt = code_of(x.t->scalar_type());
  *q = empty({x.rows, x.cols}, at::kChar, *x.t);
  *s = empty({x.rows, 1}, at::kFloat, *x.t);
  *c = empty({2, x.rows, 1}, at::kFloat, *x.t);
  return LAUNCH(fmsmo_quant_act_i8_pertoken_clips, x.p, dt, x.ld, dt, 0, (int8_t*)q->data_ptr(), x.cols,
                (float*)s->data_ptr(), (float*)c->data_ptr(), x.rows, x.cols, stream_of(*x.t));
}
// x -> (q int8 [M,K], scale fp32 [M,1], clip value [M,1], its negative)
PyObject* quant_i8_clips(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(1);
  const Mat x = mat(args[0]);
  if (!x || code_of(x.t->scalar_type()) < 0 || !here(x.t)) return none();
  at::Tensor q, s, c;
  if (!codes_and_clips(x, &q, &s, &c)) return nullptr;
  PyObject* t = PyTuple_New(4);
  PyTuple_SET_ITEM(t, 0, wrap(q));
  PyTuple_SET_ITEM(t, 1, wrap(s));
  PyTuple_SET_ITEM(t, 2, wrap(c.select(0, 0)));
  PyTuple_SET_ITEM(t, 3, wrap(c.select(0, 1)));
  return t;
  END_HANDLE_TH_ERRORS
}
// (x, scale, zp, sym) -> q
PyObject* quant_i8_static(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(4);
  const Mat x = mat(args[0]);
  if (!x || code_of(x.t->scalar_type()) < 0 || !here(x.t)) return none();
  const float scale = (float)REAL(1);
  const int zp = (int)WHOLE(2), sym = (int)WHOLE(3);
  NUMBERS_OK;
  at::Tensor q = empty({x.rows, x.cols}, at::kChar, *x.t);
  if (!LAUNCH(fmsmo_quant_act_i8_static, x.p, code_of(x.t->scalar_type()), x.ld, scale, zp, sym, (int8_t*)q.data_ptr(),
              x.cols, x.rows, x.cols, stream_of(*x.t)))
    return nullptr;
  return wrap(q);
  END_HANDLE_TH_ERRORS
}
// (x, mode, compute dtype, scale, zp, sym, clip_lo, clip_hi) -> q
PyObject* quant_i8_static_t(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(8);
  const Mat x = mat(args[0]);
  at::ScalarType ct;
  if (!x || code_of(x.t->scalar_type()) < 0 || !dtype_arg(args[2], &ct) || !here(x.t)) return none();
  const int mode = (int)WHOLE(1), sym = (int)WHOLE(5);
  const float scale = (float)REAL(3), zp = (float)REAL(4), lo = (float)REAL(6), hi = (float)REAL(7);
  NUMBERS_OK;
  at::Tensor q = empty({x.rows, x.cols}, at::kChar, *x.t);
  if (!LAUNCH(fmsmo_quant_act_i8_static_t, x.p, code_of(x.t->scalar_type()), x.ld, mode, code_of(ct), scale, zp, sym, lo,
              hi, (int8_t*)q.data_ptr(), x.cols, x.rows, x.cols, stream_of(*x.t)))
    return nullptr;
  return wrap(q);
  END_HANDLE_TH_ERRORS
}
// e4m3 codes of x and their scale(s): per token (the floor and dtype of the scale as fmsmo_quant_act_fp8_pertoken
// has them where plain_recipe) or per tensor; false with a Python error set where a launch fails
bool fp8_codes(const Mat& x, int variant, bool per_tensor, double floor, bool in_x, at::Tensor* q, at::Tensor* s) {
  *q = empty({x.rows, x.cols}, at::kFloat8_e4m3fn, *x.t);
  *s = empty({per_tensor ? 1 : x.rows}, at::kFloat, *x.t);
  const int dt = code_of(x.t->scalar_type()), sdt = in_x ? dt : FMSMO_F32;
  uint8_t* qp = (uint8_t*)q->data_ptr();
  float* sp = (float*)s->data_ptr();
  if (per_tensor) {
    at::Tensor parts = empty({256}, at::kFloat, *x.t);
    return LAUNCH(fmsmo_quant_act_fp8_tensor, x.p, dt, x.ld, variant, (float)floor, sdt, (float*)parts.data_ptr(), qp,
                  x.cols, sp, x.rows, x.cols, stream_of(*x.t));
  }
  if (floor == 1e-12 && !in_x)
    return LAUNCH(fmsmo_quant_act_fp8_pertoken, x.p, dt, x.ld, variant, 0, qp, x.cols, sp, x.rows, x.cols,
                  stream_of(*x.t));
  return LAUNCH(fmsmo_quant_act_fp8_dynamic, x.p, dt, x.ld, variant, 0, (const float*)nullptr, (float)floor, sdt, qp,
                x.cols, sp, x.rows, x.cols, stream_of(*x.t));
}
// (fmsmo_quant_act_fp8_tensor counts 8-element chunks in 31 bits)
bool fp8_tensor_ok(const Mat& x) { return x.rows > 0 && x.cols > 0 && x.rows < (1ll << 34) / x.cols; }
// (x, variant, per_tensor, scale_floor, scale_in_x_dtype) -> (q, scale)
PyObject* quant_fp8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(5);
  const Mat x = mat(args[0]);
  if (!x || code_of(x.t->scalar_type()) < 0 || !here(x.t)) return none();
  const int variant = (int)WHOLE(1);
  const bool per_tensor = PyObject_IsTrue(args[2]) == 1, in_x = PyObject_IsTrue(args[4]) == 1;
  const double floor = REAL(3);
  NUMBERS_OK;
  if (per_tensor && !fp8_tensor_ok(x)) return none();
  at::Tensor q, s;
  if (!fp8_codes(x, variant, per_tensor, floor, in_x, &q, &s)) return nullptr;
  return wrap2(q, s);
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------ products
bool run_gemm_i8(const char* a, int64_t lda, const Mat& w, const float* as, int64_t an, const at::Tensor& ws,
                 const Opt& b, int epi, const at::Tensor& y, int64_t M, int64_t K) {
  const at::Tensor scratch = workspace(p_fmsmo_gemm_workspace_bytes(M, w.rows, K), *w.t);
  return LAUNCH(fmsmo_gemm_i8_dq_ws, (const int8_t*)a, lda, (const int8_t*)w.p, w.ld, as, an, (const float*)ws.data_ptr(),
                ws.numel(), b.p, b.dt, epi, y.data_ptr(), code_of(y.scalar_type()), w.rows, M, w.rows, K,
                scratch.defined() ? scratch.data_ptr() : nullptr, scratch.defined() ? scratch.numel() : 0,
                stream_of(*w.t));
}
bool run_gemm_fp8(const char* a, int64_t lda, const Mat& w, const float* as, int64_t an, const float* ws, int64_t wn,
                  const Opt& b, const at::Tensor& y, int64_t M, int64_t K) {
  const at::Tensor scratch = workspace(p_fmsmo_gemm_fp8_workspace_bytes(M, w.rows, K), *w.t);
  return LAUNCH(fmsmo_gemm_fp8_dq_ws, (const uint8_t*)a, lda, (const uint8_t*)w.p, w.ld, as, an, ws, wn, b.p, b.dt,
                y.data_ptr(), code_of(y.scalar_type()), w.rows, M, w.rows, K,
                scratch.defined() ? scratch.data_ptr() : nullptr, scratch.defined() ? scratch.numel() : 0,
                stream_of(*w.t));
}
// (a, w, a_scale, w_scale, bias | None, out dtype, epilogue) -> y [M,N]; epilogue is ignored for e4m3
PyObject* gemm_dq(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(7);
  const Mat a = mat(args[0]), w = mat(args[1]);
  at::ScalarType ot;
  if (!a || !w || a.cols != w.cols || a.t->scalar_type() != w.t->scalar_type() || !dtype_arg(args[5], &ot)) return none();
  const bool i8 = a.t->scalar_type() == at::kChar;
  if (!i8 && a.t->scalar_type() != at::kFloat8_e4m3fn) return none();
  const at::Tensor *as = vec32(args[2], a.rows), *ws = vec32(args[3], w.rows);
  const Opt b = opt_vec(args[4], w.rows);
  if (!as || !ws || !b.ok || !here(a.t, w.t, as, ws, b.t)) return none();
  const int epi = (int)WHOLE(6);
  NUMBERS_OK;
  at::Tensor y = empty({a.rows, w.rows}, ot, *a.t);
  const bool ok = i8 ? run_gemm_i8(a.p, a.ld, w, (const float*)as->data_ptr(), as->numel(), *ws, b, epi, y, a.rows, a.cols)
                     : run_gemm_fp8(a.p, a.ld, w, (const float*)as->data_ptr(), as->numel(), (const float*)ws->data_ptr(),
                                    ws->numel(), b, y, a.rows, a.cols);
  return ok ? wrap(y) : nullptr;
  END_HANDLE_TH_ERRORS
}
bool run_decode_i8(const Mat& x, const Opt& sm, int sat, const Mat& w, const at::Tensor& ws, const Opt& b, int epi,
                   const at::Tensor& y, const at::Tensor& s) {
  return LAUNCH(fmsmo_decode_linear_i8, x.p, code_of(x.t->scalar_type()), x.ld, sm.p, sm.dt, sat, (const int8_t*)w.p, w.ld,
                (const float*)ws.data_ptr(), ws.numel(), b.p, b.dt, epi, y.data_ptr(), code_of(y.scalar_type()), w.rows,
                (float*)s.data_ptr(), x.rows, w.rows, x.cols, stream_of(*x.t));
}
// (x, w, w_scale, bias | None, smooth | None, out dtype, epilogue, saturate) -> (y, scale [M])
PyObject* decode_i8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(8);
  const Mat x = mat(args[0]), w = mat(args[1]);
  at::ScalarType ot;
  if (!x || !w || x.cols != w.cols || code_of(x.t->scalar_type()) < 0 || w.t->scalar_type() != at::kChar ||
      !dtype_arg(args[5], &ot))
    return none();
  const at::Tensor* ws = vec32(args[2], w.rows);
  const Opt b = opt_vec(args[3], w.rows), sm = opt_vec(args[4], x.cols, 16);
  if (!ws || !b.ok || !sm.ok || !here(x.t, w.t, ws, b.t, sm.t)) return none();
  const int epi = (int)WHOLE(6), sat = PyObject_IsTrue(args[7]);
  NUMBERS_OK;
  at::Tensor y = empty({x.rows, w.rows}, ot, *x.t), s = empty({x.rows}, at::kFloat, *x.t);
  if (!run_decode_i8(x, sm, sat, w, *ws, b, epi, y, s)) return nullptr;
  return wrap2(y, s);
  END_HANDLE_TH_ERRORS
}
// (x, w, w_scale, bias | None, out dtype) -> (y, scale [M])
PyObject* decode_fp8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(5);
  const Mat x = mat(args[0]), w = mat(args[1]);
  at::ScalarType ot;
  if (!x || !w || x.cols != w.cols || code_of(x.t->scalar_type()) < 0 || w.t->scalar_type() != at::kFloat8_e4m3fn ||
      !dtype_arg(args[4], &ot))
    return none();
  const at::Tensor* ws = vec32(args[2], w.rows);
  const Opt b = opt_vec(args[3], w.rows);
  if (!ws || !b.ok || !here(x.t, w.t, ws, b.t)) return none();
  at::Tensor y = empty({x.rows, w.rows}, ot, *x.t), s = empty({x.rows}, at::kFloat, *x.t);
  if (!LAUNCH(fmsmo_decode_linear_fp8, x.p, code_of(x.t->scalar_type()), x.ld, (const uint8_t*)w.p, w.ld,
              (const float*)ws->data_ptr(), ws->numel(), b.p, b.dt, y.data_ptr(), code_of(ot), w.rows,
              (float*)s.data_ptr(), x.rows, w.rows, x.cols, stream_of(*x.t)))
    return nullptr;
  return wrap2(y, s);
  END_HANDLE_TH_ERRORS
}
// (a [T,K], w [E,N,K], offsets, a_scale, w_scale, bias | None, out dtype, epilogue) -> y [T,N]
PyObject* grouped_i8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(8);
  const Mat a = mat(args[0]);
  const at::Tensor *w = plain(args[1]), *off = plain(args[2]), *as = plain(args[3]), *ws = plain(args[4]);
  at::ScalarType ot;
  if (!a || !w || !off || !as || !ws || a.t->scalar_type() != at::kChar || w->scalar_type() != at::kChar || w->dim() != 3 ||
      !w->is_contiguous() || w->size(2) != a.cols || off->scalar_type() != at::kInt || !off->is_contiguous() ||
      off->numel() != w->size(0) + 1 || !dtype_arg(args[6], &ot))
    return none();
  const int64_t E = w->size(0), N = w->size(1), K = a.cols;
  if (as->scalar_type() != at::kFloat || !as->is_contiguous() || as->numel() != a.rows || ws->scalar_type() != at::kFloat ||
      !ws->is_contiguous() || ws->numel() != E * N)
    return none();
  Opt b;
  b.ok = args[5] == Py_None;
  if (!b.ok) {
    const at::Tensor* t = plain(args[5]);
    if (!t || !t->is_contiguous() || t->numel() != E * N || code_of(t->scalar_type()) < 0) return none();
    b = Opt{true, t->data_ptr(), code_of(t->scalar_type()), t->scalar_type(), t};
  }
  if (!here(a.t, w, off, as, ws, b.t)) return none();
  const int epi = (int)WHOLE(7);
  NUMBERS_OK;
  at::Tensor y = empty({a.rows, N}, ot, *a.t);
  if (!LAUNCH(fmsmo_grouped_gemm_i8_dq, (const int8_t*)a.p, a.ld, (const int8_t*)w->data_ptr(), K, N * K,
              (const int32_t*)off->data_ptr(), (int)E, a.rows, (const float*)as->data_ptr(), (const float*)ws->data_ptr(),
              b.p, b.dt, epi, y.data_ptr(), code_of(ot), N, N, K, stream_of(*a.t)))
    return nullptr;
  return wrap(y);
  END_HANDLE_TH_ERRORS
}
// (a, w, a_scale, w_scale, bias | None, epilogue, out dtype, chunk_size, chunk_trun_bits, max_acc_bits,
//  truncate_then_accumulate, clamp_acc_to_dl16) -> y [M,N]
PyObject* chunk_dq(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(12);
  const Mat a = mat(args[0]), w = mat(args[1]);
  at::ScalarType ot;
  if (!a || !w || a.cols != w.cols || a.t->scalar_type() != w.t->scalar_type() || !dtype_arg(args[6], &ot)) return none();
  const at::ScalarType at_ = a.t->scalar_type();
  const int op = at_ == at::kChar ? FMSMO_OP_I8 : at_ == at::kFloat8_e4m3fn ? FMSMO_OP_E4M3 : at_ == at::kHalf ? FMSMO_OP_F16
                 : at_ == at::kBFloat16 ? FMSMO_OP_BF16 : at_ == at::kFloat ? FMSMO_OP_F32 : -1;
  if (op < 0) return none();
  const int64_t per16 = 16 / (int64_t)a.t->element_size(), M = a.rows, N = w.rows, K = a.cols;
  const at::Tensor *as = vec32(args[2], M), *ws = vec32(args[3], N);
  const Opt b = opt_vec(args[4], N);
  if (K % per16 || a.ld % per16 || w.ld % per16 || !as || !ws || !b.ok || !here(a.t, w.t, as, ws, b.t)) return none();
  const int epi = (int)WHOLE(5), chunk = (int)WHOLE(7), trun = (int)WHOLE(8), bits = (int)WHOLE(9);
  NUMBERS_OK;
  const int tta = PyObject_IsTrue(args[10]) == 1, dl16 = PyObject_IsTrue(args[11]) == 1;
  at::Tensor y = empty({M, N}, ot, *a.t);
  // (in floating point no workspace: the rounded chunks are to be added one after the other, see matmul_chunk)
  const at::Tensor scratch =
      workspace(op == FMSMO_OP_I8 ? p_fmsmo_matmul_chunk_workspace_bytes(op, M, N, K, chunk, tta) : 0, *a.t);
  void* wp = scratch.defined() ? scratch.data_ptr() : nullptr;
  const int64_t wb = scratch.defined() ? scratch.numel() : 0;
  const float *ap = (const float*)as->data_ptr(), *sp = (const float*)ws->data_ptr();
  const int bdt = b.p ? b.dt : FMSMO_F32;
  const bool ok =
      op == FMSMO_OP_I8
          ? LAUNCH(fmsmo_matmul_chunk_i8_dq_ws, (const int8_t*)a.p, a.ld, (const int8_t*)w.p, w.ld, ap, as->numel(), sp,
                   ws->numel(), b.p, bdt, epi, y.data_ptr(), code_of(ot), N, M, N, K, chunk, trun, bits, tta, wp, wb,
                   stream_of(*a.t))
          : LAUNCH(fmsmo_matmul_chunk_fp_dq, a.p, a.ld, w.p, w.ld, op, ap, as->numel(), sp, ws->numel(), b.p, bdt, epi,
                   y.data_ptr(), code_of(ot), N, M, N, K, chunk, trun, dl16, tta, stream_of(*a.t));
  return ok ? wrap(y) : nullptr;
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------ attention products
// int8 codes of x [B,R,C] (contiguous, element strides ldx / stride) along the last dimension of q, with their sums
struct Codes {
  at::Tensor q, sums;
  int64_t ld = 0;
  int parts = 0;
};
bool affine(const at::Tensor& like, const void* x, int64_t ldx, int64_t stride, float scale, float offset, int ct,
            bool transpose, int64_t pad, bool want_sums, int64_t B, int64_t R, int64_t C, Codes* c) {
  const int64_t inner = transpose ? R : C, rows = transpose ? C : R;
  c->ld = (inner + pad - 1) / pad * pad;
  c->q = empty({B, rows, c->ld}, at::kChar, like);
  if (want_sums) {
    c->parts = p_fmsmo_affine_sum_parts(B, R, C, transpose);
    c->sums = empty({c->parts, B, rows}, at::kInt, like);
  }
  return LAUNCH(fmsmo_quant_i8_affine_sums, x, code_of(like.scalar_type()), ldx, stride, scale, offset, ct, (int)transpose,
                (int8_t*)c->q.data_ptr(), c->ld, rows * c->ld, want_sums ? (int32_t*)c->sums.data_ptr() : nullptr, B, R, C,
                stream_of(like));
}
// (m1 [.., M, K], m2 [.., K, N], scale1, zero1, scale2, zero2, compute dtype) -> y [B, M, N]
PyObject* bmm_quantized(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(7);
  const at::Tensor *m1 = plain(args[0]), *m2 = plain(args[1]);
  at::ScalarType cst;
  if (!m1 || !m2 || m1->dim() < 2 || m1->dim() != m2->dim() || m1->scalar_type() != m2->scalar_type() ||
      code_of(m1->scalar_type()) < 0 || !dtype_arg(args[6], &cst) || m1->numel() == 0 || m2->numel() == 0)
    return none();
  const int64_t d = m1->dim(), M = m1->size(d - 2), K = m1->size(d - 1), N = m2->size(d - 1);
  if (!m1->sizes().slice(0, d - 2).equals(m2->sizes().slice(0, d - 2)) || m2->size(d - 2) != K || !m1->is_contiguous())
    return none();
  const int64_t B = m1->numel() / (M * K);
  // m2 as it lies in memory: [.., K, N], or the transposed view of [.., N, K]
  const bool by_rows = m2->stride(d - 2) == 1 && K > 1;
  if (by_rows ? !m2->transpose(d - 2, d - 1).is_contiguous() : !m2->is_contiguous()) return none();
  if (!here(m1, m2)) return none();
  const float s1 = (float)REAL(2), z1 = (float)REAL(3), s2 = (float)REAL(4), z2 = (float)REAL(5);
  const float product = (float)(REAL(2) * REAL(4));
  NUMBERS_OK;
  if (!std::isfinite(product)) return none();
  const int xt = code_of(m1->scalar_type()), ct = code_of(cst);
  const bool qa = xt != FMSMO_F32 && p_fmsmo_bmm_qa_ok(xt, ct, s1, z1, B, M, N, K);
  // scores of a head dimension up to 128 run on the kernel for a reduction of exactly 128
  const int64_t pad = K <= 128 && M > 128 && N > 128 ? 128 : 64;
  at::Tensor y = empty({B, M, N}, m1->scalar_type(), *m1);
  if (qa) {
    Codes c2;
    if (!(by_rows ? affine(*m2, m2->data_ptr(), K, N * K, s2, z2, ct, false, pad, true, B, N, K, &c2)
                  : affine(*m2, m2->data_ptr(), N, K * N, s2, z2, ct, true, pad, true, B, K, N, &c2)))
      return nullptr;
    if (!LAUNCH(fmsmo_bmm_qa_i8, m1->data_ptr(), xt, K, M * K, s1, z1, ct, (const int8_t*)c2.q.data_ptr(), c2.ld, N * c2.ld,
                s2, (int32_t*)c2.sums.data_ptr(), c2.parts, y.data_ptr(), N, B, M, N, K, stream_of(*m1)))
      return nullptr;
    return wrap(y);
  }
  // both operands' codes and the second one's sums in one launch
  const int64_t ld = (K + pad - 1) / pad * pad;
  int parts = by_rows ? 1 : p_fmsmo_affine_sum_parts(B, K, N, 1);
  at::Tensor q1 = empty({B, M, ld}, at::kChar, *m1), q2 = empty({B, N, ld}, at::kChar, *m1),
             sum = empty({parts, B, N}, at::kInt, *m1);
  int32_t* sums = (int32_t*)sum.data_ptr();
  if (!LAUNCH(fmsmo_quant_i8_affine_pair, xt, ct, B, m1->data_ptr(), K, M * K, s1, z1, (int8_t*)q1.data_ptr(), M * ld, M,
              m2->data_ptr(), by_rows ? K : N, N * K, s2, z2, by_rows ? 0 : 1, (int8_t*)q2.data_ptr(), N * ld, sums, N, K,
              ld, stream_of(*m1)))
    return nullptr;
  if (p_fmsmo_affine_parts_first(parts, M, N, ld)) {
    if (!LAUNCH(fmsmo_affine_add_parts, sums, parts, B * N, stream_of(*m1))) return nullptr;
    parts = 1;
  }
  if (!LAUNCH(fmsmo_bmm_i8_zp, (const int8_t*)q1.data_ptr(), ld, (const int8_t*)q2.data_ptr(), ld, N * ld, product, (int)z1,
              sums, parts, y.data_ptr(), xt, N, B, M, N, ld, stream_of(*m1)))
    return nullptr;
  return wrap(y);
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------ whole forwards
// Their operands are the module's.  A launch lets go of the interpreter lock, and another thread may then replace
// what the module's dicts hold: these forwards own what they go on using (the arguments of a call are its caller's).
at::Tensor owned(const at::Tensor* t) { return t ? *t : at::Tensor(); }
PyObject* item(PyObject* dict, PyObject* key) {  // borrowed, or null
  return dict && PyDict_Check(dict) ? PyDict_GetItemWithError(dict, key) : nullptr;
}
#define NAMES(X)                                                                                                \
  X(_buffers) X(_parameters) X(weight) X(bias) X(w_scale) X(smoothq_scale) X(input_scale) X(useDynMaxQfunc)      \
  X(use_int_kernel) X(chunk_size) X(truncate_lsb) X(use_fake_zero_shift) X(acc_dtype) X(_sq_kept) X(_ws_kept)    \
  X(iaddmm) X(cvs) X(weight_scale) X(_quantize) X(qa_dynamic_max_qfunc) X(_smoothq_active) X(_w_scale_f32)         \
  X(_set_input_scale) X(_sp_kept) X(usePTnativeQfunc) X(useSymAct) X(input_zp) X(quant_stepsize) X(quant_zero_point)     \
  X(qa_fmo_mo_qfunc) X(_static_params)
#define DECLARE(n) PyObject* k_##n = nullptr;
NAMES(DECLARE)
#undef DECLARE

// Is this (data pointer, version, dtype) the stamp of t as it is now?
bool same_stamp(PyObject* stamp, const at::Tensor& t) {
  if (t.is_inference() || !PyTuple_Check(stamp) || PyTuple_GET_SIZE(stamp) != 3 || !THPDtype_Check(PyTuple_GET_ITEM(stamp, 2)))
    return false;
  const unsigned long long p = PyLong_AsUnsignedLongLong(PyTuple_GET_ITEM(stamp, 0));
  const long long v = PyLong_AsLongLong(PyTuple_GET_ITEM(stamp, 1));
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return p == (unsigned long long)(uintptr_t)t.data_ptr() && v == (long long)t._version() &&
         ((THPDtype*)PyTuple_GET_ITEM(stamp, 2))->scalar_type == t.scalar_type();
}
// What the Python side found out about buffer t, kept as ((data pointer, version, dtype), finding, alias of the
// buffer): the finding (borrowed), or null where the buffer is another one or was written to since.  (The alias keeps
// the memory, so the address is the buffer's own.)
PyObject* kept_for(PyObject* kept, const at::Tensor& t) {
  if (!kept || !PyTuple_Check(kept) || PyTuple_GET_SIZE(kept) != 3) return nullptr;
  return same_stamp(PyTuple_GET_ITEM(kept, 0), t) ? PyTuple_GET_ITEM(kept, 1) : nullptr;
}
// The parameters of the static quantizer that the Python side keeps for activations of dtype xt beside the buffers they were read from
// (QLinearINT8Deploy._static_params); false where one of those is another tensor or was written to since.
struct StaticParams {
  double step = 0, qzp = 0, lo = 0, hi = 0;
  at::ScalarType T = at::kFloat;
  const at::Tensor* scale = nullptr;  // the buffer input_scale itself, one element
};
bool static_params(PyObject* self, PyObject* buffers, at::ScalarType xt, StaticParams* p) {
  PyObject *kept = item(self, k__sp_kept), *cvs = item(self, k_cvs);
  if (!kept || !PyTuple_Check(kept) || PyTuple_GET_SIZE(kept) != 3 || !cvs || !PyList_CheckExact(cvs) || PyList_GET_SIZE(cvs) < 2)
    return false;
  PyObject *stamps = PyTuple_GET_ITEM(kept, 0), *found = PyTuple_GET_ITEM(kept, 1);
  if (!PyTuple_Check(stamps) || PyTuple_GET_SIZE(stamps) != 7 || !PyDict_Check(found)) return false;
  if (!THPDtype_Check(PyTuple_GET_ITEM(stamps, 0)) || ((THPDtype*)PyTuple_GET_ITEM(stamps, 0))->scalar_type != xt) return false;
  PyObject* of[6] = {item(buffers, k_input_scale), item(buffers, k_input_zp), item(buffers, k_quant_stepsize),
                     item(buffers, k_quant_zero_point), PyList_GET_ITEM(cvs, 0), PyList_GET_ITEM(cvs, 1)};
  for (int i = 0; i < 6; ++i) {
    const at::Tensor* t = of[i] ? plain(of[i]) : nullptr;
    if (!t || !same_stamp(PyTuple_GET_ITEM(stamps, i + 1), *t)) return false;
    if (i == 0 && t->numel() != 1) return false;
  }
  const char* names[4] = {"step", "qzp", "lo", "hi"};
  double* to[4] = {&p->step, &p->qzp, &p->lo, &p->hi};
  for (int i = 0; i < 4; ++i) {
    PyObject* v = PyDict_GetItemString(found, names[i]);
    if (!v || !PyFloat_Check(v)) return false;
    *to[i] = PyFloat_AS_DOUBLE(v);
  }
  PyObject* T = PyDict_GetItemString(found, "T");
  if (!T || !dtype_arg(T, &p->T)) return false;
  p->scale = plain(of[0]);
  return code_of(p->scale->scalar_type()) >= 0 && !p->scale->requires_grad();
}

// Is a method of the class, or of this instance, another function than the one that came with it?
bool replaced(PyObject* self, PyTypeObject* cls, PyObject* name, PyObject* own) {
  return item(self, name) || _PyType_Lookup(cls, name) != own;
}
// QLinearINT8Deploy.forward with dynamic per-token scales, or static ones by the fms_mo formula, and a plain integer product: (instance
// dict, x, the class, (iaddmm_int, _smoothq_active, _w_scale_f32, _set_input_scale, _quantize, qa_dynamic_max_qfunc, qa_fmo_mo_qfunc,
// _static_params) as it came) -> y.
// The scales' host-side facts (does SmoothQuant apply, the fp32 copy of w_scale) are those the Python side
// keeps beside the buffers; where they are stale it is asked (None).
PyObject* deploy_i8(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(4);
  PyObject *self = args[0], *own_f = args[3];
  if (!PyType_Check(args[2]) || !PyTuple_CheckExact(own_f) || PyTuple_GET_SIZE(own_f) != 8) return none();
  // the methods that the forward in Python goes through: these always, its quantizer's and iaddmm on one branch below
  PyTypeObject* cls = (PyTypeObject*)args[2];
  auto other = [&](PyObject* name, int i) { return replaced(self, cls, name, PyTuple_GET_ITEM(own_f, i)); };
  if (other(k__smoothq_active, 1) || other(k__w_scale_f32, 2) || other(k__set_input_scale, 3)) return none();
  const Mat x = rows_of(args[1]);
  if (!x || x.rows == 0 || code_of(x.t->scalar_type()) < 0) return none();
  PyObject *buffers = item(self, k__buffers), *params = item(self, k__parameters);
  PyObject *dyn = item(self, k_useDynMaxQfunc), *kern = item(self, k_use_int_kernel), *acc = item(self, k_acc_dtype);
  PyObject *chunk = item(self, k_chunk_size), *lsb = item(self, k_truncate_lsb), *fzs = item(self, k_use_fake_zero_shift);
  PyObject *ow = item(params, k_weight), *osq = item(buffers, k_smoothq_scale), *ows = item(buffers, k_w_scale);
  const bool stat = dyn == Py_False;
  if (!dyn || (!stat && (!PyLong_CheckExact(dyn) || PyLong_AsLong(dyn) != -1)) || !kern || !acc || !chunk || !PyLong_Check(chunk) || !lsb || !PyLong_Check(lsb) ||
      !ow || !osq || !ows || !item(buffers, k_input_scale) || PyObject_IsTrue(kern) != 1 ||
      PyLong_AsLong(lsb) > 0 || x.cols > PyLong_AsLong(chunk) || (fzs && PyObject_IsTrue(fzs) != 0)) {
    PyErr_Clear();
    return none();
  }
  at::ScalarType acct;
  Mat w = mat(ow);
  if (!dtype_arg(acc, &acct) || acct != at::kHalf || !w || w.t->scalar_type() != at::kChar || w.cols != x.cols)
    return none();
  const at::Tensor *sq = plain(osq), *wsrc = plain(ows);
  if (!sq || !wsrc) return none();
  PyObject *on = kept_for(item(self, k__sq_kept), *sq), *own = kept_for(item(self, k__ws_kept), *wsrc);
  const at::Tensor* ws = own ? vec32(own, w.rows) : nullptr;
  const bool smooth = on == Py_True;
  if (!ws || (!smooth && on != Py_False)) return none();
  Opt sm;
  if (smooth) {
    const at::ScalarType st = sq->scalar_type();
    if (sq->numel() != x.cols || !sq->is_contiguous() || code_of(st) < 0 || (uintptr_t)sq->data_ptr() % 16) return none();
    sm = Opt{true, sq->data_ptr(), code_of(st), st, sq};
  }
  PyObject* ob = item(buffers, k_bias);
  if (!ob) ob = item(params, k_bias);
  if (!ob) return none();
  const Opt b = opt_vec(ob, w.rows);
  const at::ScalarType xt = x.t->scalar_type();
  if (!b.ok || !here(x.t, w.t, wsrc, ws, sq, b.t)) return none();
  // the epilogues round to the fp16 accumulator dtype and then to bf16 for a bf16 model
  const at::ScalarType ot = xt == at::kBFloat16 ? at::kBFloat16 : at::kHalf;
  if (xt == at::kFloat) return none();  // (the fp16 result is cast behind the product)
  const at::Tensor own_w = *w.t, own_ws = *ws, own_sm = owned(sm.t), own_b = owned(b.t);
  const THPObjectPtr own_buffers(Py_NewRef(buffers));
  w.t = &own_w;
  ws = &own_ws;
  auto plain_product = [&]() {  // the branch that ends in the module's iaddmm: only the class's own one is known here
    PyObject* f = item(self, k_iaddmm);
    return f && PyMethod_Check(f) && PyMethod_GET_FUNCTION(f) == PyTuple_GET_ITEM(own_f, 0) && !other(k__quantize, 4);
  };
  if (stat) {
    PyObject* native = item(self, k_usePTnativeQfunc);
    PyObject* sym = item(self, k_useSymAct);
    StaticParams p;
    if (smooth || native != Py_False || !sym || !plain_product() || other(k_qa_fmo_mo_qfunc, 6) || other(k__static_params, 7) ||
        !static_params(self, buffers, xt, &p) || !here(x.t, p.scale))
      return none();
    // The launches read the module's own buffer, as the general path does: a copy of it that the module kept could be
    // freed under a graph that was captured with its address, and a number would not follow the buffer when one is replayed.
    const at::Tensor own_scale = *p.scale;
    const int sdt = code_of(own_scale.scalar_type());
    const int sy = PyObject_IsTrue(sym) == 1;
    at::Tensor y = out_like(*x.t, w.rows, ot);
    if (p.T == at::kFloat && w.rows * w.ld < (1ll << 31) &&
        p_fmsmo_small_linear_static_ok(x.rows, w.rows, x.cols, (float)p.step, (float)p.qzp, (float)p.lo, (float)p.hi)) {
      if (!LAUNCH(fmsmo_small_linear_i8_static_scale, x.p, code_of(xt), x.ld, (float)p.step, (float)p.qzp, sy, (float)p.lo,
                  (float)p.hi, (const void*)own_scale.data_ptr(), sdt, (const int8_t*)w.p, w.ld, (const float*)ws->data_ptr(), ws->numel(), b.p, b.dt,
                  FMSMO_EPI_REF_F16, y.data_ptr(), code_of(ot), w.rows, x.rows, w.rows, x.cols, stream_of(*x.t)))
        return nullptr;
      return wrap(y);
    }
    at::Tensor q = empty({x.rows, x.cols}, at::kChar, *x.t), s = own_scale;
    if (sdt == FMSMO_F32) {
      if (!LAUNCH(fmsmo_quant_act_i8_static_t, x.p, code_of(xt), x.ld, FMSMO_SQ_FMO, code_of(p.T), (float)p.step, (float)p.qzp,
                  sy, (float)p.lo, (float)p.hi, (int8_t*)q.data_ptr(), x.cols, x.rows, x.cols, stream_of(*x.t)))
        return nullptr;
    } else {
      s = empty({1}, at::kFloat, *x.t);
      if (!LAUNCH(fmsmo_quant_act_i8_static_scale, x.p, code_of(xt), x.ld, FMSMO_SQ_FMO, code_of(p.T), (float)p.step,
                  (float)p.qzp, sy, (float)p.lo, (float)p.hi, (int8_t*)q.data_ptr(), x.cols,
                  (const void*)own_scale.data_ptr(), sdt, (float*)s.data_ptr(), x.rows, x.cols, stream_of(*x.t)))
        return nullptr;
    }
    if (!run_gemm_i8((const char*)q.data_ptr(), x.cols, w, (const float*)s.data_ptr(), 1, *ws, b, FMSMO_EPI_REF_F16, y,
                     x.rows, x.cols))
      return nullptr;
    return wrap(y);
  }
  at::Tensor y = out_like(*x.t, w.rows, ot), s;
  const bool f32s = smooth && sm.st == at::kFloat;
  const bool one = (!smooth || sm.st == xt || f32s) &&
                   (f32s ? p_fmsmo_decode_linear_f32s_ok(x.rows, x.cols) : p_fmsmo_decode_linear_ok(x.rows, x.cols));
  const int in_one = !one && (!smooth || sm.st == xt || f32s) && w.rows * w.ld < (1ll << 31)
                         ? p_fmsmo_small_linear_better(0, x.rows, w.rows, x.cols, f32s) : 0;
  const bool small = in_one == 1 || (in_one == 2 && !capturing(*x.t));
  if (one || smooth || small) s = empty({x.rows, 1}, at::kFloat, *x.t);
  if (one) {
    // decode step of a few tokens: quantizer and weight-streaming matmul in one launch
    if (!run_decode_i8(x, sm, 0, w, *ws, b, FMSMO_EPI_REF_F16, y, s)) return nullptr;
  } else {
    if (!smooth) {
      PyObject* cvs = item(self, k_cvs);
      if (!plain_product() || !cvs || !PyList_CheckExact(cvs) || PyList_GET_SIZE(cvs) < 2 || other(k_qa_dynamic_max_qfunc, 5))
        return none();
    }
    at::Tensor q, c;
    if (small) {  // quantizer and product in one launch, the clip values from it too
      if (!smooth) c = empty({2, x.rows, 1}, at::kFloat, *x.t);
      if (!LAUNCH(fmsmo_small_linear_i8, x.p, code_of(xt), x.ld, sm.p, sm.dt, (const int8_t*)w.p, w.ld,
                  (const float*)ws->data_ptr(), ws->numel(), b.p, b.dt, FMSMO_EPI_REF_F16, y.data_ptr(),
                  code_of(y.scalar_type()), w.rows, (float*)s.data_ptr(), smooth ? nullptr : (float*)c.data_ptr(), x.rows,
                  w.rows, x.cols, stream_of(*x.t)))
        return nullptr;
    } else if (smooth) {
      q = empty({x.rows, x.cols}, at::kChar, *x.t);
      if (!LAUNCH(fmsmo_quant_act_i8_pertoken, x.p, code_of(xt), x.ld, sm.p, sm.dt, code_of(promoted(xt, sm.st)), 0,
                  (int8_t*)q.data_ptr(), x.cols, (float*)s.data_ptr(), x.rows, x.cols, stream_of(*x.t)))
        return nullptr;
    } else if (!codes_and_clips(x, &q, &s, &c)) {
      return nullptr;
    }
    if (!small && !run_gemm_i8((const char*)q.data_ptr(), x.cols, w, (const float*)s.data_ptr(), x.rows, *ws, b,
                               FMSMO_EPI_REF_F16, y, x.rows, x.cols))
      return nullptr;
    PyObject* cvs = smooth ? nullptr : item(self, k_cvs);
    if (cvs && PyList_CheckExact(cvs) && PyList_GET_SIZE(cvs) >= 2) {
      PyList_SetItem(cvs, 0, wrap(c.select(0, 0)));
      PyList_SetItem(cvs, 1, wrap(c.select(0, 1)));
    }
  }
  PyObject* os = wrap(s);
  const int rc = PyDict_SetItem(buffers, k_input_scale, os);
  Py_DECREF(os);
  return rc ? nullptr : wrap(y);
  END_HANDLE_TH_ERRORS
}

// FP8Linear.forward with dynamic scales: (parameter dict, has_bias, x, per tensor, scale floor, scale in x's dtype) -> y
PyObject* fp8_linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  WANT(6);
  const Mat x = rows_of(args[2]);
  PyObject *ow = item(args[0], k_weight), *ows = item(args[0], k_weight_scale);
  if (!x || x.rows == 0 || code_of(x.t->scalar_type()) < 0 || !ow || !ows) return none();
  Mat w = mat(ow);
  const at::Tensor* ws = plain(ows);
  if (!w || w.t->scalar_type() != at::kFloat8_e4m3fn || w.cols != x.cols || !ws || ws->scalar_type() != at::kFloat ||
      !ws->is_contiguous() || (ws->numel() != 1 && ws->numel() != w.rows))
    return none();
  Opt b;
  b.ok = true;
  if (PyObject_IsTrue(args[1]) == 1) {
    PyObject* ob = item(args[0], k_bias);
    if (!ob || ob == Py_None) return none();
    b = opt_vec(ob, w.rows);
  }
  const bool per_tensor = PyObject_IsTrue(args[3]) == 1, in_x = PyObject_IsTrue(args[5]) == 1;
  const double floor = REAL(4);
  NUMBERS_OK;
  if (!b.ok || !here(x.t, w.t, ws, b.t) || (per_tensor && !fp8_tensor_ok(x))) return none();
  const at::ScalarType xt = x.t->scalar_type();
  const at::Tensor own_w = *w.t, own_ws = *ws, own_b = owned(b.t);
  w.t = &own_w;
  ws = &own_ws;
  const float* wp = (const float*)ws->data_ptr();
  at::Tensor y = out_like(*x.t, w.rows, xt);
  if (!per_tensor && floor == 1e-12 && !in_x && xt != at::kFloat &&
      (p_fmsmo_decode_linear_ok(x.rows, x.cols) ||
       (w.rows * w.ld < (1ll << 31) && p_fmsmo_small_linear_better(1, x.rows, w.rows, x.cols, 0)))) {
    if (!LAUNCH(fmsmo_small_linear_fp8, x.p, code_of(xt), x.ld, (const uint8_t*)w.p, w.ld, wp, ws->numel(), b.p, b.dt,
                y.data_ptr(), code_of(xt), w.rows, (float*)nullptr, x.rows, w.rows, x.cols, stream_of(*x.t)))
      return nullptr;
    return wrap(y);
  }
  at::Tensor q, s;
  if (!fp8_codes(x, FMSMO_FP8_LINEAR, per_tensor, floor, in_x, &q, &s)) return nullptr;
  if (!run_gemm_fp8((const char*)q.data_ptr(), x.cols, w, (const float*)s.data_ptr(), s.numel(), wp, ws->numel(), b, y,
                    x.rows, x.cols))
    return nullptr;
  return wrap(y);
  END_HANDLE_TH_ERRORS
}

// ------------------------------------------------------------------ module
// bind({entry point: address}, raise_status)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  WANT(2);
#define RESOLVE(f)                                                                              \
  {                                                                                             \
    PyObject* a_ = PyDict_GetItemString(args[0], #f);                                           \
    if (!a_) return PyErr_Format(PyExc_KeyError, "entry point %s", #f);                         \
    p_##f = (decltype(p_##f))PyLong_AsVoidPtr(a_);                                              \
    if (PyErr_Occurred()) return nullptr;                                                       \
  }
  ENTRIES(RESOLVE)
#undef RESOLVE
  Py_INCREF(args[1]);
  Py_XSETREF(g_raise_status, args[1]);
  Py_RETURN_NONE;
}
// the names bind() wants
PyObject* entries(PyObject*, PyObject*) {
  PyObject* l = PyList_New(0);
#define APPEND(f)                          \
  {                                        \
    PyObject* s = PyUnicode_FromString(#f); \
    PyList_Append(l, s);                   \
    Py_DECREF(s);                          \
  }
  ENTRIES(APPEND)
#undef APPEND
  return l;
}
#define FAST(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(quant_i8), FAST(quant_i8_clips), FAST(quant_i8_static), FAST(quant_i8_static_t), FAST(quant_fp8), FAST(gemm_dq),
                         FAST(decode_i8), FAST(decode_fp8), FAST(grouped_i8), FAST(chunk_dq), FAST(bmm_quantized),
                         FAST(deploy_i8), FAST(fp8_linear), FAST(bind), {"entries", entries, METH_NOARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fmsmo_host", nullptr, -1, methods};

}  // namespace

#define TEXT_(x) #x
#define TEXT(x) TEXT_(x)
PyMODINIT_FUNC PyInit__fmsmo_host() {
#define INTERN(n) k_##n = PyUnicode_InternFromString(#n);
  NAMES(INTERN)
#undef INTERN
  PyObject* m = PyModule_Create(&module);
  // what this file was compiled against: neither torch's nor Python's ABI is in the file's name
  if (m && PyModule_AddStringConstant(m, "built_for", "torch " FMSMO_TORCH_VERSION ", Python " TEXT(PY_MAJOR_VERSION) "." TEXT(
                                                          PY_MINOR_VERSION)))
    return nullptr;
  return m;
}
