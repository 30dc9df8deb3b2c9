// Native host side of the operator wrappers: argument checks, output and scratch allocation through
// torch's caching allocator, the current stream, and the C-ABI launches of a whole linear in one call
// from Python.  No arithmetic happens here.
//
// Why it exists: an eager call of a decode-sized linear was bound by what the host did per call, not by
// its kernels.  (One token through a 4096 x 4096 int8 linear: 18 us per forward of Python-level checks
// and ctypes marshalling around a 5.6 us kernel.)
//
// Every function takes the common case only -- plain, well-formed tensors on the current GPU, laid out
// as the kernels read them -- and returns None for anything else, which then goes through the general
// Python wrappers and gets their conversions and error messages.
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/fmsmo_hip.h"

namespace {

using at::Tensor;

constexpr int BAD_DTYPE = -1;

int dt_code(at::ScalarType t) {
  switch (t) {
    case at::kHalf: return FMSMO_F16;
    case at::kBFloat16: return FMSMO_BF16;
    case at::kFloat: return FMSMO_F32;
    default: return BAD_DTYPE;
  }
}

at::ScalarType dt_torch(int code) {
  return code == FMSMO_F16 ? at::kHalf : code == FMSMO_BF16 ? at::kBFloat16 : at::kFloat;
}

// The tensor of a plain torch.Tensor / Parameter object on the GPU, else nullptr.
const Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const Tensor& t = THPVariable_Unpack(o);
  return t.is_cuda() ? &t : nullptr;
}

struct Mat {
  void* p = nullptr;
  int64_t rows = 0, cols = 0, ld = 0;
};

// 2-D, unit inner stride, rows that do not overlap
bool mat(const Tensor* t, Mat& m) {
  if (!t || t->dim() != 2) return false;
  m.rows = t->size(0);
  m.cols = t->size(1);
  const int64_t s0 = t->stride(0);
  if (t->stride(1) != 1 || (m.rows > 1 && s0 < m.cols)) return false;
  m.ld = m.rows > 1 ? s0 : std::max(m.cols, s0);
  m.p = t->data_ptr();
  return true;
}

// contiguous fp32 vector of 1 or n values (any shape of them)
bool scale_vec(const Tensor* t, int64_t n) {
  return t && t->scalar_type() == at::kFloat && t->is_contiguous() && (t->numel() == n || t->numel() == 1);
}

// optional [n] vector of a 16- or 32-bit float dtype; `given` tells None from a vector
bool opt_vec(PyObject* o, int64_t n, const Tensor*& t, bool& given) {
  given = o != Py_None;
  if (!given) return true;
  t = plain(o);
  return t && t->dim() == 1 && t->numel() == n && t->is_contiguous() && dt_code(t->scalar_type()) != BAD_DTYPE;
}

bool current_device(const Tensor& t) { return c10::hip::current_device() == t.get_device(); }

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.get_device()).stream(); }

Tensor new_like(const Tensor& ref, at::IntArrayRef size, at::ScalarType dtype) {
  return at::empty(size, ref.options().dtype(dtype).requires_grad(false));
}

PyObject* none() { Py_RETURN_NONE; }

// the Python exception of a non-zero status
PyObject* fail(const char* name, int rc) {
  PyObject* lib = PyImport_ImportModule("fms_mo_amd._lib");
  if (lib) {
    PyObject* r = PyObject_CallMethod(lib, "raise_status", "si", name, rc);
    Py_XDECREF(r);
    Py_DECREF(lib);
  }
  if (!PyErr_Occurred()) PyErr_Format(PyExc_RuntimeError, "%s failed with status %d", name, rc);
  return nullptr;
}

PyObject* pair(Tensor a, Tensor b) {
  PyObject* r = PyTuple_New(2);
  if (!r) return nullptr;
  PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(a)));
  PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(b)));
  return r;
}

bool arg_count(Py_ssize_t n, Py_ssize_t want, const char* name) {
  if (n == want) return true;
  PyErr_Format(PyExc_TypeError, "%s takes %zd arguments (%zd given)", name, want, n);
  return false;
}

// C++ exceptions of the allocator become Python ones
template <class F>
PyObject* guarded(F&& f) {
  try {
    return f();
  } catch (const std::exception& e) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

struct Bias {
  const void* p = nullptr;
  int dt = 0;
};

// ---------------------------------------------------------------- the GEMM of a linear, i8 or e4m3
// y [M, N] = epilogue(a [M, K] . w [N, K]^T); split-K scratch from the caching allocator.
int gemm_dq(const Tensor& ref, bool fp8, const void* a, int64_t lda, const Mat& w, const float* a_scale, int64_t a_n,
            const float* w_scale, int64_t w_n, Bias bias, int epilogue, void* y, int out_dt, int64_t M, void* st) {
  const int64_t N = w.rows, K = w.cols;
  const int64_t need = fmsmo_gemm_workspace_bytes(M, N, K);
  Tensor ws;
  if (need > 0) ws = new_like(ref, {need}, at::kByte);
  void* wp = need > 0 ? ws.data_ptr() : nullptr;
  if (fp8)
    return fmsmo_gemm_fp8_dq_ws((const uint8_t*)a, lda, (const uint8_t*)w.p, w.ld, a_scale, a_n, w_scale, w_n, bias.p,
                                bias.dt, y, out_dt, N, M, N, K, wp, need, st);
  return fmsmo_gemm_i8_dq_ws((const int8_t*)a, lda, (const int8_t*)w.p, w.ld, a_scale, a_n, w_scale, w_n, bias.p, bias.dt,
                             epilogue, y, out_dt, N, M, N, K, wp, need, st);
}

// gemm_dq(a, w, a_scale, w_scale, bias, epilogue, out_dt) -> y
PyObject* py_gemm_dq(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (!arg_count(n, 7, "gemm_dq")) return nullptr;
  return guarded([&]() -> PyObject* {
    const Tensor *a = plain(v[0]), *w = plain(v[1]), *as = plain(v[2]), *ws = plain(v[3]), *b = nullptr;
    Mat ma, mw;
    bool has_b;
    if (!mat(a, ma) || !mat(w, mw) || ma.cols != mw.cols || a->scalar_type() != w->scalar_type() ||
        !scale_vec(as, ma.rows) || !scale_vec(ws, mw.rows) || as->dim() != 1 || ws->dim() != 1 ||
        as->requires_grad() || ws->requires_grad() || !opt_vec(v[4], mw.rows, b, has_b) || !current_device(*a))
      return none();
    const bool fp8 = a->scalar_type() == at::kFloat8_e4m3fn;
    if (!fp8 && a->scalar_type() != at::kChar) return none();
    const int epi = (int)PyLong_AsLong(v[5]), od = (int)PyLong_AsLong(v[6]);
    Tensor y = new_like(*a, {ma.rows, mw.rows}, dt_torch(od));
    Bias bias;
    if (has_b) bias = {b->data_ptr(), dt_code(b->scalar_type())};
    const int rc = gemm_dq(*a, fp8, ma.p, ma.ld, mw, (const float*)as->data_ptr(), as->numel(), (const float*)ws->data_ptr(),
                           ws->numel(), bias, epi, y.data_ptr(), od, ma.rows, stream_of(*a));
    if (rc) return fail(fp8 ? "fmsmo_gemm_fp8_dq" : "fmsmo_gemm_i8_dq", rc);
    return THPVariable_Wrap(std::move(y));
  });
}

// ---------------------------------------------------------------- quantizers
bool smooth_vec(PyObject* o, int64_t K, const void*& p, int& dt) {
  const Tensor* t = nullptr;
  bool given;
  if (!opt_vec(o, K, t, given)) return false;
  p = nullptr;
  dt = 0;
  if (given) {
    p = t->data_ptr();
    dt = dt_code(t->scalar_type());
    if ((uintptr_t)p & 15) return false;
  }
  return true;
}

// quant_i8_pertoken(x, smooth, compute_dt, saturate) -> (q, scale)
PyObject* py_quant_i8_pertoken(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (!arg_count(n, 4, "quant_i8_pertoken")) return nullptr;
  return guarded([&]() -> PyObject* {
    const Tensor* x = plain(v[0]);
    Mat m;
    const void* sp;
    int sdt;
    if (!mat(x, m) || dt_code(x->scalar_type()) == BAD_DTYPE || !smooth_vec(v[1], m.cols, sp, sdt) || !current_device(*x))
      return none();
    Tensor q = new_like(*x, {m.rows, m.cols}, at::kChar), s = new_like(*x, {m.rows}, at::kFloat);
    const int rc = fmsmo_quant_act_i8_pertoken(m.p, dt_code(x->scalar_type()), m.ld, sp, sdt, (int)PyLong_AsLong(v[2]),
                                               (int)PyLong_AsLong(v[3]), (int8_t*)q.data_ptr(), m.cols,
                                               (float*)s.data_ptr(), m.rows, m.cols, stream_of(*x));
    if (rc) return fail("fmsmo_quant_act_i8_pertoken", rc);
    return pair(std::move(q), std::move(s));
  });
}

// ---------------------------------------------------------------- whole linears
// linear_i8(x, w, w_scale, bias, smooth, compute_dt, out_dt) -> (y, token scales): per-token quantizer
// and int8 GEMM with the reference epilogue; the fused decode kernel where it serves the shape.
PyObject* py_linear_i8(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (!arg_count(n, 7, "linear_i8")) return nullptr;
  return guarded([&]() -> PyObject* {
    const Tensor *x = plain(v[0]), *w = plain(v[1]), *ws = plain(v[2]), *b = nullptr;
    Mat mx, mw;
    bool has_b;
    const void* sp;
    int sdt;
    if (!mat(x, mx) || !mat(w, mw) || mx.cols != mw.cols || w->scalar_type() != at::kChar || !scale_vec(ws, mw.rows) ||
        !opt_vec(v[3], mw.rows, b, has_b) || !smooth_vec(v[4], mx.cols, sp, sdt) || !current_device(*x))
      return none();
    const int xdt = dt_code(x->scalar_type());
    if (xdt == BAD_DTYPE) return none();
    const int cdt = (int)PyLong_AsLong(v[5]), od = (int)PyLong_AsLong(v[6]);
    const int64_t M = mx.rows, N = mw.rows, K = mw.cols;
    void* st = stream_of(*x);
    Bias bias;
    if (has_b) bias = {b->data_ptr(), dt_code(b->scalar_type())};
    Tensor y = new_like(*x, {M, N}, dt_torch(od)), s = new_like(*x, {M}, at::kFloat);
    const bool sf32 = sp && sdt == FMSMO_F32;
    if (M > 0 && xdt != FMSMO_F32 && (!sp || sf32 || sdt == xdt) &&
        (sf32 ? fmsmo_decode_linear_f32s_ok(M, K) : fmsmo_decode_linear_ok(M, K))) {
      const int rc = fmsmo_decode_linear_i8(mx.p, xdt, mx.ld, sp, sdt, 0, (const int8_t*)mw.p, mw.ld,
                                            (const float*)ws->data_ptr(), ws->numel(), bias.p, bias.dt, FMSMO_EPI_REF_F16,
                                            y.data_ptr(), od, N, (float*)s.data_ptr(), M, N, K, st);
      if (rc) return fail("fmsmo_decode_linear_i8", rc);
      return pair(std::move(y), std::move(s));
    }
    Tensor q = new_like(*x, {M, K}, at::kChar);
    int rc = fmsmo_quant_act_i8_pertoken(mx.p, xdt, mx.ld, sp, sdt, cdt, 0, (int8_t*)q.data_ptr(), K, (float*)s.data_ptr(),
                                         M, K, st);
    if (rc) return fail("fmsmo_quant_act_i8_pertoken", rc);
    rc = gemm_dq(*x, false, q.data_ptr(), K, mw, (const float*)s.data_ptr(), M, (const float*)ws->data_ptr(), ws->numel(),
                 bias, FMSMO_EPI_REF_F16, y.data_ptr(), od, M, st);
    if (rc) return fail("fmsmo_gemm_i8_dq", rc);
    return pair(std::move(y), std::move(s));
  });
}

// linear_i8_static(x, w, a_scale, w_scale, bias, kind, compute_dt, scale, zp, sym, lo, hi, out_dt) -> y:
// static quantizer (kind -1: the fp32 per-tensor form, else one of FMSMO_SQ_*), then the GEMM.
PyObject* py_linear_i8_static(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (!arg_count(n, 13, "linear_i8_static")) return nullptr;
  return guarded([&]() -> PyObject* {
    const Tensor *x = plain(v[0]), *w = plain(v[1]), *as = plain(v[2]), *ws = plain(v[3]), *b = nullptr;
    Mat mx, mw;
    bool has_b;
    if (!mat(x, mx) || !mat(w, mw) || mx.cols != mw.cols || w->scalar_type() != at::kChar || !scale_vec(as, 1) ||
        !scale_vec(ws, mw.rows) || !opt_vec(v[4], mw.rows, b, has_b) || !current_device(*x))
      return none();
    const int xdt = dt_code(x->scalar_type());
    if (xdt == BAD_DTYPE) return none();
    const int kind = (int)PyLong_AsLong(v[5]), cdt = (int)PyLong_AsLong(v[6]), sym = (int)PyLong_AsLong(v[9]);
    const double scale = PyFloat_AsDouble(v[7]), zp = PyFloat_AsDouble(v[8]), lo = PyFloat_AsDouble(v[10]),
                 hi = PyFloat_AsDouble(v[11]);
    const int od = (int)PyLong_AsLong(v[12]);
    if (PyErr_Occurred()) return nullptr;
    const int64_t M = mx.rows, N = mw.rows, K = mw.cols;
    void* st = stream_of(*x);
    Bias bias;
    if (has_b) bias = {b->data_ptr(), dt_code(b->scalar_type())};
    Tensor y = new_like(*x, {M, N}, dt_torch(od)), q = new_like(*x, {M, K}, at::kChar);
    int rc = kind < 0 ? fmsmo_quant_act_i8_static(mx.p, xdt, mx.ld, (float)scale, (int)zp, sym, (int8_t*)q.data_ptr(), K, M,
                                                  K, st)
                      : fmsmo_quant_act_i8_static_t(mx.p, xdt, mx.ld, kind, cdt, (float)scale, (float)zp, sym, (float)lo,
                                                    (float)hi, (int8_t*)q.data_ptr(), K, M, K, st);
    if (rc) return fail("fmsmo_quant_act_i8_static", rc);
    rc = gemm_dq(*x, false, q.data_ptr(), K, mw, (const float*)as->data_ptr(), 1, (const float*)ws->data_ptr(), ws->numel(),
                 bias, FMSMO_EPI_REF_F16, y.data_ptr(), od, M, st);
    if (rc) return fail("fmsmo_gemm_i8_dq", rc);
    return THPVariable_Wrap(std::move(y));
  });
}

// linear_fp8(x, w, w_scale, bias, per_tensor, floor, in_x_dtype, out_dt) -> y: dynamic e4m3 quantizer
// (per token or per tensor) and the GEMM; the fused decode kernel for the plain per-token rule.
PyObject* py_linear_fp8(PyObject*, PyObject* const* v, Py_ssize_t n) {
  if (!arg_count(n, 8, "linear_fp8")) return nullptr;
  return guarded([&]() -> PyObject* {
    const Tensor *x = plain(v[0]), *w = plain(v[1]), *ws = plain(v[2]), *b = nullptr;
    Mat mx, mw;
    bool has_b;
    if (!mat(x, mx) || !mat(w, mw) || mx.cols != mw.cols || w->scalar_type() != at::kFloat8_e4m3fn ||
        !scale_vec(ws, mw.rows) || !opt_vec(v[3], mw.rows, b, has_b) || !current_device(*x))
      return none();
    const int xdt = dt_code(x->scalar_type());
    if (xdt == BAD_DTYPE) return none();
    const bool per_tensor = PyObject_IsTrue(v[4]), in_x = PyObject_IsTrue(v[6]);
    const double floor_v = PyFloat_AsDouble(v[5]);
    const int od = (int)PyLong_AsLong(v[7]);
    if (PyErr_Occurred()) return nullptr;
    const bool plain_rule = !per_tensor && !in_x && floor_v == 1e-12;
    const int64_t M = mx.rows, N = mw.rows, K = mw.cols;
    void* st = stream_of(*x);
    Bias bias;
    if (has_b) bias = {b->data_ptr(), dt_code(b->scalar_type())};
    Tensor y = new_like(*x, {M, N}, dt_torch(od)), s = new_like(*x, {per_tensor ? 1 : M}, at::kFloat);
    if (plain_rule && xdt != FMSMO_F32 && M > 0 && fmsmo_decode_linear_ok(M, K)) {
      const int rc = fmsmo_decode_linear_fp8(mx.p, xdt, mx.ld, (const uint8_t*)mw.p, mw.ld, (const float*)ws->data_ptr(),
                                             ws->numel(), bias.p, bias.dt, y.data_ptr(), od, N, (float*)s.data_ptr(), M, N,
                                             K, st);
      if (rc) return fail("fmsmo_decode_linear_fp8", rc);
      return THPVariable_Wrap(std::move(y));
    }
    Tensor q = new_like(*x, {M, K}, at::kFloat8_e4m3fn);
    int rc;
    if (plain_rule) {
      rc = fmsmo_quant_act_fp8_pertoken(mx.p, xdt, mx.ld, FMSMO_FP8_LINEAR, 0, (uint8_t*)q.data_ptr(), K,
                                        (float*)s.data_ptr(), M, K, st);
    } else {
      const int64_t need = per_tensor ? fmsmo_quant_act_fp8_scratch_bytes(M, K) : 0;
      Tensor scratch;
      if (need > 0) scratch = new_like(*x, {need}, at::kByte);
      rc = fmsmo_quant_act_fp8_dynamic_ws(mx.p, xdt, mx.ld, FMSMO_FP8_LINEAR, per_tensor, (float)floor_v,
                                          in_x ? xdt : FMSMO_F32, need > 0 ? scratch.data_ptr() : nullptr, need,
                                          (uint8_t*)q.data_ptr(), K, (float*)s.data_ptr(), M, K, st);
    }
    if (rc) return fail("fmsmo_quant_act_fp8", rc);
    rc = gemm_dq(*x, true, q.data_ptr(), K, mw, (const float*)s.data_ptr(), per_tensor ? 1 : M,
                 (const float*)ws->data_ptr(), ws->numel(), bias, FMSMO_EPI_F32, y.data_ptr(), od, M, st);
    if (rc) return fail("fmsmo_gemm_fp8_dq", rc);
    return THPVariable_Wrap(std::move(y));
  });
}

// state_key(t, ...) -> bytes naming where each tensor lives, its version, dtype and size: equal keys
// mean that what was derived from these tensors still holds (None for anything but plain tensors)
PyObject* py_state_key(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded([&]() -> PyObject* {
    int64_t k[4 * 8];
    if (n < 1 || n > 8) return none();
    for (Py_ssize_t i = 0; i < n; ++i) {
      const Tensor* t = plain(v[i]);
      if (!t) return none();
      k[4 * i] = (int64_t)t->data_ptr();
      k[4 * i + 1] = (int64_t)t->_version();
      k[4 * i + 2] = (int64_t)t->scalar_type();
      k[4 * i + 3] = t->numel();
    }
    return PyBytes_FromStringAndSize((const char*)k, (Py_ssize_t)(n * 4 * sizeof(int64_t)));
  });
}

#define FAST(f) ((PyCFunction)(void (*)(void))(f))
PyMethodDef methods[] = {
    {"gemm_dq", FAST(py_gemm_dq), METH_FASTCALL, nullptr},
    {"quant_i8_pertoken", FAST(py_quant_i8_pertoken), METH_FASTCALL, nullptr},
    {"linear_i8", FAST(py_linear_i8), METH_FASTCALL, nullptr},
    {"linear_i8_static", FAST(py_linear_i8_static), METH_FASTCALL, nullptr},
    {"linear_fp8", FAST(py_linear_fp8), METH_FASTCALL, nullptr},
    {"state_key", FAST(py_state_key), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "fmsmo_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_fmsmo_host() { return PyModule_Create(&module_def); }
