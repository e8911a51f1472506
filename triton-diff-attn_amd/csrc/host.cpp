// The host side of one operator call -- input checks, output and workspace allocation, the call into libdiffattn -- as a
// CPython extension module.  kernel.py wires it into autograd and keeps what is not on every call's way: error
// messages, copies of inputs that cannot be read in place, a lambda given as a number, calls for another device than the
// current one.  (A small call is bound by its host work, and most of that was the interpreter walking over strides and
// marshalling some 25 arguments through ctypes: B1 H16 N77 D64 forward 20 us a call for a 10 us kernel.)
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>

#include "../../include/diffattn.h"

namespace {

constexpr int64_t kSeqMultiple = 128;

bool aligned(const at::Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// Whether the kernels can read t in place: contiguous rows, every other stride a non-negative multiple of 8 elements
// (16-byte aligned rows), base pointer 16-byte aligned.
bool strides_ok(const at::Tensor& t) {
  const auto s = t.strides();
  return s[3] == 1 && s[2] >= t.size(3) && s[2] % 8 == 0 && s[0] % 8 == 0 && s[1] % 8 == 0 && s[0] >= 0 && s[1] >= 0 &&
         s[2] <= (int64_t(1) << 26) && aligned(t);
}

// Whether b's elements lie where a's do, each from its base pointer: equal sizes and strides, but for the strides of
// dimensions of size 1, which address nothing (a slice of a fused [1, 2, H, N, d] projection keeps the stride of the whole).
bool same_layout(const at::Tensor& a, const at::Tensor& b) {
  if (a.sizes() != b.sizes()) return false;
  for (int64_t i = 0; i < a.dim(); ++i)
    if (a.size(i) != 1 && a.stride(i) != b.stride(i)) return false;
  return true;
}

bool is_dense(const at::Tensor& t) {
  const auto s = t.strides();
  const int64_t H = t.size(1), N = t.size(2), C = t.size(3);
  return s[3] == 1 && s[2] == C && s[1] == N * C && s[0] == H * N * C;
}

void put(long long* dst, const at::Tensor& t) {
  const auto s = t.strides();
  dst[0] = s[0]; dst[1] = s[1]; dst[2] = s[2];
}

bool unpack(PyObject* o, at::Tensor& t) {
  if (!THPVariable_Check(o)) return false;
  t = THPVariable_Unpack(o);
  return true;
}

PyObject* wrap(const at::Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}

void* ptr(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

PyObject* library_error(int rc) {
  return PyErr_Format(PyExc_RuntimeError, "libdiffattn: %s (code %d)", diffattn_strerror(rc), rc);
}

// Other threads run while a call allocates and launches: either may wait for the device.
struct Released {
  PyThreadState* state = PyEval_SaveThread();
  ~Released() { PyEval_RestoreThread(state); }
};

bool numbers_ok() { return !PyErr_Occurred(); }

// readable(t) -> whether the kernels can read the 4-dimensional tensor t in place (strides_ok above)
PyObject* readable(PyObject*, PyObject* o) {
  HANDLE_TH_ERRORS
  at::Tensor t;
  if (!unpack(o, t) || t.dim() != 4) return PyErr_Format(PyExc_TypeError, "readable takes a tensor of four dimensions");
  return PyBool_FromLong(strides_ok(t));
  END_HANDLE_TH_ERRORS
}

// forward(q1, q2, k1, k2, v, lambda, sm_scale, lambda_init, flags, dropout_p, dropout_seed, differentiable, device, stream,
//         as_is)
//   -> None when an input is not what the kernels read in place, else (y, u2, lse1, lse2, rinv, flags, n_pad)
// `as_is`: the caller has copied what copying helps; strides or pointers that the kernels still cannot read go to the library,
// whose refusal says what is wrong with them.
// u2, the two logsumexps and, with rms_norm, the norm statistic are what only a backward reads: None unless
// `differentiable`.  `flags`: DIFFATTN_RMS_NORM and DIFFATTN_CAUSAL from the caller, the others are added here.
PyObject* forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 15) return PyErr_Format(PyExc_TypeError, "forward takes 15 arguments");
  at::Tensor q[4], v, lam;
  for (int i = 0; i < 4; ++i)
    if (!unpack(a[i], q[i])) Py_RETURN_NONE;
  if (!unpack(a[4], v) || !unpack(a[5], lam)) Py_RETURN_NONE;
  const double sm_scale = PyFloat_AsDouble(a[6]), lambda_init = PyFloat_AsDouble(a[7]);
  int flags = (int)PyLong_AsLong(a[8]);
  const double p = PyFloat_AsDouble(a[9]);
  const unsigned long long seed = PyLong_AsUnsignedLongLongMask(a[10]);
  const bool differentiable = PyObject_IsTrue(a[11]) == 1;
  const long device = PyLong_AsLong(a[12]);
  void* const stream = PyLong_AsVoidPtr(a[13]);
  const bool as_is = PyObject_IsTrue(a[14]) == 1;
  if (!numbers_ok()) return nullptr;

  const auto type = q[0].scalar_type();
  if (type != at::kHalf && type != at::kBFloat16) Py_RETURN_NONE;
  for (const at::Tensor* t : {&q[0], &q[1], &q[2], &q[3], &v})
    if (t->scalar_type() != type || t->dim() != 4 || !t->is_cuda() || t->get_device() != device) Py_RETURN_NONE;
  const int64_t B = q[0].size(0), H = q[0].size(1), N = q[0].size(2), D = q[0].size(3);
  if (!as_is && !(strides_ok(q[0]) && strides_ok(v))) Py_RETURN_NONE;
  for (int i = 1; i < 4; ++i)       // the four q/k tensors are read through the strides of the first
    if (!same_layout(q[0], q[i]) || !(as_is || aligned(q[i]))) Py_RETURN_NONE;
  if (v.size(0) != B || v.size(1) != H || v.size(2) != N || v.size(3) != 2 * D || (D != 32 && D != 64 && D != 128) || N < 1) Py_RETURN_NONE;
  if (B > INT32_MAX || H > INT32_MAX || N > INT32_MAX - kSeqMultiple) Py_RETURN_NONE;
  if (!lam.is_cuda() || lam.get_device() != device || (lam.scalar_type() != type && lam.scalar_type() != at::kFloat) ||
      (lam.numel() != 1 && lam.numel() != H) || !lam.is_contiguous())
    Py_RETURN_NONE;

  const int64_t n_pad = (N + kSeqMultiple - 1) / kSeqMultiple * kSeqMultiple;
  const bool rms = flags & DIFFATTN_RMS_NORM;
  if (type == at::kBFloat16) flags |= DIFFATTN_BF16;
  if (lam.numel() > 1) flags |= DIFFATTN_LAMBDA_PER_HEAD;
  if (lam.scalar_type() == at::kFloat) flags |= DIFFATTN_LAMBDA_FP32;
  if (n_pad != N) flags |= DIFFATTN_UNPADDED;
  at::Tensor y, u2, lse1, lse2, rinv;
  int rc;
  {
    const Released released;
    y = at::empty_like(v);                                     // in v's layout when v is a permuted dense buffer, else dense
    if (differentiable) {
      u2 = at::empty({B, H, n_pad, 2 * D}, v.options());
      // the two logsumexps and the norm statistic share one allocation
      at::Tensor stats = at::empty({rms ? 3 : 2, B, H, n_pad}, v.options().dtype(at::kFloat));
      lse1 = stats.select(0, 0); lse2 = stats.select(0, 1);
      if (rms) rinv = stats.select(0, 2);
    }
    diffattn_layout layout = {};
    const bool dense = is_dense(q[0]) && is_dense(v) && is_dense(y);
    if (!dense) { put(&layout.qk_b, q[0]); put(&layout.v_b, v); put(&layout.y_b, y); put(&layout.dy_b, y); }
    const diffattn_dropout drop = {(float)p, seed};
    rc = diffattn_forward_padded(q[0].data_ptr(), q[1].data_ptr(), q[2].data_ptr(), q[3].data_ptr(), v.data_ptr(),
                                 lam.data_ptr(), y.data_ptr(), ptr(u2), (float*)ptr(lse1), (float*)ptr(lse2), (float*)ptr(rinv),
                                 (int)B, (int)H, (int)n_pad, (int)N, (int)D, (float)sm_scale, (float)lambda_init, flags,
                                 dense ? nullptr : &layout, p > 0 ? &drop : nullptr, stream);
  }
  if (rc != DIFFATTN_OK) return library_error(rc);
  return Py_BuildValue("(NNNNNiL)", wrap(y), wrap(u2), wrap(lse1), wrap(lse2), wrap(rinv), flags, (long long)n_pad);
  END_HANDLE_TH_ERRORS
}

// backward(q1, q2, k1, k2, v, y, u2, lse1, lse2, rinv, lambda, dy,
//          sm_scale, lambda_init, flags, n_pad, dropout_p, dropout_seed, stages, stream)
//   -> (dq1, dq2, dk1, dk2, dv, dlambda), None for what `stages` (the library's stage bits) does not ask for
// rinv may be None (no rms_norm).
// Gradients are written in the memory layout of the tensors they belong to (autograd would otherwise copy each one into
// its leaf's layout).  The four q/k gradients share one set of strides, like q1..k2.
PyObject* backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 20) return PyErr_Format(PyExc_TypeError, "backward takes 20 arguments");
  at::Tensor t[12];
  for (int i = 0; i < 12; ++i)
    if (!unpack(a[i], t[i]) && !(i == 9 && a[i] == Py_None)) return PyErr_Format(PyExc_TypeError, "argument %d of backward must be a tensor", i);
  const at::Tensor &q1 = t[0], &v = t[4], &y = t[5], &u2 = t[6], &lse1 = t[7], &lse2 = t[8], &rinv = t[9], &lam = t[10];
  const double sm_scale = PyFloat_AsDouble(a[12]), lambda_init = PyFloat_AsDouble(a[13]);
  const int flags = (int)PyLong_AsLong(a[14]);
  const int64_t n_pad = PyLong_AsLongLong(a[15]);
  const double p = PyFloat_AsDouble(a[16]);
  const unsigned long long seed = PyLong_AsUnsignedLongLongMask(a[17]);
  const unsigned stages = (unsigned)PyLong_AsUnsignedLong(a[18]);
  void* const stream = PyLong_AsVoidPtr(a[19]);
  if (!numbers_ok()) return nullptr;

  at::Tensor dq1, dq2, dk1, dk2, dv, dlam;
  int rc;
  {
    const Released released;
    at::Tensor dy = t[11];
    if (dy.scalar_type() != q1.scalar_type()) dy = dy.to(q1.scalar_type());
    if (!strides_ok(dy)) dy = dy.contiguous();
    const int64_t B = q1.size(0), H = q1.size(1), N = q1.size(2), D = q1.size(3);
    const bool want_kv = stages & DIFFATTN_STAGE_DKDV, want_q = stages & DIFFATTN_STAGE_DQ;
    if (want_q) { dq1 = at::empty_like(q1); dq2 = at::empty_like(q1); }
    if (want_kv) { dk1 = at::empty_like(q1); dk2 = at::empty_like(q1); dv = at::empty_like(v); }
    if (stages & DIFFATTN_STAGE_DLAMBDA) dlam = at::empty({lam.numel()}, lam.options());
    diffattn_layout layout = {};
    const bool dense = is_dense(q1) && is_dense(v) && is_dense(y) && is_dense(dy);
    if (!dense) {
      put(&layout.qk_b, q1); put(&layout.v_b, v); put(&layout.y_b, y); put(&layout.dy_b, dy);
      if (want_q || want_kv) put(&layout.dqk_b, want_q ? dq1 : dk1);   // (of a view that is not a permuted dense buffer: dense)
      if (want_kv) put(&layout.dv_b, dv);
    }
    const size_t ws_bytes = diffattn_backward_workspace_bytes((int)B, (int)H, (int)n_pad, (int)D, flags);
    at::Tensor ws = at::empty({(int64_t)ws_bytes}, q1.options().dtype(at::kByte));
    const diffattn_dropout drop = {(float)p, seed};
    rc = diffattn_backward_stages(q1.data_ptr(), t[1].data_ptr(), t[2].data_ptr(), t[3].data_ptr(), v.data_ptr(),
                                  lam.data_ptr(), y.data_ptr(), u2.data_ptr(), (const float*)lse1.data_ptr(),
                                  (const float*)lse2.data_ptr(), (const float*)ptr(rinv), dy.data_ptr(),
                                  ptr(dq1), ptr(dq2), ptr(dk1), ptr(dk2), ptr(dv), ptr(dlam), ws.data_ptr(), ws_bytes,
                                  (int)B, (int)H, (int)n_pad, (int)N, (int)D, (float)sm_scale, (float)lambda_init, flags,
                                  stages, dense ? nullptr : &layout, p > 0 ? &drop : nullptr, stream);
  }
  if (rc != DIFFATTN_OK) return library_error(rc);
  return Py_BuildValue("(NNNNNN)", wrap(dq1), wrap(dq2), wrap(dk1), wrap(dk2), wrap(dv), wrap(dlam));
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"readable", (PyCFunction)readable, METH_O, nullptr},
    {"forward", (PyCFunction)(void (*)())forward, METH_FASTCALL, nullptr},
    {"backward", (PyCFunction)(void (*)())backward, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "diffattn_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// A module that was built against another version of the library would call it with the wrong arguments.
PyMODINIT_FUNC PyInit_diffattn_host(void) {
  if (diffattn_abi_version() != DIFFATTN_ABI_VERSION)
    return PyErr_Format(PyExc_ImportError, "libdiffattn has ABI version %d, diffattn_host was built against %d: rebuild both",
                        diffattn_abi_version(), DIFFATTN_ABI_VERSION);
  return PyModule_Create(&module);
}
