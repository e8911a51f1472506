// One training or inference step of the layer around the operator (modules.DiffAttn) as two calls of a CPython extension
// module: the four projections are plain library products, everything between and behind them the library's kernels.
// modules.py decides when a layer goes this way and wires it into autograd.
//
// What the module's own graph of single operations spent beside the operator and its eight large products, B8 H8 N1024 d64
// causal fp16, in us of 709: four weight gradients 221 (library tiles of 64 x 64), the two q/k gradients put side by side 30,
// the three input gradients added up 17, the gain and its gradient 47, lambda and its gradients some 45 in 18 launches.
// Here the operator reads q, k and v from one [tokens, 3E] buffer that the projections fill and writes its gradients into another.
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <c10/core/impl/LocalDispatchKeySet.h>

#include "dispatch.hpp"
#include "layer_abi.h"

namespace {

constexpr int64_t kSeqMultiple = 128;

struct Released {
  PyThreadState* state = PyEval_SaveThread();
  ~Released() { PyEval_RestoreThread(state); }
};

PyObject* wrap(const at::Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}

// None is an undefined tensor where `optional` allows it
bool tensors(PyObject* const* a, int n, at::Tensor* out, bool optional = false) {
  for (int i = 0; i < n; ++i) {
    if (optional && a[i] == Py_None) continue;
    if (!THPVariable_Check(a[i])) {
      PyErr_Format(PyExc_TypeError, "argument %d must be a tensor", i);
      return false;
    }
    out[i] = THPVariable_Unpack(a[i]);
  }
  return true;
}

void check(int rc) {
  TORCH_CHECK(rc == DIFFATTN_OK, "libdiffattn: ", diffattn_strerror(rc), " (code ", rc, ")");
}

// t as the kernels read it: dense, 16-byte aligned (what autograd's saved-tensor hooks hand back may be neither) and without
// a pending negation, which only torch's own operations know of
at::Tensor dense(const at::Tensor& t) {
  if (!t.defined()) return t;
  at::Tensor c = t.resolve_neg().contiguous();
  return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 == 0 ? c : c.clone();
}

// t in another shape, for a result that nothing else holds.  Autograd would know a view as one made in a custom function, or
// under no_grad, and refuse to have it written in place, which the output of a layer often is (a residual added to it).
at::Tensor not_a_view(const at::Tensor& t, at::IntArrayRef sizes) { return at::_unsafe_view(t, sizes); }

// Sizes of a call.  d is the width of a q/k head; a value head is 2d wide and E = 2 H d.
struct Sizes {
  int64_t B, N, E, H, d, T, n_pad;
  int flags;
  Sizes(at::IntArrayRef x, at::ScalarType type, int64_t n_lambda, int64_t heads, bool causal)
      : B(x[0]), N(x[1]), E(x[2]), H(heads), d(E / (2 * heads)), T(B * N),
        n_pad((N + kSeqMultiple - 1) / kSeqMultiple * kSeqMultiple) {
    flags = DIFFATTN_RMS_NORM | DIFFATTN_LAMBDA_FP32;
    if (causal) flags |= DIFFATTN_CAUSAL;
    if (type == at::kBFloat16) flags |= DIFFATTN_BF16;
    if (n_lambda > 1) flags |= DIFFATTN_LAMBDA_PER_HEAD;
    if (n_pad != N) flags |= DIFFATTN_UNPADDED;
  }
  float sm_scale() const { return (float)(1.0 / std::sqrt((double)d)); }
  // q, k, v and their gradients in [tokens, 3E] buffers, heads and theirs in [tokens, E]
  diffattn_layout layout() const {
    const long long b3 = 3 * N * E, n3 = 3 * E, h = 2 * d, b1 = N * E, n1 = E;
    return {b3, h, n3, b3, h, n3, b1, h, n1, b1, h, n1, b3, h, n3, b3, h, n3};
  }
};

struct Parts { char *q1, *q2, *k1, *k2, *v; };
Parts parts(const at::Tensor& qkv, const Sizes& s) {
  char* p = (char*)qkv.data_ptr();
  const int64_t b = qkv.element_size();
  return {p, p + s.d * b, p + s.E * b, p + (s.E + s.d) * b, p + 2 * s.E * b};
}

diffattn_lambda_vectors vectors(const at::Tensor* l, const Sizes& s) {
  return {(const float*)l[0].data_ptr(), (const float*)l[1].data_ptr(), (const float*)l[2].data_ptr(), (const float*)l[3].data_ptr(),
          (int)(l[0].numel() / s.d), (int)s.d};
}

at::Tensor pack(const at::Tensor* w, const Sizes& s, const diffattn_lambda_vectors* vec, float lambda_init, float* lambda, void* stream) {
  const at::Tensor packed = at::empty({3 * s.E, s.E}, w[0].options());
  check(diffattn_layer_pack(w[0].data_ptr(), w[1].data_ptr(), w[2].data_ptr(), packed.data_ptr(), w[0].nbytes(), vec, lambda_init, lambda, stream));
  return packed;
}

// dqkv [T, 3E] times the three weights one below another: a single sum, rounded once, also where it is three products
at::Tensor input_gradient(const at::Tensor& dqkv, const at::Tensor* w, const Sizes& s, void* stream) {
  if (da_abi::layer_packed(true, s.E, s.T)) return at::mm(dqkv, pack(w, s, nullptr, 0.f, nullptr, stream));
  at::Tensor sum = at::mm(dqkv.narrow(1, 0, s.E), w[0], at::kFloat);
  for (int i = 1; i < 3; ++i) at::addmm_out(sum, sum, dqkv.narrow(1, i * s.E, s.E), w[i], at::kFloat);
  return sum.to(dqkv.scalar_type());
}

// out = a^T b for each job: one launch of the framework's kernel, or a library product each
struct Wgrad { at::Tensor a, b; };
bool wgrad_own(const std::vector<Wgrad>& jobs, int64_t E, int64_t T) { return T <= INT32_MAX && da_abi::wgrad_own((int)jobs.size(), E, T); }

std::vector<at::Tensor> weight_gradients(const std::vector<Wgrad>& jobs, int64_t E, int64_t T, int flags, bool own, void* stream) {
  std::vector<at::Tensor> out;
  if (jobs.empty()) return out;
  if (!own) {
    for (const Wgrad& j : jobs) out.push_back(at::mm(j.a.t(), j.b));
    return out;
  }
  diffattn_wgrad_job c[4];
  for (size_t i = 0; i < jobs.size(); ++i) {
    out.push_back(at::empty({E, E}, jobs[i].b.options()));
    c[i] = {jobs[i].a.data_ptr(), jobs[i].b.data_ptr(), out[i].data_ptr(), jobs[i].a.stride(0), jobs[i].b.stride(0)};
  }
  const size_t bytes = diffattn_layer_wgrad_workspace_bytes((int)jobs.size(), (int)T, (int)E);
  at::Tensor ws;
  if (bytes) ws = at::empty({(int64_t)bytes}, jobs[0].b.options().dtype(at::kByte));
  check(diffattn_layer_wgrad(c, (int)jobs.size(), (int)T, (int)E, bytes ? ws.data_ptr() : nullptr, bytes, flags & DIFFATTN_BF16, stream));
  return out;
}

// The projections run in the type of the layer, also where a backward is called under autocast.
const c10::DispatchKeySet kNoAutocast = c10::autocast_dispatch_keyset;

// layer_forward(x, wq, wk, wv, wo, gain, lq1, lk1, lq2, lk2, heads, causal, lambda_init, inner, outer, stream)
//   -> (y, qkv, heads, scaled heads, u2, row statistics, lambda).  `inner`: a backward will go behind the output projection;
//   without, qkv, heads, u2, the statistics and lambda are None.  `outer`: it will want that projection's weight gradient;
//   without, the scaled heads are None.
PyObject* layer_forward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 16) return PyErr_Format(PyExc_TypeError, "layer_forward takes 16 arguments");
  at::Tensor t[10];
  if (!tensors(a, 10, t)) return nullptr;
  const int64_t heads = PyLong_AsLongLong(a[10]);
  const bool causal = PyObject_IsTrue(a[11]) == 1;
  const double lambda_init = PyFloat_AsDouble(a[12]);
  const bool inner = PyObject_IsTrue(a[13]) == 1, outer = PyObject_IsTrue(a[14]) == 1;
  void* const stream = PyLong_AsVoidPtr(a[15]);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor y, qkv, hd, hg, u2, stats, lam;
  {
    const Released released;
    const c10::impl::ExcludeDispatchKeyGuard no_autocast(kNoAutocast);
    const at::Tensor &x = t[0], &wo = t[4], &gain = t[5];
    const Sizes s(x.sizes(), x.scalar_type(), t[6].dim() > 1 ? t[6].size(0) : 1, heads, causal);
    const at::Tensor x2 = x.reshape({s.T, s.E});
    lam = at::empty({t[6].numel() / s.d}, t[6].options());
    const diffattn_lambda_vectors vec = vectors(t + 6, s);
    if (da_abi::layer_packed(false, s.E, s.T)) {
      qkv = at::mm(x2, pack(t + 1, s, &vec, (float)lambda_init, (float*)lam.data_ptr(), stream).t());
    } else {
      check(diffattn_layer_pack(nullptr, nullptr, nullptr, nullptr, 0, &vec, (float)lambda_init, (float*)lam.data_ptr(), stream));
      qkv = at::empty({s.T, 3 * s.E}, x.options());
      for (int i = 0; i < 3; ++i) {
        at::Tensor out = qkv.narrow(1, i * s.E, s.E);
        at::mm_out(out, x2, t[1 + i].t());
      }
    }
    hg = at::empty({s.T, s.E}, qkv.options());
    float* st = nullptr;
    const int64_t rows = s.B * s.H * s.n_pad;
    if (inner) {
      hd = at::empty({s.T, s.E}, qkv.options());
      u2 = at::empty({s.B, s.H, s.n_pad, 2 * s.d}, qkv.options());
      stats = at::empty({3, rows}, qkv.options().dtype(at::kFloat));
      st = (float*)stats.data_ptr();
    }
    const Parts p = parts(qkv, s);
    const diffattn_layout layout = s.layout();
    check(diffattn_layer_forward(p.q1, p.q2, p.k1, p.k2, p.v, lam.data_ptr(), inner ? hd.data_ptr() : nullptr,
                                 inner ? u2.data_ptr() : nullptr, st, st ? st + rows : nullptr, st ? st + 2 * rows : nullptr,
                                 (int)s.B, (int)s.H, (int)s.n_pad, (int)s.N, (int)s.d, s.sm_scale(), (float)lambda_init, s.flags, &layout,
                                 gain.data_ptr(), hg.data_ptr(), stream));
    y = not_a_view(at::mm(hg, wo.t()), {s.B, s.N, s.E});
    if (!inner) qkv = lam = at::Tensor();
    if (!outer) hg = at::Tensor();
  }
  return Py_BuildValue("(NNNNNNN)", wrap(y), wrap(qkv), wrap(hd), wrap(hg), wrap(u2), wrap(stats), wrap(lam));
  END_HANDLE_TH_ERRORS
}

// wanted(ctx) -> bit i: the backward that is running wants a gradient of the i-th of the first ten tensors of the function
// that ctx belongs to.  ctx.needs_input_grad is fixed by the forward; grad(loss, x), or a backward with a list of inputs, wants
// less, and of the single operations the engine would run none behind the rest.  (A stand-in for the context, as compiled
// autograd has one, is no node that the engine could be asked about: all that needs a gradient is wanted.)
PyObject* wanted(PyObject*, PyObject* ctx) {
  HANDLE_TH_ERRORS
  unsigned bits = 0;
  THPObjectPtr need(PyObject_GetAttrString(ctx, "needs_input_grad"));
  if (!need) return nullptr;
  std::shared_ptr<torch::autograd::PyNode> node;
  if (THPFunction_Check(ctx)) node = ((THPFunction*)ctx)->cdata.lock();
  for (int i = 0; i < 10; ++i) {
    THPObjectPtr bit(PySequence_GetItem(need.get(), i));
    if (!bit) return nullptr;
    if (PyObject_IsTrue(bit.get()) == 1 && (!node || node->task_should_compute_output(i))) bits |= 1u << i;
  }
  return PyLong_FromUnsignedLong(bits);
  END_HANDLE_TH_ERRORS
}

// input_edge(ctx, i, like, sizes...) -> a tensor of unset values that stands in autograd's graph where tensor i of the function
// of ctx does: for a gradient that goes on to an input whose values nobody saved, because no gradient reads them
PyObject* input_edge(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n < 4 || !THPFunction_Check(a[0]) || !THPVariable_Check(a[2])) return PyErr_Format(PyExc_TypeError, "input_edge takes a context, an index, a tensor and sizes");
  const long i = PyLong_AsLong(a[1]);
  std::vector<int64_t> sizes;
  for (Py_ssize_t k = 3; k < n; ++k) sizes.push_back(PyLong_AsLongLong(a[k]));
  if (PyErr_Occurred()) return nullptr;
  const std::shared_ptr<torch::autograd::PyNode> node = ((THPFunction*)a[0])->cdata.lock();
  TORCH_CHECK(node && i >= 0 && (size_t)i < node->num_outputs(), "no such input");
  at::Tensor t = at::empty(sizes, THPVariable_Unpack(a[2]).options());
  if (node->next_edge(i).is_valid()) torch::autograd::impl::set_gradient_edge(t, node->next_edge(i));
  return wrap(t);
  END_HANDLE_TH_ERRORS
}

// layer_backward(x, wq, wk, wv, wo, gain, lq1, lk1, lq2, lk2, qkv, heads, scaled heads, u2, row statistics, lambda, dy,
//                B, N, heads, causal, lambda_init, wanted, stream)
//   -> the gradients of the first ten arguments; `wanted`: bit i says whether argument i's is, None where not.
//   What those do not take may be None: x without one of the q, k and v weights, these without x, and so on.
PyObject* layer_backward(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 24) return PyErr_Format(PyExc_TypeError, "layer_backward takes 24 arguments");
  at::Tensor t[17], grad[10];
  if (!tensors(a, 16, t, true) || !tensors(a + 16, 1, t + 16)) return nullptr;
  const int64_t B = PyLong_AsLongLong(a[17]), N = PyLong_AsLongLong(a[18]), heads = PyLong_AsLongLong(a[19]);
  const bool causal = PyObject_IsTrue(a[20]) == 1;
  const double lambda_init = PyFloat_AsDouble(a[21]);
  const unsigned wanted = (unsigned)PyLong_AsUnsignedLong(a[22]);
  void* const stream = PyLong_AsVoidPtr(a[23]);
  if (PyErr_Occurred()) return nullptr;
  {
    const Released released;
    const c10::impl::ExcludeDispatchKeyGuard no_autocast(kNoAutocast);
    auto want = [&](int i) { return (wanted >> i & 1u) != 0; };
    // of the tensors that a backward goes through first, one is always there
    const at::ScalarType type = (t[11].defined() ? t[11] : t[12]).scalar_type();
    const Sizes s({B, N, t[16].size(2)}, type, t[15].defined() ? t[15].numel() : 1, heads, causal);
    for (int i = 1; i < 16; ++i) t[i] = dense(t[i]);
    const at::Tensor x2 = t[0].defined() ? dense(t[0].reshape({s.T, s.E})) : t[0], dy = dense(t[16].to(type).reshape({s.T, s.E}));
    const at::Tensor &qkv = t[10], &hd = t[11], &hg = t[12], &u2 = t[13], &stats = t[14], &lam = t[15];
    const bool want_q = want(0) || want(1), want_kv = want(0) || want(2) || want(3);
    const bool want_lam = want(6) || want(7) || want(8) || want(9);
    std::vector<Wgrad> jobs;
    std::vector<int> which;
    at::Tensor dqkv, dlam, gpart;
    if (want_q || want_kv || want_lam || want(5)) {
      at::Tensor dhg = at::mm(dy, t[4]);
      dqkv = at::empty({s.T, 3 * s.E}, qkv.options());
      dlam = at::empty_like(lam);
      const int64_t n_part = (int64_t)diffattn_layer_gain_parts((int)s.B, (int)s.H, (int)s.n_pad, (int)s.d), rows = s.B * s.H * s.n_pad;
      gpart = at::empty({n_part, 2 * s.d}, lam.options());
      const size_t ws_bytes = diffattn_backward_workspace_bytes((int)s.B, (int)s.H, (int)s.n_pad, (int)s.d, s.flags);
      at::Tensor ws = at::empty({(int64_t)ws_bytes}, qkv.options().dtype(at::kByte));
      const unsigned stages = DIFFATTN_STAGE_PREP | (want_lam ? DIFFATTN_STAGE_DLAMBDA : 0u) | (want_kv ? DIFFATTN_STAGE_DKDV : 0u) |
                              (want_q ? DIFFATTN_STAGE_DQ : 0u);
      const Parts p = parts(qkv, s), d = parts(dqkv, s);
      const diffattn_layout layout = s.layout();
      const float* st = (const float*)stats.data_ptr();
      check(diffattn_layer_backward(p.q1, p.q2, p.k1, p.k2, p.v, lam.data_ptr(), hd.data_ptr(), u2.data_ptr(), st, st + rows, st + 2 * rows,
                                    dhg.data_ptr(), d.q1, d.q2, d.k1, d.k2, d.v, dlam.data_ptr(), ws.data_ptr(), ws_bytes,
                                    (int)s.B, (int)s.H, (int)s.n_pad, (int)s.N, (int)s.d, s.sm_scale(), (float)lambda_init, s.flags, stages,
                                    &layout, t[5].data_ptr(), (float*)gpart.data_ptr(), stream));
      dhg.reset();        // what follows on this stream may have their memory
      ws.reset();
      if (want(0)) grad[0] = not_a_view(input_gradient(dqkv, t + 1, s, stream), {s.B, s.N, s.E});
      if (want(5)) grad[5] = at::empty({2 * s.d}, hd.options());
      if (want_lam)
        for (int i = 6; i < 10; ++i) grad[i] = at::empty_like(t[i]);
      if (want(5) || want_lam) {
        const diffattn_lambda_vectors vec = want_lam ? vectors(t + 6, s) : diffattn_lambda_vectors{};
        auto f = [&](int i) { return want_lam ? (float*)grad[i].data_ptr() : nullptr; };
        check(diffattn_layer_finish((const float*)gpart.data_ptr(), (int)n_part, (int)(2 * s.d), want(5) ? grad[5].data_ptr() : nullptr, &vec,
                                    want_lam ? (const float*)dlam.data_ptr() : nullptr, f(6), f(7), f(8), f(9), s.flags & DIFFATTN_BF16, stream));
      }
      for (int i = 1; i < 4; ++i)
        if (want(i)) { jobs.push_back({dqkv.narrow(1, (i - 1) * s.E, s.E), x2}); which.push_back(i); }
    }
    if (want(4)) { jobs.push_back({dy, hg}); which.push_back(4); }
    const std::vector<at::Tensor> dw = weight_gradients(jobs, s.E, s.T, s.flags, wgrad_own(jobs, s.E, s.T), stream);
    for (size_t i = 0; i < dw.size(); ++i) grad[which[i]] = dw[i];
    for (int i = 6; i < 10; ++i)
      if (!want(i)) grad[i] = at::Tensor();
  }
  PyObject* out = PyTuple_New(10);
  if (!out) return nullptr;
  for (int i = 0; i < 10; ++i) {
    PyObject* g = wrap(grad[i]);
    if (!g) { Py_DECREF(out); return nullptr; }
    PyTuple_SET_ITEM(out, i, g);
  }
  return out;
  END_HANDLE_TH_ERRORS
}

// weight_gradient(a, b, stream) -> a^T b for [T, E] tensors, by the kernel that layer_backward uses for several weights
PyObject* weight_gradient(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3) return PyErr_Format(PyExc_TypeError, "weight_gradient takes 3 arguments");
  at::Tensor t[2], out;
  if (!tensors(a, 2, t)) return nullptr;
  void* const stream = PyLong_AsVoidPtr(a[2]);
  if (PyErr_Occurred()) return nullptr;
  TORCH_CHECK(t[0].dim() == 2 && t[0].sizes() == t[1].sizes() && t[0].is_cuda() && t[1].device() == t[0].device() &&
              t[0].scalar_type() == t[1].scalar_type() && (t[0].scalar_type() == at::kHalf || t[0].scalar_type() == at::kBFloat16) &&
              t[0].stride(1) == 1 && t[1].stride(1) == 1 && t[0].size(0) > 0 && t[0].size(0) <= INT32_MAX,
              "two 16-bit [T, E] tensors with contiguous rows");
  {
    const Released released;
    out = weight_gradients({{t[0], t[1]}}, t[0].size(1), t[0].size(0), t[0].scalar_type() == at::kBFloat16 ? DIFFATTN_BF16 : 0,
                           da_abi::wgrad_own(4, t[0].size(1), t[0].size(0)), stream)[0];
  }
  return wrap(out);
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"layer_forward", (PyCFunction)(void (*)())layer_forward, METH_FASTCALL, nullptr},
    {"layer_backward", (PyCFunction)(void (*)())layer_backward, METH_FASTCALL, nullptr},
    {"input_edge", (PyCFunction)(void (*)())input_edge, METH_FASTCALL, nullptr},
    {"wanted", (PyCFunction)wanted, METH_O, nullptr},
    {"weight_gradient", (PyCFunction)(void (*)())weight_gradient, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "diffattn_layer", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// A module that was built against another version of the library would call it with the wrong arguments.  The layer's
// functions change without those of diffattn.h, so both versions are asked for.
PyMODINIT_FUNC PyInit_diffattn_layer(void) {
  if (diffattn_layer_version() != DIFFATTN_LAYER_VERSION)
    return PyErr_Format(PyExc_ImportError, "libdiffattn has version %d of the layer's functions, diffattn_layer was built against %d: rebuild both",
                        diffattn_layer_version(), DIFFATTN_LAYER_VERSION);
  if (diffattn_abi_version() != DIFFATTN_ABI_VERSION)
    return PyErr_Format(PyExc_ImportError, "libdiffattn has ABI version %d, diffattn_layer was built against %d: rebuild both",
                        diffattn_abi_version(), DIFFATTN_ABI_VERSION);
  return PyModule_Create(&module);
}
