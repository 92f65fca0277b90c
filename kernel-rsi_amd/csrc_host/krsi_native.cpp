// Eager path of the public functions in native code: argument tests, output and workspace allocation,
// launch, and the autograd node, for the plain case of each call. The kernels are those of the C ABI;
// what this replaces is the Python around them, whose backward ran in torch's device thread, took
// the interpreter lock there and cost more than the kernels at the smaller sizes (host time of a
// forward and backward of rmsnorm x [256, 1152]: 102 -> 32 us, of which torch takes 20 for any node).
//
// Every function returns None for whatever is not the plain case (tracing, functorch transforms, dispatch
// modes, tensor subclasses, forward-mode duals, layouts that need a copy, arguments that are refused): the
// caller then takes its Python path, which handles it or raises. So no message or rule of
// validation is repeated here, and nothing has been launched when None is returned.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <ATen/ATen.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <pybind11/pybind11.h>

#include "krsi.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// A status other than KRSI_OK in a forward: nothing was launched; the Python path reports it.
struct NotPlain {};

void* stream_of(const Tensor& t) {
  return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream();
}

void forward_status(int rc) {
  if (rc != KRSI_OK) throw NotPlain{};
}

// The module that holds the type of a kernel status as an error, KrsiError, and the assignable workspace cap
// RELPOS_BWD_WORKSPACE_MAX (None or bytes).
PyObject* g_hip_module = nullptr;

// A Python error raised here, as torch's own, which its engine carries between threads. With the
// interpreter lock held.
[[noreturn]] void throw_python_error() {
  python_error err;
  err.persist();
  throw err;
}
void backward_status(int rc) {
  if (rc == KRSI_OK) return;
  pybind11::gil_scoped_acquire lock;
  PyObject* type = g_hip_module ? PyObject_GetAttrString(g_hip_module, "KrsiError") : nullptr;
  if (type) {
    PyErr_SetString(type, krsi_error_string(rc));
    Py_DECREF(type);
  } else if (!PyErr_Occurred()) {
    PyErr_SetString(PyExc_RuntimeError, krsi_error_string(rc));
  }
  throw_python_error();
}

// KRSI_DTYPE_* of an activation dtype, or -1.
int dtype_code(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kBFloat16: return KRSI_DTYPE_BF16;
    case at::kHalf: return KRSI_DTYPE_F16;
    case at::kFloat: return KRSI_DTYPE_F32;
    default: return -1;
  }
}

bool aligned16(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }

// No transform, mode or tracer that has to see the call.
bool plain_context() {
  if (torch::jit::tracer::isTracing() || c10::impl::TorchDispatchModeTLS::any_modes_set()) return false;
  const auto on = c10::impl::tls_local_dispatch_key_set().included_;
  return !on.has_any(c10::DispatchKeySet({c10::DispatchKey::FuncTorchDynamicLayerFrontMode,
                                          c10::DispatchKey::FuncTorchDynamicLayerBackMode, c10::DispatchKey::Python,
                                          c10::DispatchKey::Functionalize}));
}
// A strided GPU tensor with storage: no subclass that dispatches, no wrapper, no dual, not nested (whose sizes
// throw).
bool plain(const Tensor& t) {
  if (t.is_nested() || !t.is_cuda() || t.layout() != at::kStrided || !t.has_storage() || t.is_conj() || t.is_neg()) return false;
  const auto keys = t.key_set();
  if (keys.has_any(c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                        c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize})))
    return false;
  return !t._fw_grad(0).defined();
}

// A saved tensor can come back from a saved-tensor hook as anything: what a kernel reads by pointer has
// to be where, of the type and of the shape that the forward saved.
void check_saved(const char* name, const Tensor& t, const Tensor& grad, at::ScalarType dtype, at::IntArrayRef sizes) {
  TORCH_CHECK_VALUE(t.is_cuda() && t.device() == grad.device(), "saved ", name, " came back on ", t.device(),
                    ", the gradient is on ", grad.device());
  TORCH_CHECK_TYPE(t.scalar_type() == dtype, "saved ", name, " came back as ", t.scalar_type(), ", not ", dtype);
  TORCH_CHECK_VALUE(t.sizes() == sizes, "saved ", name, " came back with shape ", t.sizes(), ", not ", sizes);
}

// ------------------------------------------------------------------- RMSNorm
struct RmsNormFn : torch::autograd::Function<RmsNormFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, double eps) {
    const int64_t rows = x.size(0), n = x.size(1);
    Tensor y = at::empty_like(x), rstd = at::empty({rows}, x.options().dtype(at::kFloat));
    forward_status(krsi_rmsnorm_fwd(x.data_ptr(), w.data_ptr(), y.data_ptr(), rstd.data_ptr<float>(), rows, (int)n,
                                    (float)eps, dtype_code(x), stream_of(x)));
    ctx->save_for_backward({x, w, rstd});
    return y;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor g = grads[0].contiguous(), x = saved[0].contiguous(), w = saved[1].contiguous(),
                 rstd = saved[2].contiguous();
    const int64_t rows = g.size(0), n = g.size(1);
    check_saved("x2d", x, g, g.scalar_type(), {rows, n});
    check_saved("weight", w, g, g.scalar_type(), {n});
    check_saved("rstd", rstd, g, at::kFloat, {rows});
    Tensor dx = at::empty_like(x), dw = at::empty({n}, w.options());
    const size_t bytes = krsi_rmsnorm_bwd_workspace_bytes(rows, (int)n);
    Tensor ws = at::empty({(int64_t)bytes}, x.options().dtype(at::kByte));
    backward_status(krsi_rmsnorm_bwd(g.data_ptr(), x.data_ptr(), w.data_ptr(), rstd.data_ptr<float>(), dx.data_ptr(),
                                     dw.data_ptr(), ws.data_ptr(), bytes, rows, (int)n, dtype_code(x), stream_of(x)));
    return {dx, dw, Tensor()};
  }
};

// --------------------------------------------------------------------- GEGLU
struct GegluFn : torch::autograd::Function<GegluFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& u, int64_t approximate) {
    const int64_t rows = u.size(0), f = u.size(1) / 2;
    Tensor out = at::empty({rows, f}, u.options());
    forward_status(krsi_geglu_fwd(u.data_ptr(), out.data_ptr(), rows, (int)f, (int)approximate, dtype_code(u),
                                  stream_of(u)));
    ctx->save_for_backward({u});
    ctx->saved_data["approximate"] = approximate;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const Tensor g = grads[0].contiguous(), u = ctx->get_saved_variables()[0].contiguous();
    check_saved("u", u, g, g.scalar_type(), {g.size(0), 2 * g.size(1)});
    Tensor du = at::empty_like(u);
    backward_status(krsi_geglu_bwd(g.data_ptr(), u.data_ptr(), du.data_ptr(), u.size(0), (int)(u.size(1) / 2),
                                   (int)ctx->saved_data["approximate"].toInt(), dtype_code(u), stream_of(u)));
    return {du, Tensor()};
  }
};

struct GegluLinearFn : torch::autograd::Function<GegluLinearFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, int64_t approximate) {
    const int64_t rows = x.size(0), k = x.size(1), f = w.size(0) / 2;
    Tensor out = at::empty({rows, f}, x.options());
    forward_status(krsi_geglu_linear_fwd(x.data_ptr(), w.data_ptr(), out.data_ptr(), rows, (int)k, (int)f,
                                         (int)approximate, dtype_code(x), stream_of(x)));
    ctx->save_for_backward({x, w});
    ctx->saved_data["approximate"] = approximate;
    ctx->saved_data["k"] = k;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const Tensor &x = saved[0], &w = saved[1];
    const int approximate = (int)ctx->saved_data["approximate"].toInt();
    const int64_t rows = grads[0].size(0), k = ctx->saved_data["k"].toInt(), f = grads[0].size(1);
    check_saved("x", x, grads[0], grads[0].scalar_type(), {rows, k});
    check_saved("weight", w, grads[0], grads[0].scalar_type(), {2 * f, k});
    const Tensor g = grads[0].contiguous(), xc = x.contiguous(), wc = w.contiguous();
    Tensor du = at::empty({rows, 2 * f}, x.options());
    if (aligned16(xc) && aligned16(wc)) {
      backward_status(krsi_geglu_linear_bwd(g.data_ptr(), xc.data_ptr(), wc.data_ptr(), du.data_ptr(), rows, (int)k,
                                            (int)f, approximate, dtype_code(x), stream_of(x)));
    } else {  // a saved tensor that came back elsewhere
      const Tensor u = at::linear(xc, wc);
      backward_status(krsi_geglu_bwd(g.data_ptr(), u.data_ptr(), du.data_ptr(), rows, (int)f, approximate,
                                     dtype_code(x), stream_of(x)));
    }
    const bool need_dx = ctx->needs_input_grad(0), need_dw = ctx->needs_input_grad(1);
    // Not under create_graph, where torch's products carry a graph on.
    if (!at::GradMode::is_enabled() && x.is_contiguous() && w.is_contiguous() &&
        aligned16(x) && aligned16(w) && krsi_geglu_linear_grads_pays(rows, (int)k, (int)f, need_dx, need_dw) == 1) {
      Tensor dx, dw, ws;
      const size_t bytes = krsi_geglu_linear_grads_workspace_bytes(rows, (int)k, (int)f);
      if (bytes) ws = at::empty({(int64_t)bytes}, x.options().dtype(at::kByte));
      if (need_dx) dx = at::empty_like(x);
      if (need_dw) dw = at::empty_like(w);
      backward_status(krsi_geglu_linear_grads(du.data_ptr(), x.data_ptr(), w.data_ptr(),
                                              need_dx ? dx.data_ptr() : nullptr, need_dw ? dw.data_ptr() : nullptr,
                                              bytes ? ws.data_ptr() : nullptr, bytes, rows, (int)k, (int)f,
                                              dtype_code(x), stream_of(x)));
      return {dx, dw, Tensor()};
    }
    return {need_dx ? at::mm(du, w) : Tensor(), need_dw ? at::mm(du.t(), x) : Tensor(), Tensor()};
  }
};

// ------------------------------------------------ relative-position attention
// The workspace of a backward whose full size is `full`: the cap where one is assigned, but no less than
// `least`. Takes the interpreter lock, which torch's device thread owns a state for.
size_t workspace_bytes(size_t full, size_t least) {
  pybind11::gil_scoped_acquire lock;
  if (!g_hip_module) return full;
  try {
    const pybind11::object cap = pybind11::handle(g_hip_module).attr("RELPOS_BWD_WORKSPACE_MAX");
    if (cap.is_none() || !(cap < pybind11::int_(full))) return full;  // raises for what is no number
    const int64_t bytes = pybind11::int_(cap).cast<int64_t>();        // below full, which fits
    return bytes < (int64_t)least ? least : (size_t)bytes;
  } catch (pybind11::error_already_set& e) {
    e.restore();
    throw_python_error();
  }
}

struct Dims {
  int B, S, H, D;
  double scale;
};

Tensor relpos_forward(const Tensor& qkv, const Tensor& pd, const Dims& d, Tensor* out32, Tensor* lse) {
  const Tensor p = pd.contiguous();
  Tensor out = at::empty({(int64_t)d.B * d.S, (int64_t)d.H * d.D}, qkv.options());
  if (out32) {
    *out32 = at::empty(out.sizes(), qkv.options().dtype(at::kFloat));
    *lse = at::empty({(int64_t)d.B * d.H, d.S}, qkv.options().dtype(at::kFloat));
  }
  forward_status(krsi_relpos_fwd(qkv.data_ptr(), qkv.stride(0), p.data_ptr<float>(), out.data_ptr(),
                                 out32 ? out32->data_ptr<float>() : nullptr, lse ? lse->data_ptr<float>() : nullptr,
                                 d.B, d.S, d.H, d.D, (float)d.scale, dtype_code(qkv), stream_of(qkv)));
  return out;
}

struct RelposFn : torch::autograd::Function<RelposFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& qkv, const Tensor& pd, int64_t B, int64_t S, int64_t H,
                        int64_t D, double scale) {
    Tensor out32, lse;
    Tensor out = relpos_forward(qkv, pd, Dims{(int)B, (int)S, (int)H, (int)D, scale}, &out32, &lse);
    ctx->save_for_backward({qkv, pd, out32, lse});
    ctx->saved_data["dims"] = std::vector<int64_t>{B, S, H, D};
    ctx->saved_data["scale"] = scale;
    return out;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto saved = ctx->get_saved_variables();
    const auto d = ctx->saved_data["dims"].toIntVector();
    const int64_t B = d[0], S = d[1], H = d[2], D = d[3], cols = 3 * H * D;
    const Tensor &qkv = saved[0], dout = grads[0].contiguous(), pd = saved[1].contiguous(),
                 out32 = saved[2].contiguous(), lse = saved[3].contiguous();
    check_saved("qkv", qkv, dout, dout.scalar_type(), {B * S, qkv.dim() == 2 ? qkv.size(1) : cols});
    TORCH_CHECK_VALUE(qkv.size(1) >= cols && qkv.stride(1) == 1, "saved qkv came back with shape ", qkv.sizes(),
                      " and strides ", qkv.strides());
    check_saved("pd", pd, dout, at::kFloat, {H, 2 * S - 1});
    check_saved("out32", out32, dout, at::kFloat, {B * S, H * D});
    check_saved("lse", lse, dout, at::kFloat, {B * H, S});
    // Rows on 16-byte boundaries, which the width of a slice may not give.
    const int64_t per = 16 / qkv.element_size(), width = qkv.size(1), ld = (width + per - 1) / per * per;
    Tensor dqkv = at::empty({B * S, ld}, qkv.options());
    if (ld > width) dqkv = dqkv.narrow(1, 0, width);
    if (width > cols) dqkv.narrow(1, cols, width - cols).zero_();
    Tensor dpd = at::empty({H, 2 * S - 1}, pd.options());
    const size_t bytes = workspace_bytes(krsi_relpos_bwd_workspace_bytes((int)B, (int)S, (int)H, (int)D),
                                         krsi_relpos_bwd_workspace_min_bytes((int)B, (int)S, (int)H, (int)D));
    Tensor ws = at::empty({(int64_t)bytes}, qkv.options().dtype(at::kByte));
    backward_status(krsi_relpos_bwd(dout.data_ptr(), qkv.data_ptr(), qkv.stride(0), pd.data_ptr<float>(),
                                    out32.data_ptr<float>(), lse.data_ptr<float>(), dqkv.data_ptr(), dqkv.stride(0),
                                    dpd.data_ptr<float>(), ws.data_ptr(), bytes, (int)B, (int)S, (int)H, (int)D,
                                    (float)ctx->saved_data["scale"].toDouble(), dtype_code(qkv), stream_of(qkv)));
    return {dqkv, dpd, Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

struct BucketFn : torch::autograd::Function<BucketFn> {
  static Tensor forward(AutogradContext* ctx, const Tensor& table, const Tensor& bucket, int64_t S) {
    const Tensor t = table.contiguous();
    const int64_t nb = t.size(0), H = t.size(1);
    Tensor pd = at::empty({H, 2 * S - 1}, t.options());
    forward_status(krsi_relpos_bucket_gather(t.data_ptr<float>(), bucket.data_ptr<int32_t>(), pd.data_ptr<float>(),
                                             (int)S, (int)H, (int)nb, stream_of(t)));
    ctx->save_for_backward({bucket});
    ctx->saved_data["dims"] = std::vector<int64_t>{S, nb};
    return pd;
  }
  static variable_list backward(AutogradContext* ctx, variable_list grads) {
    const auto d = ctx->saved_data["dims"].toIntVector();
    const int64_t S = d[0], nb = d[1];
    const Tensor g = grads[0].contiguous(), bucket = ctx->get_saved_variables()[0].contiguous();
    check_saved("bucket", bucket, g, at::kInt, {2 * S - 1});
    Tensor dtable = at::empty({nb, g.size(0)}, g.options());
    backward_status(krsi_relpos_bucket_sum(g.data_ptr<float>(), bucket.data_ptr<int32_t>(), dtable.data_ptr<float>(),
                                           (int)S, (int)g.size(0), (int)nb, stream_of(g)));
    return {dtable, Tensor(), Tensor()};
  }
};

// ---------------------------------------------------------------- Python entries
// An entry as Python calls it: C++ exceptions, of the argument tests too, become Python ones.
using Args = PyObject* const*;
template <PyObject* (*F)(Args, Py_ssize_t)>
PyObject* entry(PyObject*, Args a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  return F(a, n);
  END_HANDLE_TH_ERRORS
}

// The result of fn, None when the call is not plain.
struct ReleaseLock {  // the interpreter lock, as torch's own bindings release it around an operator
  PyThreadState* state = PyEval_SaveThread();
  ~ReleaseLock() { PyEval_RestoreThread(state); }
};
template <typename Fn>
PyObject* unlocked(Fn&& fn) {
  try {
    Tensor out;
    {
      ReleaseLock released;
      out = fn();
    }
    return THPVariable_Wrap(std::move(out));
  } catch (const NotPlain&) {
    Py_RETURN_NONE;
  }
}

bool tensor_arg(PyObject* o, const Tensor** t) {
  if (!THPVariable_CheckExact(o)) return false;  // Tensor or Parameter: a subclass keeps its type in Python
  *t = &THPVariable_Unpack(o);
  return plain(**t);
}
bool int_arg(PyObject* o, int64_t lo, int64_t hi, int64_t* v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  *v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return !overflow && *v >= lo && *v <= hi;
}
bool float_arg(PyObject* o, double* v) {
  if (!PyFloat_CheckExact(o)) return false;
  *v = PyFloat_AS_DOUBLE(o);
  return true;
}
constexpr int64_t kIntMax = 0x7fffffff;

PyObject* py_rmsnorm(Args a, Py_ssize_t n) {
  const Tensor *x, *w;
  double eps;
  if (n != 3 || !plain_context() || !tensor_arg(a[0], &x) || !tensor_arg(a[1], &w) || !float_arg(a[2], &eps))
    Py_RETURN_NONE;
  if (x->dim() != 2 || !x->is_contiguous() || x->size(0) == 0 || dtype_code(*x) < 0 ||
      w->scalar_type() != x->scalar_type() || w->dim() != 1 || w->size(0) != x->size(1) || !w->is_contiguous() ||
      w->device() != x->device() || x->size(1) > kIntMax)
    Py_RETURN_NONE;
  return unlocked([&] { return RmsNormFn::apply(*x, *w, eps); });
}

PyObject* py_geglu(Args a, Py_ssize_t n) {
  const Tensor* u;
  int64_t approximate;
  if (n != 2 || !plain_context() || !tensor_arg(a[0], &u) || !int_arg(a[1], 0, 1, &approximate)) Py_RETURN_NONE;
  if (u->dim() != 2 || !u->is_contiguous() || u->numel() == 0 || u->size(1) % 2 || dtype_code(*u) < 0 ||
      u->size(1) > kIntMax)
    Py_RETURN_NONE;
  return unlocked([&] { return GegluFn::apply(*u, approximate); });
}

PyObject* py_geglu_linear(Args a, Py_ssize_t n) {
  const Tensor *x, *w;
  int64_t approximate;
  if (n != 3 || !plain_context() || !tensor_arg(a[0], &x) || !tensor_arg(a[1], &w) ||
      !int_arg(a[2], 0, 1, &approximate))
    Py_RETURN_NONE;
  if (x->dim() != 2 || w->dim() != 2 || (x->scalar_type() != at::kBFloat16 && x->scalar_type() != at::kHalf) ||
      w->scalar_type() != x->scalar_type() || w->device() != x->device() || w->size(1) != x->size(1) ||
      x->size(0) == 0 || x->size(1) % 64 || w->size(0) % 128 || x->size(1) > kIntMax || w->size(0) > kIntMax ||
      !x->is_contiguous() || !w->is_contiguous())
    Py_RETURN_NONE;
  return unlocked([&] { return GegluLinearFn::apply(*x, *w, approximate); });
}

PyObject* py_relpos_attention(Args a, Py_ssize_t n) {
  const Tensor *qkv, *pd;
  int64_t B, S, H, D;
  double scale;
  if (n != 7 || !plain_context() || !tensor_arg(a[0], &qkv) || !tensor_arg(a[1], &pd) ||
      !int_arg(a[2], 1, kIntMax, &B) || !int_arg(a[3], 1, kIntMax, &S) || !int_arg(a[4], 1, kIntMax, &H) ||
      !int_arg(a[5], 8, 128, &D) || !float_arg(a[6], &scale))
    Py_RETURN_NONE;
  if (qkv->dim() != 2 || dtype_code(*qkv) < 0 || D % 8 || qkv->stride(1) != 1 ||
      qkv->stride(0) * qkv->element_size() % 16 || !aligned16(*qkv) || qkv->size(0) != B * S ||
      qkv->size(1) / 3 < H * D || pd->scalar_type() != at::kFloat || pd->dim() != 2 || pd->size(0) != H ||
      pd->size(1) != 2 * S - 1 || pd->device() != qkv->device())
    Py_RETURN_NONE;
  if (at::GradMode::is_enabled() && (qkv->requires_grad() || pd->requires_grad()))
    return unlocked([&] { return RelposFn::apply(*qkv, *pd, B, S, H, D, scale); });
  // No backward can follow: the kernels skip the fp32 output and lse it would need.
  return unlocked([&] {
    at::NoGradGuard no_grad;
    return relpos_forward(*qkv, *pd, Dims{(int)B, (int)S, (int)H, (int)D, scale}, nullptr, nullptr);
  });
}

PyObject* py_bucket_table(Args a, Py_ssize_t n) {
  const Tensor *table, *bucket;
  int64_t S;
  if (n != 3 || !plain_context() || !tensor_arg(a[0], &table) || !tensor_arg(a[1], &bucket) ||
      !int_arg(a[2], 1, kIntMax, &S))
    Py_RETURN_NONE;
  if (table->scalar_type() != at::kFloat || table->dim() != 2 || table->numel() == 0 ||
      table->size(0) > kIntMax || table->size(1) > kIntMax || bucket->scalar_type() != at::kInt ||
      bucket->dim() != 1 || bucket->size(0) != 2 * S - 1 || !bucket->is_contiguous() ||
      bucket->device() != table->device())
    Py_RETURN_NONE;
  return unlocked([&] { return BucketFn::apply(*table, *bucket, S); });
}

PyObject* py_set_module(PyObject*, PyObject* m) {
  Py_XDECREF(g_hip_module);
  Py_INCREF(m);
  g_hip_module = m;
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"rmsnorm", (PyCFunction)(void*)entry<py_rmsnorm>, METH_FASTCALL, nullptr},
    {"geglu", (PyCFunction)(void*)entry<py_geglu>, METH_FASTCALL, nullptr},
    {"geglu_linear", (PyCFunction)(void*)entry<py_geglu_linear>, METH_FASTCALL, nullptr},
    {"relpos_attention", (PyCFunction)(void*)entry<py_relpos_attention>, METH_FASTCALL, nullptr},
    {"bucket_table", (PyCFunction)(void*)entry<py_bucket_table>, METH_FASTCALL, nullptr},
    {"set_module", py_set_module, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_krsi_native", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// built_for: the torch, Python and krsi.h this file was compiled against, which its loader compares with its own.
PyMODINIT_FUNC PyInit__krsi_native() {
  PyObject* m = PyModule_Create(&kModule);
  PyObject* v = m ? Py_BuildValue("(siii)", KRSI_TORCH_VERSION, PY_MAJOR_VERSION, PY_MINOR_VERSION, KRSI_ABI_VERSION)
                  : nullptr;
  if (!v || PyModule_AddObject(m, "built_for", v) < 0) {
    Py_XDECREF(v);
    Py_XDECREF(m);
    return nullptr;
  }
  return m;
}
