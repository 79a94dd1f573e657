// Native host side of the operators: the dispatcher entries of alexdremov_streaming_attention::{forward, backward} and
// alexdremov_flash_attention::forward, their autograd, and the eager call path of the public Python functions
// (module streaming_attention._native).
//
// A call costs the host about as much as the kernels of a small problem run for, so nothing of it is Python: argument
// checks, output allocation, the current stream and the launch through the C ABI (include/streaming_attention.h) happen here.
// Measured on an MI355X, per call in a loop: float16 forward of B=1, H=8, T=200, D=64 17.7 us through Python adapters and
// ctypes, 7.5 us here (its kernel alone runs for 8 when traced); float32 training step of B=2, H=4, T=512, D=64 162 us, 69 us
// here (kernels 62); training step of B=16, H=8, T=2048 ragged, D=128 167 us, 132 us here, bound by its kernels.
//
// The shared library is opened on the first call, the one that STREAMING_ATTENTION_LIB names or the one beside this
// module; there is no other implementation.  Invalid arguments are handed to streaming_attention.ops._validate, which
// names the condition (AssertionError).
#include <Python.h>
#include <dlfcn.h>

#include <mutex>
#include <string>

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/library.h>

#include "../../include/streaming_attention.h"

namespace {

using at::Tensor;
using c10::SymInt;
using OptTensor = std::optional<Tensor>;

// ---- the shared library -------------------------------------------------------------------------------------
struct Api {
  decltype(&sa_forward) forward;
  decltype(&sa_backward) backward;
  decltype(&sa_error_string) error_string;
};

Api open_library() {
  std::string path;
  if (const char* env = getenv("STREAMING_ATTENTION_LIB")) {
    path = env;
  } else {
    Dl_info info;
    TORCH_CHECK(dladdr(reinterpret_cast<void*>(&open_library), &info) != 0, "cannot locate this module");
    path = info.dli_fname;
    path = path.substr(0, path.rfind('/') + 1) + "libstreaming_attention.so";
  }
  void* lib = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
  TORCH_CHECK(lib, "libstreaming_attention.so not found at ", path, " (", dlerror(),
              "): build it with `make -C kernels_amd/csrc`. There is no fallback implementation.");
  auto symbol = [&](const char* name) {
    void* p = dlsym(lib, name);
    TORCH_CHECK(p, path, " has no symbol ", name);
    return p;
  };
  return Api{reinterpret_cast<decltype(&sa_forward)>(symbol("sa_forward")),
             reinterpret_cast<decltype(&sa_backward)>(symbol("sa_backward")),
             reinterpret_cast<decltype(&sa_error_string)>(symbol("sa_error_string"))};
}
const Api& api() {
  static const Api a = open_library();   // tried again by the next call if it throws
  return a;
}
void check(int rc, const char* what) {
  TORCH_CHECK(rc == 0, what, " failed with code ", rc, ": ", api().error_string(rc));
}

// ---- argument checks and layout -------------------------------------------------------------------------------
int dtype_id(const Tensor& t) {
  switch (t.scalar_type()) {
    case at::kFloat: return SA_DTYPE_F32;
    case at::kHalf: return SA_DTYPE_F16;
    case at::kBFloat16: return SA_DTYPE_BF16;
    default: return -1;
  }
}

bool known_head_dim(int64_t d) { return d == 16 || d == 32 || d == 64 || d == 128 || d == 256; }

// q, k, v and `more` are alike in shape and device, and lens fits them.
bool plain(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& lens, std::initializer_list<const Tensor*> more) {
  if (q.dim() != 4 || dtype_id(q) < 0 || !known_head_dim(q.size(3))) return false;
  if (k.sizes() != q.sizes() || v.sizes() != q.sizes() || k.device() != q.device() || v.device() != q.device()) return false;
  if (k.scalar_type() != q.scalar_type() || v.scalar_type() != q.scalar_type()) return false;
  for (const Tensor* t : more)
    if (t->sizes() != q.sizes() || t->device() != q.device()) return false;
  return !lens || (lens->scalar_type() == at::kInt && lens->dim() == 1 && lens->size(0) == q.size(0) && lens->device() == q.device());
}

// Have Python's checks name what is wrong.
[[noreturn]] void explain(const char* module, const char* function, std::initializer_list<PyObject*> args) {
  PyObject* tuple = PyTuple_New((Py_ssize_t)args.size());
  Py_ssize_t i = 0;
  for (PyObject* a : args) PyTuple_SET_ITEM(tuple, i++, a);   // takes the reference
  PyObject* m = PyImport_ImportModule(module);
  PyObject* f = m ? PyObject_GetAttrString(m, function) : nullptr;
  PyObject* r = f ? PyObject_CallObject(f, tuple) : nullptr;
  Py_XDECREF(r);
  Py_XDECREF(f);
  Py_XDECREF(m);
  Py_DECREF(tuple);
  if (PyErr_Occurred()) throw python_error();
  TORCH_CHECK(false, "unsupported arguments");
}
PyObject* wrap(const OptTensor& t) {
  if (t) return THPVariable_Wrap(*t);
  Py_RETURN_NONE;
}

// The tensor itself when the kernels can read it in place (unit stride along the head dimension, the others and the base
// address multiples of 16 bytes, rows that advance), otherwise a contiguous copy.  The 16-bit kernels for head
// dimensions from 32 on address the rows of a (batch, head) slice with 32-bit byte offsets.
Tensor kernel_layout(const Tensor& t) {
  const int64_t es = t.element_size(), vec = 16 / es, T = t.size(2);
  const auto s = t.strides();
  const bool fits = !(es == 2 && t.size(3) >= 32) || (T + 1024) * s[2] * es < (int64_t(1) << 32);
  const bool ok = s[3] == 1 && s[0] % vec == 0 && s[1] % vec == 0 && s[2] % vec == 0 && (s[2] > 0 || T <= 1) &&
                  reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0 && fits;
  if (ok) return t;
  return t.is_contiguous() ? t.clone(at::MemoryFormat::Contiguous) : t.contiguous();
}

int clamp_int(int64_t x) { return (int)std::min<int64_t>(x, 0x7fffffff); }

struct Launch {   // what every launch on q's problem takes
  c10::OptionalDeviceGuard guard;
  const int32_t* lens = nullptr;
  int64_t lens_stride = 0;
  int B, H, T, D, dtype;
  void* stream;
  Launch(const Tensor& q, const OptTensor& l)
      : guard(q.device()), B((int)q.size(0)), H((int)q.size(1)), T((int)q.size(2)), D((int)q.size(3)), dtype(dtype_id(q)),
        stream(c10::hip::getCurrentHIPStream(q.device().index()).stream()) {
    if (l) lens = l->const_data_ptr<int32_t>(), lens_stride = l->stride(0);
  }
};
const void* ptr(const Tensor& t) { return t.const_data_ptr(); }
void* out_ptr(const Tensor& t) { return t.mutable_data_ptr(); }

Tensor empty_rows(const Tensor& q) { return at::empty({q.size(0), q.size(1), q.size(2)}, q.options().dtype(at::kFloat)); }
Tensor empty_same(const Tensor& q) { return at::empty(q.sizes(), q.options()); }

// ---- streaming attention --------------------------------------------------------------------------------------
void validate(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& lens, int64_t context_size,
              int64_t back_contexts, double sm_scale, std::initializer_list<const Tensor*> more = {}) {
  if (C10_LIKELY(back_contexts >= 0 && context_size >= 1 && plain(q, k, v, lens, more))) return;
  PyGILState_STATE gil = PyGILState_Ensure();
  struct Release { PyGILState_STATE s; ~Release() { PyGILState_Release(s); } } release{gil};
  PyObject *q_ = THPVariable_Wrap(q), *k_ = THPVariable_Wrap(k), *v_ = THPVariable_Wrap(v), *l_ = wrap(lens);
  PyObject *c_ = PyLong_FromLongLong(context_size), *r_ = PyLong_FromLongLong(back_contexts), *s_ = PyFloat_FromDouble(sm_scale);
  if (more.size() == 2)
    explain("streaming_attention.ops", "_validate",
            {q_, k_, v_, l_, c_, r_, s_, THPVariable_Wrap(**more.begin()), THPVariable_Wrap(**(more.begin() + 1))});
  explain("streaming_attention.ops", "_validate", {q_, k_, v_, l_, c_, r_, s_});
}

std::tuple<Tensor, Tensor> forward_gpu(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& lens,
                                       int64_t context_size, int64_t back_contexts, double sm_scale, bool autotune,
                                       bool return_lse, bool prescale_qk, c10::string_view precision) {
  validate(q, k, v, lens, context_size, back_contexts, sm_scale);
  const Api& a = api();
  Launch l(q, lens);
  // the kernel writes every element (zeros at padded positions included)
  Tensor o = empty_same(q);
  Tensor lse = return_lse ? empty_rows(q) : at::empty({0});
  if (q.numel() > 0) {
    const Tensor qk = kernel_layout(q), kk = kernel_layout(k), vk = kernel_layout(v);
    check(a.forward(ptr(qk), ptr(kk), ptr(vk), l.lens, l.lens_stride, out_ptr(o),
                    return_lse ? (float*)out_ptr(lse) : nullptr, qk.strides().data(), kk.strides().data(), vk.strides().data(),
                    l.B, l.H, l.T, l.D, clamp_int(context_size), clamp_int(back_contexts), (float)sm_scale, l.dtype, l.stream),
          "sa_forward");
  }
  return {std::move(o), std::move(lse)};
}

std::tuple<Tensor, Tensor, Tensor> backward_gpu(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& lens,
                                                const Tensor& o, const Tensor& lse_in, const Tensor& d_o,
                                                int64_t context_size, int64_t back_contexts, double sm_scale,
                                                bool autotune, bool prescale_qk, c10::string_view precision) {
  validate(q, k, v, lens, context_size, back_contexts, sm_scale, {&o, &d_o});
  const Api& a = api();
  Launch l(q, lens);
  Tensor dq = empty_same(q), dk = empty_same(q), dv = empty_same(q);
  if (q.numel() == 0) return {std::move(dq), std::move(dk), std::move(dv)};
  const Tensor qk = kernel_layout(q), kk = kernel_layout(k), vk = kernel_layout(v);
  // the upstream gradient may arrive in another type and with arbitrary strides
  const Tensor gk = kernel_layout(d_o.to(q.scalar_type())), ok = kernel_layout(o.to(q.scalar_type()));
  const int C = clamp_int(context_size), R = clamp_int(back_contexts);
  Tensor lse = lse_in;
  if (lse.numel() != q.numel() / l.D || lse.device() != q.device()) {
    // forward was run with return_lse=False: rebuild the log-sum-exp
    lse = empty_rows(q);
    Tensor scratch = empty_same(q);
    check(a.forward(ptr(qk), ptr(kk), ptr(vk), l.lens, l.lens_stride, out_ptr(scratch), (float*)out_ptr(lse),
                    qk.strides().data(), kk.strides().data(), vk.strides().data(), l.B, l.H, l.T, l.D, C, R, (float)sm_scale,
                    l.dtype, l.stream),
          "sa_forward (log-sum-exp rebuild)");
  }
  lse = lse.to(at::kFloat).contiguous();
  Tensor delta = empty_rows(q);
  check(a.backward(ptr(qk), ptr(kk), ptr(vk), l.lens, l.lens_stride, ptr(ok), ptr(gk), (const float*)ptr(lse),
                   (float*)out_ptr(delta), out_ptr(dq), out_ptr(dk), out_ptr(dv), qk.strides().data(), kk.strides().data(),
                   vk.strides().data(), ok.strides().data(), gk.strides().data(), l.B, l.H, l.T, l.D, C, R, (float)sm_scale,
                   l.dtype, l.stream),
        "sa_backward");
  return {std::move(dq), std::move(dk), std::move(dv)};
}

using ForwardOp = std::tuple<Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const OptTensor&, SymInt, SymInt,
                                             double, bool, bool, bool, c10::string_view);
using BackwardOp = std::tuple<Tensor, Tensor, Tensor>(const Tensor&, const Tensor&, const Tensor&, const OptTensor&,
                                                      const Tensor&, const Tensor&, const Tensor&, SymInt, SymInt, double,
                                                      bool, bool, c10::string_view);
const c10::TypedOperatorHandle<ForwardOp>& forward_op() {
  static const auto op = c10::Dispatcher::singleton()
                             .findSchemaOrThrow("alexdremov_streaming_attention::forward", "")
                             .typed<ForwardOp>();
  return op;
}
const c10::TypedOperatorHandle<BackwardOp>& backward_op() {
  static const auto op = c10::Dispatcher::singleton()
                             .findSchemaOrThrow("alexdremov_streaming_attention::backward", "")
                             .typed<BackwardOp>();
  return op;
}

// Autograd glue of the forward op (src/streaming_attention/kernel.py:1467-1530): saves q, k, v, O, LSE and lens, hands dO to
// the backward op, lets no gradient flow through the log-sum-exp (kernel.py:1498): it leaves through lse_out, beside the
// node's one output.  An output marked as not differentiable would be refused by compiled autograd, which takes native
// nodes without such marks only.
struct StreamingAttention : torch::autograd::Function<StreamingAttention> {
  static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k, const Tensor& v,
                        const OptTensor& lens, SymInt context_size, SymInt back_contexts, double sm_scale, bool autotune,
                        bool return_lse, bool prescale_qk, std::string precision, Tensor* lse_out) {
    at::AutoDispatchBelowADInplaceOrView below;
    auto [o, lse] = forward_op().call(q, k, v, lens, context_size, back_contexts, sm_scale, autotune, return_lse,
                                      prescale_qk, precision);
    ctx->save_for_backward({q, k, v, o, lse, lens ? *lens : Tensor()});
    ctx->saved_data["context_size"] = context_size;
    ctx->saved_data["back_contexts"] = back_contexts;
    ctx->saved_data["sm_scale"] = sm_scale;
    ctx->saved_data["flags"] = (int64_t)(autotune ? 1 : 0) | (prescale_qk ? 2 : 0);
    ctx->saved_data["precision"] = std::move(precision);
    ctx->set_materialize_grads(false);   // a missing gradient of O is made in backward, in O's own type and layout
    *lse_out = std::move(lse);
    return o;
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                 torch::autograd::variable_list grads) {
    torch::autograd::variable_list out(12);   // one per argument of forward
    const auto saved = ctx->get_saved_variables();
    const Tensor d_o = grads[0].defined() ? grads[0] : at::zeros_like(saved[3]);
    const int64_t flags = ctx->saved_data["flags"].toInt();
    const std::string precision = ctx->saved_data["precision"].toStringRef();
    auto [dq, dk, dv] = backward_op().call(saved[0], saved[1], saved[2], saved[5].defined() ? OptTensor(saved[5]) : OptTensor(),
                                           saved[3], saved[4], d_o, ctx->saved_data["context_size"].toSymInt(),
                                           ctx->saved_data["back_contexts"].toSymInt(), ctx->saved_data["sm_scale"].toDouble(),
                                           (flags & 1) != 0, (flags & 2) != 0, precision);
    out[0] = std::move(dq), out[1] = std::move(dk), out[2] = std::move(dv);
    return out;
  }
};

bool wants_grad(std::initializer_list<const Tensor*> ts) {
  if (!at::GradMode::is_enabled()) return false;
  for (const Tensor* t : ts)
    if (t->requires_grad()) return true;
  return false;
}

bool has_tangent(std::initializer_list<const Tensor*> ts) {
  for (const Tensor* t : ts)
    if (t->_fw_grad(0).defined()) return true;
  return false;
}

std::tuple<Tensor, Tensor> forward_autograd(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& lens,
                                            SymInt context_size, SymInt back_contexts, double sm_scale, bool autotune,
                                            bool return_lse, bool prescale_qk, c10::string_view precision) {
  // a tangent must not be dropped in silence
  TORCH_CHECK_NOT_IMPLEMENTED(!has_tangent({&q, &k, &v}),
                              "alexdremov_streaming_attention::forward has no forward-mode derivative");
  if (!wants_grad({&q, &k, &v})) {
    at::AutoDispatchBelowADInplaceOrView below;
    return forward_op().call(q, k, v, lens, std::move(context_size), std::move(back_contexts), sm_scale, autotune, return_lse,
                             prescale_qk, precision);
  }
  Tensor lse;
  Tensor o = StreamingAttention::apply(q, k, v, lens, std::move(context_size), std::move(back_contexts), sm_scale, autotune,
                                       return_lse, prescale_qk, std::string(precision), &lse);
  return {std::move(o), std::move(lse)};
}

// Marks the outputs of the backward op as not differentiable a second time: the reference registers no autograd formula
// for ::backward (kernel.py:1360-1442), so differentiating through it raises there, and here.
struct NoDoubleBackward : torch::autograd::Function<NoDoubleBackward> {
  static torch::autograd::variable_list forward(torch::autograd::AutogradContext*, const Tensor& dq, const Tensor& dk,
                                                const Tensor& dv, const Tensor&, const Tensor&, const Tensor&, const Tensor&,
                                                const Tensor&) {
    return {dq.view_as(dq), dk.view_as(dk), dv.view_as(dv)};
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext*, torch::autograd::variable_list) {
    TORCH_CHECK(false, "alexdremov_streaming_attention::backward has no autograd formula: differentiating through the "
                       "backward pass (double backward) is not supported");
  }
};

std::tuple<Tensor, Tensor, Tensor> backward_autograd(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& lens,
                                                     const Tensor& o, const Tensor& lse, const Tensor& d_o, SymInt context_size,
                                                     SymInt back_contexts, double sm_scale, bool autotune, bool prescale_qk,
                                                     c10::string_view precision) {
  // under an ordinary .backward() gradient mode is off and nothing is recorded
  const bool record = wants_grad({&q, &k, &v, &o, &d_o});
  std::tuple<Tensor, Tensor, Tensor> r;
  {
    at::AutoDispatchBelowADInplaceOrView below;
    r = backward_op().call(q, k, v, lens, o, lse, d_o, std::move(context_size), std::move(back_contexts), sm_scale, autotune,
                           prescale_qk, precision);
  }
  if (!record) return r;
  auto g = NoDoubleBackward::apply(std::get<0>(r), std::get<1>(r), std::get<2>(r), q, k, v, o, d_o);
  return {std::move(g[0]), std::move(g[1]), std::move(g[2])};
}

// ---- dense attention: one chunk that covers the whole sequence ----------------------------------------------------
Tensor dense_gpu(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& lens, double sm_scale, bool autotune,
                 bool prescale) {
  if (C10_UNLIKELY(!plain(q, k, v, lens, {}))) {
    PyGILState_STATE gil = PyGILState_Ensure();
    struct Release { PyGILState_STATE s; ~Release() { PyGILState_Release(s); } } release{gil};
    explain("self_attention.kernel", "_validate", {THPVariable_Wrap(q), THPVariable_Wrap(k), THPVariable_Wrap(v), wrap(lens)});
  }
  const Api& a = api();
  Launch l(q, lens);
  Tensor o = empty_same(q);
  if (q.numel() == 0) return o;
  const Tensor qk = kernel_layout(q), kk = kernel_layout(k), vk = kernel_layout(v);
  check(a.forward(ptr(qk), ptr(kk), ptr(vk), l.lens, l.lens_stride, out_ptr(o), nullptr, qk.strides().data(),
                  kk.strides().data(), vk.strides().data(), l.B, l.H, l.T, l.D, l.T, 0, (float)sm_scale, l.dtype, l.stream),
        "sa_forward (self attention)");
  return o;
}
using DenseOp = Tensor(const Tensor&, const Tensor&, const Tensor&, const OptTensor&, double, bool, bool);
const c10::TypedOperatorHandle<DenseOp>& dense_op() {
  static const auto op =
      c10::Dispatcher::singleton().findSchemaOrThrow("alexdremov_flash_attention::forward", "").typed<DenseOp>();
  return op;
}

// Forward only: the result of inputs that require a gradient requires one too, and asking for it raises.
struct DenseAttention : torch::autograd::Function<DenseAttention> {
  static Tensor forward(torch::autograd::AutogradContext*, const Tensor& q, const Tensor& k, const Tensor& v,
                        const OptTensor& lens, double sm_scale, bool autotune, bool prescale) {
    at::AutoDispatchBelowADInplaceOrView below;
    return dense_op().call(q, k, v, lens, sm_scale, autotune, prescale);
  }
  static torch::autograd::variable_list backward(torch::autograd::AutogradContext*, torch::autograd::variable_list) {
    TORCH_CHECK(false, "Trying to backward through alexdremov_flash_attention.forward.default but no autograd formula was "
                       "registered: dense attention is forward only");
  }
};
Tensor dense_autograd(const Tensor& q, const Tensor& k, const Tensor& v, const OptTensor& lens, double sm_scale,
                      bool autotune, bool prescale) {
  if (wants_grad({&q, &k, &v})) return DenseAttention::apply(q, k, v, lens, sm_scale, autotune, prescale);
  at::AutoDispatchBelowADInplaceOrView below;
  return dense_op().call(q, k, v, lens, sm_scale, autotune, prescale);
}

// ---- eager call path of the public functions ------------------------------------------------------------------------
// Arguments come positionally and already complete from the Python functions, which keep their signatures and defaults.
// An argument that is not of the plain type (a flag given as an int, a scale as a tensor, a mistake) returns NotImplemented:
// the Python functions then call the op itself, which converts or refuses it.
bool tensor_args(PyObject* const* args, Tensor (&t)[4], bool& has_lens) {
  has_lens = args[3] != Py_None;
  for (int i = 0; i < (has_lens ? 4 : 3); ++i) {
    if (!THPVariable_Check(args[i])) return false;
    t[i] = THPVariable_Unpack(args[i]);
  }
  return t[0].dim() > 0;
}
bool int_arg(PyObject* x, int64_t& value) {
  int overflow = 0;
  if (!PyLong_CheckExact(x)) return false;
  value = PyLong_AsLongLongAndOverflow(x, &overflow);
  return overflow == 0;
}
bool scale_arg(PyObject* x, const Tensor& q, double& value) {
  if (x != Py_None && !PyFloat_CheckExact(x)) return false;
  value = x == Py_None ? 1.0 / std::sqrt((double)q.size(-1)) : PyFloat_AS_DOUBLE(x);
  return true;
}
bool flag_args(PyObject* const* args, int n) {
  for (int i = 0; i < n; ++i)
    if (!PyBool_Check(args[i])) return false;
  return true;
}

// streaming_attention(q, k, v, lens, context_size, back_contexts, sm_scale or None, autotune, return_lse, prescale_qk, precision)
PyObject* py_streaming_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor t[4];
  bool has_lens;
  int64_t context_size, back_contexts;
  double sm_scale;
  if (n != 11 || !tensor_args(args, t, has_lens) || !int_arg(args[4], context_size) || !int_arg(args[5], back_contexts) ||
      !scale_arg(args[6], t[0], sm_scale) || !flag_args(args + 7, 3) || !PyUnicode_CheckExact(args[10]))
    Py_RETURN_NOTIMPLEMENTED;
  Py_ssize_t len = 0;
  const char* precision = PyUnicode_AsUTF8AndSize(args[10], &len);
  if (!precision) return nullptr;
  const bool autotune = args[7] == Py_True, return_lse = args[8] == Py_True, prescale = args[9] == Py_True;
  // the log-sum-exp is needed by the backward pass whenever a gradient is wanted
  const bool need_lse = return_lse || t[0].requires_grad() || t[1].requires_grad() || t[2].requires_grad();
  std::tuple<Tensor, Tensor> r;
  {
    pybind11::gil_scoped_release no_gil;
    r = forward_op().call(t[0], t[1], t[2], has_lens ? OptTensor(t[3]) : OptTensor(), context_size, back_contexts, sm_scale,
                          autotune, need_lse, prescale, c10::string_view(precision, (size_t)len));
  }
  PyObject* o = THPVariable_Wrap(std::get<0>(r));
  if (!return_lse || !o) return o;
  return Py_BuildValue("(NN)", o, THPVariable_Wrap(std::get<1>(r)));
  END_HANDLE_TH_ERRORS
}

// self_attention(q, k, v, lens, sm_scale or None, autotune, prescale)
PyObject* py_self_attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  Tensor t[4];
  bool has_lens;
  double sm_scale;
  if (n != 7 || !tensor_args(args, t, has_lens) || !scale_arg(args[4], t[0], sm_scale) || !flag_args(args + 5, 2))
    Py_RETURN_NOTIMPLEMENTED;
  const bool autotune = args[5] == Py_True, prescale = args[6] == Py_True;
  Tensor o;
  {
    pybind11::gil_scoped_release no_gil;
    o = dense_op().call(t[0], t[1], t[2], has_lens ? OptTensor(t[3]) : OptTensor(), sm_scale, autotune, prescale);
  }
  return THPVariable_Wrap(o);
  END_HANDLE_TH_ERRORS
}

// kernel_layout(tensor): what the kernels get for it.
PyObject* py_kernel_layout(PyObject*, PyObject* t) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(THPVariable_Check(t), "kernel_layout takes a tensor");
  const Tensor& x = THPVariable_Unpack(t);
  TORCH_CHECK_VALUE(x.dim() == 4, "kernel_layout takes a [B, H, T, D] tensor");
  return THPVariable_Wrap(kernel_layout(x));
  END_HANDLE_TH_ERRORS
}

// Whether the environment routes calls through the compiled wrapper (read on every call: it may change at run time).
PyObject* py_env_asks_for_wrapper(PyObject*, PyObject*) {
  const char* compiled = getenv("STREAMING_ATTENTION_COMPILED");
  const char* eager = getenv("STREAMING_ATTENTION_EAGER");
  return PyBool_FromLong((compiled && std::string_view(compiled) == "1") || (eager && std::string_view(eager) == "0"));
}

PyMethodDef methods[] = {
    {"kernel_layout", py_kernel_layout, METH_O, nullptr},
    {"env_asks_for_wrapper", py_env_asks_for_wrapper, METH_NOARGS, nullptr},
    {"streaming_attention", (PyCFunction)(void (*)())py_streaming_attention, METH_FASTCALL, nullptr},
    {"self_attention", (PyCFunction)(void (*)())py_self_attention, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// The schemas are those that the reference's torch.library.custom_op decorators infer (kernel.py:1270-1284, 1360-1376;
// src/self_attention/kernel.py:359-371), with the pt2-compliance tag that the decorator sets.
TORCH_LIBRARY(alexdremov_streaming_attention, m) {
  m.def("forward(Tensor q, Tensor k, Tensor v, Tensor? lens, SymInt context_size, SymInt back_contexts, "
        "float sm_scale, bool autotune, bool return_lse, bool prescale_qk, str precision) -> (Tensor, Tensor)",
        {at::Tag::pt2_compliant_tag});
  m.def("backward(Tensor q, Tensor k, Tensor v, Tensor? lens, Tensor o, Tensor lse, Tensor do, "
        "SymInt context_size, SymInt back_contexts, float sm_scale, bool autotune, bool prescale_qk, "
        "str precision) -> (Tensor, Tensor, Tensor)",
        {at::Tag::pt2_compliant_tag});
}
TORCH_LIBRARY_IMPL(alexdremov_streaming_attention, CUDA, m) {
  m.impl("forward", TORCH_FN(forward_gpu));
  m.impl("backward", TORCH_FN(backward_gpu));
}
TORCH_LIBRARY_IMPL(alexdremov_streaming_attention, Autograd, m) {
  m.impl("forward", TORCH_FN(forward_autograd));
  m.impl("backward", TORCH_FN(backward_autograd));
}
TORCH_LIBRARY(alexdremov_flash_attention, m) {
  m.def("forward(Tensor q, Tensor k, Tensor v, Tensor? lens, float sm_scale, bool autotune, bool prescale) -> Tensor",
        {at::Tag::pt2_compliant_tag});
}
TORCH_LIBRARY_IMPL(alexdremov_flash_attention, CUDA, m) { m.impl("forward", TORCH_FN(dense_gpu)); }
TORCH_LIBRARY_IMPL(alexdremov_flash_attention, Autograd, m) {
  m.impl("forward", TORCH_FN(dense_autograd));
}

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
