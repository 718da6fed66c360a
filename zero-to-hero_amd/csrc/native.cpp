// Native host path of ppo_amd: the extension module ppo_amd._native.
//
// ops.py's entry points spend 20-100 us of Python per call on checking tensors,
// allocating outputs, filling ctypes arguments and walking nn.Modules, several
// times their kernels' time at the sizes of a minibatch or an environment
// step.  Each function here does the same for the ordinary call -- plain
// contiguous fp32 tensors of matching shapes on one GPU, no output arguments
// beyond those named -- and returns None for any other, which ops.py then takes
// through its own checks (and errors) as before.  The losses' autograd node is
// here as well, so a backward pass runs without the interpreter.
//
// Measured on MI355X, us a call among others, through Python and here:
// gae_normalize T x N = 128 x 8 25.3 and 16.5; the categorical loss with its
// backward, B = 100,003, A = 4, 94 and 52; the Gaussian one, B = 2,097,152, D = 6,
// 102 and 56; action selection for 4096 environments 42.4 and 7.5.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/SavedTensorHooks.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Generator.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/graph_task.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/utils/pybind.h>

#include "ppo_amd.h"
#include "scale.hpp"

namespace {

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// What init() hands over: the workspace pool, the LossStats class, the function
// that raises for a library error code, and torch.nn's classes.
struct Python {
  PyObject* pool = nullptr;
  PyObject* stats = nullptr;
  PyObject* fail = nullptr;
  PyObject *sequential = nullptr, *linear = nullptr, *relu = nullptr, *tanh = nullptr;
  PyObject* scalar_names[PPO_NUM_SCALARS] = {};
  PyObject *get = nullptr, *modules = nullptr, *parameters = nullptr, *net = nullptr,
           *weight = nullptr, *bias = nullptr, *in_features = nullptr, *out_features = nullptr;
} P;

// Thrown for a call that is not the ordinary one (entry clears a Python error that
// a look at its arguments has set).
struct NotPlain {};

void need(bool ok) {
  if (!ok) throw NotPlain{};
}

// Modes, transforms and traces that want to see torch operators or autograd
// functions: not for this path.
bool plain_mode() {
  return !torch::jit::tracer::isTracing() && !at::impl::torch_function_mode_enabled() &&
         !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         !c10::impl::tls_is_dispatch_key_included(
             c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

void need_plain_mode() { need(plain_mode()); }

// Keys of tensors that stand for another tensor, or for none: no storage of
// their own to read.
constexpr c10::DispatchKeySet kWrapped({c10::DispatchKey::Python, c10::DispatchKey::Batched,
                                        c10::DispatchKey::FuncTorchBatched,
                                        c10::DispatchKey::FuncTorchGradWrapper,
                                        c10::DispatchKey::Functionalize,
                                        c10::DispatchKey::Negative, c10::DispatchKey::Conjugate,
                                        c10::DispatchKey::ZeroTensor});

// A torch.Tensor (or Parameter) itself: no subclass, no wrapper, dense GPU
// storage, contiguous.
const Tensor& plain(PyObject* o, at::ScalarType type) {
  need(THPVariable_CheckExact(o));
  const Tensor& t = THPVariable_Unpack(o);
  need(t.defined() && t.is_cuda() && t.layout() == at::kStrided &&
       !t.key_set().has_any(kWrapped) && t.scalar_type() == type && t.is_contiguous());
  return t;
}

const Tensor& plain(PyObject* o, at::ScalarType type, const at::Device& device) {
  const Tensor& t = plain(o, type);
  need(t.device() == device);
  return t;
}

const Tensor& plain_rows(PyObject* o, const at::Device& device, int64_t n) {
  const Tensor& t = plain(o, at::kFloat, device);
  need(t.dim() == 1 && t.size(0) == n);
  return t;
}

double number(PyObject* o) {
  need(PyFloat_CheckExact(o) || PyLong_CheckExact(o));
  const double x = PyFloat_AsDouble(o);
  need(x != -1.0 || !PyErr_Occurred());
  return x;
}

int64_t integer(PyObject* o) {
  const int64_t x = PyLong_AsLongLong(o);
  need(x != -1 || !PyErr_Occurred());
  return x;
}

const float* in(const Tensor& t) { return t.const_data_ptr<float>(); }
float* out(const Tensor& t) { return t.data_ptr<float>(); }

void* current_stream(const at::Device& device) {
  return c10::hip::getCurrentHIPStream(device.index()).stream();
}

// The pool's buffer for (device, stream): ops._WorkspacePool.get.
Tensor workspace(const at::Device& device, void* stream, size_t nbytes) {
  py::object dev = py::reinterpret_steal<py::object>(THPDevice_New(device));
  py::int_ s(reinterpret_cast<uintptr_t>(stream)), n(nbytes);
  PyObject* args[] = {P.pool, dev.ptr(), s.ptr(), n.ptr()};
  PyObject* r = PyObject_VectorcallMethod(P.get, args, 4, nullptr);
  if (!r) throw py::error_already_set();
  py::object buf = py::reinterpret_steal<py::object>(r);
  return THPVariable_Unpack(r);
}

// Allocations and the library call, outside the GIL: other Python threads run
// while this one waits for memory or for room in a full hardware queue.
template <typename F>
int unlocked(F f) {
  py::gil_scoped_release no_gil;
  return f();
}

// Raises PPOLibraryError (ops._native_failed) for a non-zero status.
void check(const char* name, int code, const at::Device& device, void* stream) {
  if (code == PPO_OK) return;
  py::object dev = py::reinterpret_steal<py::object>(THPDevice_New(device));
  py::reinterpret_borrow<py::object>(P.fail)(name, code, dev,
                                             reinterpret_cast<uintptr_t>(stream));
}

// Element i of a 1-D fp32 tensor as a 0-d tensor on the same storage (no
// autograd view).
Tensor element(const Tensor& t, int64_t i) {
  auto impl = c10::make_intrusive<c10::TensorImpl>(c10::Storage(t.storage()), t.key_set(),
                                                   t.dtype());
  impl->set_sizes_contiguous(at::IntArrayRef{});
  impl->set_storage_offset(t.storage_offset() + i);
  return Tensor(std::move(impl));
}

PyObject* wrap(const Tensor& t) {
  PyObject* o = THPVariable_Wrap(t);
  if (!o) throw py::error_already_set();
  return o;
}

PyObject* tuple_of(std::initializer_list<Tensor> ts) {
  py::tuple r(ts.size());
  size_t k = 0;
  for (const Tensor& t : ts) PyTuple_SET_ITEM(r.ptr(), k++, wrap(t));
  return r.release().ptr();
}

// LossStats of a [6] tensor.
py::object loss_stats(const Tensor& scalars) {
  py::object d = py::reinterpret_steal<py::object>(PyObject_CallNoArgs(P.stats));
  if (!d) throw py::error_already_set();
  for (int i = 0; i < PPO_NUM_SCALARS; ++i) {
    py::object v = py::reinterpret_steal<py::object>(wrap(element(scalars, i)));
    if (PyDict_SetItem(d.ptr(), P.scalar_names[i], v.ptr())) throw py::error_already_set();
  }
  return d;
}

// --- GAE ---------------------------------------------------------------------------

struct Rollout {
  const Tensor *r, *v, *d, *lv = nullptr;
  int64_t T, N;
  double gamma, lam;
  Tensor ws;
  void* stream;

  Rollout(PyObject* const* a) {  // rewards, values, dones, last_value, gamma, lam
    r = &plain(a[0], at::kFloat);
    const at::Device dev = r->device();
    v = &plain(a[1], at::kFloat, dev);
    need(THPVariable_CheckExact(a[2]));
    const at::ScalarType dt = THPVariable_Unpack(a[2]).scalar_type();
    need(dt == at::kByte || dt == at::kBool);
    d = &plain(a[2], dt, dev);
    need((r->dim() == 1 || r->dim() == 2) && v->sizes() == r->sizes() && d->sizes() == r->sizes());
    T = r->size(0);
    N = r->dim() == 2 ? r->size(1) : 1;
    need(T > 0 && N > 0);
    if (a[3] != Py_None) {
      lv = &plain(a[3], at::kFloat, dev);
      need(lv->numel() == N);
    }
    gamma = number(a[4]);
    lam = number(a[5]);
    stream = current_stream(dev);
    ws = workspace(dev, stream, ppo_gae_workspace_bytes(T, N));
  }
  const uint8_t* dones() const { return static_cast<const uint8_t*>(d->const_data_ptr()); }
  const float* last() const { return lv ? in(*lv) : nullptr; }
};

PyObject* gae(PyObject* const* a) {
  const Rollout x(a);
  Tensor adv, ret;
  const int code = unlocked([&] {
    adv = at::empty(x.r->sizes(), x.r->options());
    ret = at::empty_like(adv);
    return ppo_gae_f32(in(*x.r), in(*x.v), x.dones(), x.last(), x.T, x.N, x.gamma, x.lam,
                       out(adv), out(ret), x.ws.data_ptr(), x.ws.numel(), x.stream);
  });
  check("ppo_gae_f32", code, x.r->device(), x.stream);
  return tuple_of({adv, ret});
}

PyObject* gae_normalize(PyObject* const* a) {  // ..., eps
  const Rollout x(a);
  const double eps = number(a[6]);
  Tensor adv, ret, adv_n, stats;
  const int code = unlocked([&] {
    adv = at::empty(x.r->sizes(), x.r->options());
    ret = at::empty_like(adv);
    adv_n = at::empty_like(adv);
    stats = at::empty({2}, x.r->options());
    return ppo_gae_norm_f32(in(*x.r), in(*x.v), x.dones(), x.last(), x.T, x.N, x.gamma, x.lam,
                            eps, out(adv), out(ret), out(adv_n), out(stats), x.ws.data_ptr(),
                            x.ws.numel(), x.stream);
  });
  check("ppo_gae_norm_f32", code, x.r->device(), x.stream);
  return tuple_of({adv, ret, adv_n, stats});
}

// --- losses --------------------------------------------------------------------------

ppo_loss_params loss_params(PyObject* clip, PyObject* vf, PyObject* value_coef,
                            PyObject* entropy_coef) {
  ppo_loss_params p = {number(clip), vf == Py_None ? 0.0 : number(vf), number(value_coef),
                       number(entropy_coef)};
  need(p.clip_ratio >= 0.0 && (vf == Py_None || p.vf_clip > 0.0));
  return p;
}

// The launch's results: scalars [6] and the gradients of the differentiable
// inputs, in their order.
struct Loss {
  variable_list inputs, grads;
  Tensor scalars;
};

// old_log_probs, advantages, returns, values, old_values (or None), clip_ratio,
// vf_clip, value_coef, entropy_coef from a[0]
struct Rows {
  const Tensor *old_lp, *adv, *ret, *val, *old_val = nullptr;
  ppo_loss_params p;

  Rows(PyObject* const* a, const at::Device& dev, int64_t B) {
    old_lp = &plain_rows(a[0], dev, B);
    adv = &plain_rows(a[1], dev, B);
    ret = &plain_rows(a[2], dev, B);
    val = &plain_rows(a[3], dev, B);
    if (a[4] != Py_None) old_val = &plain_rows(a[4], dev, B);
    need(old_val || a[6] == Py_None);
    p = loss_params(a[5], a[6], a[7], a[8]);
  }
  const float* old_values() const { return old_val ? in(*old_val) : nullptr; }
};

Loss loss_discrete_launch(PyObject* const* a) {  // logits, actions, rows...
  const Tensor& z = plain(a[0], at::kFloat);
  const at::Device dev = z.device();
  need(z.dim() == 2 && z.size(0) > 0 && z.size(1) > 0 && z.size(1) <= INT32_MAX);
  const int64_t B = z.size(0);
  const int32_t A = (int32_t)z.size(1);
  need(THPVariable_CheckExact(a[1]));
  const at::ScalarType at_ = THPVariable_Unpack(a[1]).scalar_type();
  need(at_ == at::kInt || at_ == at::kLong);
  const Tensor& act = plain(a[1], at_, dev);
  need(act.dim() == 1 && act.size(0) == B);
  const Rows r(a + 2, dev, B);
  void* stream = current_stream(dev);
  const Tensor ws = workspace(dev, stream, ppo_loss_cat_workspace_bytes(B, A));
  at::AutoDispatchBelowADInplaceOrView below;
  Loss l;
  const int code = unlocked([&] {
    const Tensor dz = at::empty({B, A}, z.options()), dv = at::empty({B}, z.options());
    l.scalars = at::empty({PPO_NUM_SCALARS}, z.options());
    l.grads = {dz, dv};
    return ppo_loss_cat_f32(in(z), B, A, act.const_data_ptr(), at_ == at::kLong, in(*r.old_lp),
                            in(*r.adv), in(*r.ret), in(*r.val), r.old_values(), &r.p, out(dz),
                            out(dv), out(l.scalars), ws.data_ptr(), ws.numel(), stream);
  });
  check("ppo_loss_cat_f32", code, dev, stream);
  l.inputs = {z, *r.val};
  return l;
}

Loss loss_gaussian_launch(PyObject* const* a) {  // mu, log_std, actions, rows...
  const Tensor& mu = plain(a[0], at::kFloat);
  const at::Device dev = mu.device();
  need(mu.dim() == 2 && mu.size(0) > 0 && mu.size(1) > 0 && mu.size(1) <= 24);
  const int64_t B = mu.size(0);
  const int32_t D = (int32_t)mu.size(1);
  const Tensor& ls = plain_rows(a[1], dev, D);
  const Tensor& act = plain(a[2], at::kFloat, dev);
  need(act.sizes() == mu.sizes());
  const Rows r(a + 3, dev, B);
  void* stream = current_stream(dev);
  const Tensor ws = workspace(dev, stream, ppo_loss_gauss_workspace_bytes(B, D));
  at::AutoDispatchBelowADInplaceOrView below;
  Loss l;
  const int code = unlocked([&] {
    const Tensor dmu = at::empty({B, D}, mu.options()), dls = at::empty({D}, mu.options()),
                 dv = at::empty({B}, mu.options());
    l.scalars = at::empty({PPO_NUM_SCALARS}, mu.options());
    l.grads = {dmu, dls, dv};
    return ppo_loss_gauss_f32(in(mu), in(ls), B, D, in(act), in(*r.old_lp), in(*r.adv),
                              in(*r.ret), in(*r.val), r.old_values(), &r.p, out(dmu), out(dls),
                              out(dv), out(l.scalars), ws.data_ptr(), ws.numel(), stream);
  });
  check("ppo_loss_gauss_f32", code, dev, stream);
  l.inputs = {mu, ls, *r.val};
  return l;
}

// A tensor that the scale kernel can read: dense fp32 with storage of its own on
// `device`.
bool plain_f32(const Tensor& t, const at::Device& device) {
  return t.is_cuda() && t.layout() == at::kStrided && !t.key_set().has_any(kWrapped) &&
         t.scalar_type() == at::kFloat && t.is_contiguous() && t.device() == device;
}

// Whether the scale kernel may multiply `grads` by `scale`.  Batched gradients
// (is_grads_batched), fake tensors and dispatch modes see torch's products
// instead, and so do saved tensors that a hook replaced by views, other types or
// other devices' tensors.
bool plain_scale(const variable_list& grads, const Tensor& scale) {
  if (!plain_mode() || scale.numel() != 1 || !plain_f32(scale, scale.device())) return false;
  for (const Tensor& t : grads)
    if (!plain_f32(t, scale.device())) return false;
  return true;
}

// grads[k] * scale in one launch, into the tensors themselves (`own`) or new ones.
// A captured launch always writes new ones: the graph may be replayed more often
// than the forward that fills the saved ones.
variable_list scaled(const variable_list& grads, const Tensor& scale, bool own) {
  own = own && c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None;
  variable_list dst = grads;
  ppo::ScaleArray a[ppo::kMaxScaleArrays];
  for (size_t k = 0; k < grads.size(); ++k) {
    if (!own) dst[k] = at::empty_like(grads[k]);
    a[k] = {in(grads[k]), out(dst[k]), dst[k].numel()};
  }
  const int code =
      ppo::launch_scale(a, (int)grads.size(), in(scale), current_stream(scale.device()));
  TORCH_CHECK(code == PPO_OK, "scaling the loss gradients failed with code ", code);
  return dst;
}

// The losses' node: saved gradients times the loss's incoming gradient (the
// rules of ops._scaled_grads).
struct LossNode : public torch::autograd::Function<LossNode> {
  static Tensor forward(AutogradContext* ctx, at::TensorList, const Loss* l) {
    ctx->save_for_backward(l->grads);
    ctx->set_materialize_grads(false);
    // (saved-tensor hooks hand backward whatever they like)
    ctx->saved_data["hooked"] = at::SavedTensorDefaultHooks::get_hooks().has_value();
    // a 0-d tensor on the scalars' storage: an indexed view's backward would
    // build and fill a [6] gradient
    return element(l->scalars, PPO_SCALAR_LOSS);
  }

  static variable_list backward(AutogradContext* ctx, variable_list g) {
    variable_list grads = ctx->get_saved_variables();
    const size_t n = grads.size();
    if (!g[0].defined()) return variable_list(n + 1);
    const Tensor& scale = g[0];
    if (at::GradMode::is_enabled() || ctx->saved_data["hooked"].toBool() ||
        !plain_scale(grads, scale)) {
      for (Tensor& t : grads) t = t * scale;
    } else {
      // sole owners: the saved variable and `grads`
      bool own = !torch::autograd::get_current_graph_task_keep_graph();
      for (const Tensor& t : grads) own = own && t.use_count() == 2;
      grads = scaled(grads, scale, own);
    }
    grads.resize(n + 1);  // (the launch's results are no differentiable input)
    return grads;
  }
};

PyObject* with_autograd(const Loss& l) {
  const Tensor loss = LossNode::apply(at::TensorList(l.inputs), &l);
  py::object stats = loss_stats(l.scalars);
  py::tuple r(2);
  PyTuple_SET_ITEM(r.ptr(), 0, wrap(loss));
  PyTuple_SET_ITEM(r.ptr(), 1, stats.release().ptr());
  return r.release().ptr();
}

// Forward-mode tangents are for ops' autograd functions (to refuse), before
// anything is launched.
void need_no_tangent(PyObject* o) {
  need(THPVariable_CheckExact(o) && !THPVariable_Unpack(o)._fw_grad(0).defined());
}

PyObject* loss_discrete(PyObject* const* a) {  // logits, actions, rows...
  need_no_tangent(a[0]);
  need_no_tangent(a[5]);
  return with_autograd(loss_discrete_launch(a));
}

PyObject* loss_gaussian(PyObject* const* a) {  // mu, log_std, actions, rows...
  for (int k : {0, 1, 6}) need_no_tangent(a[k]);
  return with_autograd(loss_gaussian_launch(a));
}

PyObject* loss_discrete_fused(PyObject* const* a) {
  const Loss l = loss_discrete_launch(a);
  return tuple_of({l.scalars, l.grads[0], l.grads[1]});
}
PyObject* loss_gaussian_fused(PyObject* const* a) {
  const Loss l = loss_gaussian_launch(a);
  return tuple_of({l.scalars, l.grads[0], l.grads[1], l.grads[2]});
}

// --- MLPs ----------------------------------------------------------------------------

PyObject* item(PyObject* dict, PyObject* key) {
  PyObject* v = dict ? PyDict_GetItemWithError(dict, key) : nullptr;
  need(v != nullptr);
  return v;
}

PyObject* instance_dict(PyObject* o) {
  PyObject** d = _PyObject_GetDictPtr(o);
  need(d && *d && PyDict_CheckExact(*d));
  return *d;
}

// The network of ops.mlp_structure: `module.net` (or the module itself), a
// Sequential of Linear-act-Linear-act-Linear.
struct Net {
  const Tensor *w[3], *b[3];
  int64_t D, H, O;
  bool tanh;

  explicit Net(PyObject* module) {
    PyObject* seq = module;
    PyObject* mods = item(instance_dict(module), P.modules);
    need(PyDict_CheckExact(mods));
    if (Py_TYPE(module) != (PyTypeObject*)P.sequential) {
      // (a class attribute of that name would hide the submodule)
      need(_PyType_Lookup(Py_TYPE(module), P.net) == nullptr &&
           PyDict_GetItemWithError(instance_dict(module), P.net) == nullptr);
      seq = item(mods, P.net);
      need(Py_TYPE(seq) == (PyTypeObject*)P.sequential);
      mods = item(instance_dict(seq), P.modules);
      need(PyDict_CheckExact(mods));
    } else {
      need(PyDict_GetItemWithError(mods, P.net) == nullptr);
    }
    need(PyDict_Size(mods) == 5);
    PyObject *key, *m[5];
    Py_ssize_t pos = 0;
    for (int k = 0; k < 5; ++k) need(PyDict_Next(mods, &pos, &key, &m[k]) != 0);
    tanh = Py_TYPE(m[1]) == (PyTypeObject*)P.tanh;
    for (int k = 1; k < 5; k += 2)
      need(Py_TYPE(m[k]) == (PyTypeObject*)(tanh ? P.tanh : P.relu));
    int64_t dim[4];
    for (int l = 0; l < 3; ++l) {
      PyObject* lin = m[2 * l];
      need(Py_TYPE(lin) == (PyTypeObject*)P.linear);
      PyObject* d = instance_dict(lin);
      PyObject* params = item(d, P.parameters);
      need(PyDict_CheckExact(params) && PyDict_GetItemWithError(d, P.weight) == nullptr &&
           PyDict_GetItemWithError(d, P.bias) == nullptr);
      w[l] = &plain(item(params, P.weight), at::kFloat);
      b[l] = &plain(item(params, P.bias), at::kFloat);
      const int64_t i = integer(item(d, P.in_features)), o = integer(item(d, P.out_features));
      need(w[l]->dim() == 2 && w[l]->size(0) == o && w[l]->size(1) == i && b[l]->dim() == 1 &&
           b[l]->size(0) == o && (l == 0 || dim[l] == i) && b[l]->device() == w[0]->device() &&
           w[l]->device() == w[0]->device());
      dim[l] = i;
      dim[l + 1] = o;
    }
    D = dim[0];
    H = dim[1];
    need(dim[2] == H);
    O = dim[3];
  }

  // with_grads: every parameter has a gradient buffer to write
  ppo_mlp3_f32 pointers(bool with_grads) const {
    ppo_mlp3_f32 s = {};
    for (int l = 0; l < 3; ++l) {
      s.weight[l] = in(*w[l]);
      s.bias[l] = in(*b[l]);
      if (!with_grads) continue;
      s.weight_grad[l] = grad(*w[l]);
      s.bias_grad[l] = grad(*b[l]);
    }
    return s;
  }

  static float* grad(const Tensor& p) {
    const Tensor& g = p.grad();
    need(g.defined() && g.scalar_type() == at::kFloat && g.is_contiguous() &&
         g.sizes() == p.sizes() && g.device() == p.device() && g.layout() == at::kStrided);
    return out(g);
  }
};

// Both networks of one actor-critic pair (ops.mlp_fusable).
struct Pair {
  Net actor, critic;
  Pair(PyObject* policy, PyObject* value) : actor(policy), critic(value) {
    const int64_t H = actor.H;
    need(actor.tanh == critic.tanh && critic.D == actor.D && critic.H == H && critic.O == 1 &&
         (H == 16 || H == 32 || H == 64 || H == 128) && actor.D <= 64 && actor.O <= 32 &&
         critic.w[0]->device() == actor.w[0]->device());
  }
  int activation() const { return actor.tanh ? PPO_ACT_TANH : PPO_ACT_RELU; }
};

// An output argument (None: undefined, for new_if_none).
Tensor given(PyObject* o, at::IntArrayRef sizes, at::ScalarType type, const at::Device& dev) {
  if (o == Py_None) return {};
  const Tensor& t = plain(o, type, dev);
  need(t.sizes() == sizes);
  return t;
}

void new_if_none(Tensor& t, at::IntArrayRef sizes, at::ScalarType type, const at::Device& dev) {
  if (!t.defined()) t = at::empty(sizes, at::TensorOptions().dtype(type).device(dev));
}

// policy, value, observations, uniforms, generator, observations_out,
// actions_out, log_probs_out, values_out
PyObject* mlp_act(PyObject* const* a) {
  const Pair nets(a[0], a[1]);
  const at::Device dev = nets.actor.w[0]->device();
  const Tensor& obs = plain(a[2], at::kFloat, dev);
  need(obs.dim() == 2 && obs.size(1) == nets.actor.D);
  const int64_t N = obs.size(0);
  float* obs_out = nullptr;
  if (a[5] != Py_None) {
    const Tensor& t = plain(a[5], at::kFloat, dev);
    need(t.numel() == obs.numel());
    obs_out = out(t);
  }
  at::AutoDispatchBelowADInplaceOrView below;
  Tensor act = given(a[6], {N}, at::kInt, dev), lp = given(a[7], {N}, at::kFloat, dev),
         val = given(a[8], {N}, at::kFloat, dev), u;
  std::optional<at::Generator> gen;
  if (a[3] != Py_None) {
    u = plain_rows(a[3], dev, N);
  } else if (a[4] != Py_None) {
    need(THPGenerator_Check(a[4]));
    gen = THPGenerator_Unwrap(a[4]);
  }
  const ppo_mlp3_f32 pa = nets.actor.pointers(false), pc = nets.critic.pointers(false);
  void* stream = current_stream(dev);
  const int code = unlocked([&] {
    new_if_none(act, {N}, at::kInt, dev);
    new_if_none(lp, {N}, at::kFloat, dev);
    new_if_none(val, {N}, at::kFloat, dev);
    if (!u.defined()) u = at::rand({N}, gen, obs.options());
    return ppo_mlp_act_cat_f32(&pa, &pc, (int32_t)nets.actor.D, (int32_t)nets.actor.H,
                               (int32_t)nets.actor.O, nets.activation(), in(obs), N, in(u),
                               obs_out, act.data_ptr<int32_t>(), out(lp), out(val), stream);
  });
  check("ppo_mlp_act_cat_f32", code, dev, stream);
  py::tuple r(3);
  const Tensor* ts[] = {&act, &lp, &val};
  for (int k = 0; k < 3; ++k) {
    PyObject* given = a[6 + k];
    PyTuple_SET_ITEM(r.ptr(), k, given != Py_None ? Py_NewRef(given) : wrap(*ts[k]));
  }
  return r.release().ptr();
}

// policy, value, observations, actions, old_log_probs, advantages, returns,
// old_values, index, clip_ratio, vf_clip, value_coef, entropy_coef, scalars_out
PyObject* mlp_grads(PyObject* const* a) {
  const Pair nets(a[0], a[1]);
  const at::Device dev = nets.actor.w[0]->device();
  const Tensor& obs = plain(a[2], at::kFloat, dev);
  need(obs.dim() == 2 && obs.size(1) == nets.actor.D);
  const int64_t n = obs.size(0);
  need(THPVariable_CheckExact(a[3]));
  const at::ScalarType type = THPVariable_Unpack(a[3]).scalar_type();
  need(type == at::kInt || type == at::kLong);
  const Tensor& act = plain(a[3], type, dev);
  need(act.dim() == 1 && act.size(0) == n);
  const Tensor &old_lp = plain_rows(a[4], dev, n), &adv = plain_rows(a[5], dev, n),
               &ret = plain_rows(a[6], dev, n);
  const ppo_loss_params p = loss_params(a[9], a[10], a[11], a[12]);
  const float* old_val = a[10] == Py_None ? nullptr : in(plain_rows(a[7], dev, n));
  const int64_t* idx = nullptr;
  int64_t B = n;
  if (a[8] != Py_None) {
    const Tensor& t = plain(a[8], at::kLong, dev);
    need(t.dim() == 1);
    B = t.size(0);
    idx = t.const_data_ptr<int64_t>();
  }
  need(B > 0);
  const ppo_mlp3_f32 pa = nets.actor.pointers(true), pc = nets.critic.pointers(true);
  at::AutoDispatchBelowADInplaceOrView below;
  Tensor scalars = given(a[13], {PPO_NUM_SCALARS}, at::kFloat, dev);
  const int32_t D = (int32_t)nets.actor.D, H = (int32_t)nets.actor.H, A = (int32_t)nets.actor.O;
  void* stream = current_stream(dev);
  const Tensor ws = workspace(dev, stream, ppo_mlp_cat_grad_workspace_bytes(B, D, H, A));
  const int code = unlocked([&] {
    new_if_none(scalars, {PPO_NUM_SCALARS}, at::kFloat, dev);
    return ppo_mlp_cat_grad_f32(&pa, &pc, D, H, A, nets.activation(), in(obs), n, idx, B,
                                act.const_data_ptr(), type == at::kLong, in(old_lp), in(adv),
                                in(ret), old_val, &p, out(scalars), ws.data_ptr(), ws.numel(),
                                stream);
  });
  check("ppo_mlp_cat_grad_f32", code, dev, stream);
  return loss_stats(scalars).release().ptr();
}

// --- module ----------------------------------------------------------------------------

template <PyObject* (*kFn)(PyObject* const*), int kArgs>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != kArgs) {
    PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
    return nullptr;
  }
  try {
    need(P.pool != nullptr);
    need_plain_mode();
    return kFn(args);
  } catch (const NotPlain&) {
    PyErr_Clear();
    Py_RETURN_NONE;
  } catch (py::error_already_set& e) {
    e.restore();
    return nullptr;
  } catch (const std::exception&) {
    torch::translate_exception_to_python(std::current_exception());
    return nullptr;
  }
}

#define PPO_ENTRY(name, fn, nargs) \
  {name, (PyCFunction)(void (*)(void))(&entry<fn, nargs>), METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    PPO_ENTRY("gae", gae, 6),
    PPO_ENTRY("gae_normalize", gae_normalize, 7),
    PPO_ENTRY("loss_discrete", loss_discrete, 11),
    PPO_ENTRY("loss_discrete_fused", loss_discrete_fused, 11),
    PPO_ENTRY("loss_gaussian", loss_gaussian, 12),
    PPO_ENTRY("loss_gaussian_fused", loss_gaussian_fused, 12),
    PPO_ENTRY("mlp_act", mlp_act, 9),
    PPO_ENTRY("mlp_grads", mlp_grads, 14),
    {nullptr, nullptr, 0, nullptr}};
#undef PPO_ENTRY

// The reference counts of a tensor with one owner in C++ (as a saved variable is)
// and one reference to its Python object (as the tuple of saved tensors holds),
// which depend on whether the tensor itself keeps its Python object alive.
struct SoleOwners {
  Py_ssize_t object;
  size_t tensor;
  SoleOwners() {
    const Tensor t = at::empty({0}, at::kCPU);
    const py::object o = py::reinterpret_steal<py::object>(wrap(t));
    object = Py_REFCNT(o.ptr());
    tensor = t.use_count();
  }
};

// ops._scaled_grads: every tensor of the tuple that ctx.saved_tensors gave times
// `scale`, in one launch, or None for tensors that torch's products have to take.
// In place where the graph is released and nobody else holds them (SoleOwners).
py::object scale_grads(const py::tuple& saved, const Tensor& scale) {
  TORCH_CHECK(saved.size() > 0 && saved.size() <= ppo::kMaxScaleArrays, "scale_grads takes 1 to ",
              ppo::kMaxScaleArrays, " tensors");
  static const SoleOwners sole;
  bool own = !torch::autograd::get_current_graph_task_keep_graph();
  variable_list grads;
  for (size_t k = 0; k < saved.size(); ++k) {
    PyObject* o = PyTuple_GET_ITEM(saved.ptr(), k);
    if (!THPVariable_CheckExact(o)) return py::none();
    const Tensor& t = THPVariable_Unpack(o);
    own = own && Py_REFCNT(o) == sole.object && t.use_count() == sole.tensor;
    grads.push_back(t);
  }
  if (!plain_scale(grads, scale)) return py::none();
  {
    py::gil_scoped_release no_gil;
    grads = scaled(grads, scale, own);
  }
  return py::cast(grads);
}

void init(py::object pool, py::object stats, py::object fail, const std::vector<std::string>& names,
          py::object sequential, py::object linear, py::object relu, py::object tanh) {
  TORCH_CHECK(names.size() == PPO_NUM_SCALARS, "expected ", PPO_NUM_SCALARS, " scalar names");
  for (int i = 0; i < PPO_NUM_SCALARS; ++i)
    P.scalar_names[i] = PyUnicode_InternFromString(names[i].c_str());
  P.get = PyUnicode_InternFromString("get");
  P.modules = PyUnicode_InternFromString("_modules");
  P.parameters = PyUnicode_InternFromString("_parameters");
  P.net = PyUnicode_InternFromString("net");
  P.weight = PyUnicode_InternFromString("weight");
  P.bias = PyUnicode_InternFromString("bias");
  P.in_features = PyUnicode_InternFromString("in_features");
  P.out_features = PyUnicode_InternFromString("out_features");
  P.stats = stats.release().ptr();
  P.fail = fail.release().ptr();
  P.sequential = sequential.release().ptr();
  P.linear = linear.release().ptr();
  P.relu = relu.release().ptr();
  P.tanh = tanh.release().ptr();
  P.pool = pool.release().ptr();
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  m.def("init", &init);
  m.def("scale_grads", &scale_grads);
  if (PyModule_AddFunctions(m.ptr(), kMethods)) throw py::error_already_set();
}
