// The bundled operators for torch tensors on a GPU, without Python between the call
// and the launcher: `mobula.op.ROIAlign(...)` and `mobula.op.Conv2D(...)` hand their
// arguments here (glue/torch_glue.py: _offer_direct_call), forward runs at once, backward is
// a node of torch's graph that runs on the engine's thread without the interpreter.
//
// What it saves: a forward + backward of eight boxes keeps the GPU busy for 24 us (four kernels), and
// took 140-270 us (by the host) through the operator classes: two rounds of argument
// inspection, type resolution and marshalling of thirteen values each, a module object
// per call, and the interpreter lock handed to the engine's thread and back.
//
// A call this file does not take (other tensor types, arguments it cannot read, shapes
// the operator class would refuse, calls under a transform of torch's or with hooks on all
// modules) is answered with NotImplemented, and the operator class takes it as before: what is
// an error stays the error it was.
//
// Semantics are those of opzoo/ROIAlign/ROIAlign.py and opzoo/Convolution/Convolution.py
// under the torch glue: fresh outputs and gradients, boxes get zeros, channels-last maps
// keep their format, other strided tensors go through dense copies.  Gradients nobody
// asked for are not computed.
#define PY_SSIZE_T_CLEAN   // (before Python.h)
#include <Python.h>

#include <climits>
#include <stdexcept>
#include <string>
#include <vector>

#include <ATen/ATen.h>
#include <ATen/TracerMode.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/variable.h>

#include "mobula_roialign.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::variable_list;

// Stream and element counts of the next call of this thread (see mobula_roialign.h).
void begin(const Tensor& on, std::initializer_list<long long> extents) {
  mobula_hip_set_stream(c10::hip::getCurrentHIPStream(on.device().index()).stream(), 0);
  mobula_hip_set_arg_extents(extents.begin(), static_cast<int>(extents.size()));
}

void raise_if_failed(const char* what) {
  const char* text = mobula_hip_last_error();
  if (text == nullptr) return;
  const std::string message = std::string(what) + ": " + text;
  mobula_hip_clear_error();
  throw std::runtime_error(message);
}

// A gradient whose values lie in memory of its own (a batched one, or one without values, has none).
const Tensor& with_values(const Tensor& dy) {
  TORCH_CHECK(dy.has_storage() && (dy.numel() == 0 || dy.const_data_ptr() != nullptr),
              "the gradient of the output has no values in memory: batched and fake tensors are not taken");
  return dy;
}

bool is_channels_last(const Tensor& t) {
  return !t.is_contiguous() && t.is_contiguous(at::MemoryFormat::ChannelsLast);
}

// ---- ROIAlign ---------------------------------------------------------------

struct RoiAlignArgs {
  int PH, PW, S;
  double scale;
};

// The four entry points of an element type; channels-last ones may be missing (binary64).
template <typename T, typename B>
struct RoiAlignSymbols {
  void (*forward)(int, int, const T*, B, int, int, int, int, int, int, const B*, T*);
  void (*assign)(int, int, const T*, B, int, int, int, int, int, int, int, T*, const B*);
  void (*forward_nhwc)(int, int, const T*, float, int, int, int, int, int, int, const float*, T*);
  void (*assign_nhwc)(int, int, const T*, float, int, int, int, int, int, int, int, T*, const float*);
};
const RoiAlignSymbols<float, float> kFloat = {roi_align_forward_ab78de3c, roi_align_backward_assign_a8793cbe,
                                              roi_align_forward_nhwc_ab78de3c, roi_align_backward_nhwc_assign_a8793cbe};
const RoiAlignSymbols<unsigned short, float> kHalf = {roi_align_forward_e874c59a, roi_align_backward_assign_7924dbc8,
                                                      roi_align_forward_nhwc_e874c59a,
                                                      roi_align_backward_nhwc_assign_7924dbc8};
const RoiAlignSymbols<unsigned short, float> kBFloat16 = {roi_align_forward_f951d439, roi_align_backward_assign_86156afd,
                                                          roi_align_forward_nhwc_f951d439,
                                                          roi_align_backward_nhwc_assign_86156afd};
const RoiAlignSymbols<double, double> kDouble = {roi_align_forward_6b9e6c9b, roi_align_backward_assign_4620f85e,
                                                 nullptr, nullptr};

// f(symbols of the tensor's element type)
template <typename F>
void with_symbols(at::ScalarType type, const F& f) {
  if (type == at::kFloat) f(kFloat);
  else if (type == at::kHalf) f(kHalf);
  else if (type == at::kBFloat16) f(kBFloat16);
  else f(kDouble);
}

template <typename T, typename B>
void call_forward(const RoiAlignSymbols<T, B>& s, bool nhwc, const Tensor& x, const Tensor& rois, const Tensor& y,
                  const RoiAlignArgs& a) {
  const int dev = x.device().index(), n = static_cast<int>(y.numel());
  const int C = x.size(1), H = x.size(2), W = x.size(3);
  begin(x, {-1, x.numel(), -1, -1, -1, -1, -1, -1, -1, rois.numel(), y.numel()});
  const T* xp = static_cast<const T*>(x.data_ptr());
  T* yp = static_cast<T*>(y.data_ptr());
  if (nhwc)
    s.forward_nhwc(dev, n, xp, static_cast<float>(a.scale), C, H, W, a.PH, a.PW, a.S,
                   static_cast<const float*>(rois.data_ptr()), yp);
  else
    s.forward(dev, n, xp, static_cast<B>(a.scale), C, H, W, a.PH, a.PW, a.S, static_cast<const B*>(rois.data_ptr()), yp);
  raise_if_failed(nhwc ? "roi_align_forward_nhwc" : "roi_align_forward");
}

// false: the channels-last entry point had no room for a larger grid's weights, where the other one falls back
template <typename T, typename B>
bool call_assign(const RoiAlignSymbols<T, B>& s, bool nhwc, const Tensor& dy, const Tensor& rois, const Tensor& dx,
                 const RoiAlignArgs& a) {
  const int dev = dx.device().index(), n = static_cast<int>(dy.numel());
  const int N = dx.size(0), C = dx.size(1), H = dx.size(2), W = dx.size(3);
  begin(dx, {-1, dy.numel(), -1, -1, -1, -1, -1, -1, -1, -1, dx.numel(), rois.numel()});
  const T* dyp = static_cast<const T*>(dy.data_ptr());
  T* dxp = static_cast<T*>(dx.data_ptr());
  if (nhwc) {
    s.assign_nhwc(dev, n, dyp, static_cast<float>(a.scale), C, H, W, a.PH, a.PW, a.S, N, dxp,
                  static_cast<const float*>(rois.data_ptr()));
    if (mobula_hip_last_error() != nullptr && a.S != 1 && a.S != 2) {
      mobula_hip_clear_error();
      return false;
    }
  } else {
    s.assign(dev, n, dyp, static_cast<B>(a.scale), C, H, W, a.PH, a.PW, a.S, N, dxp,
             static_cast<const B*>(rois.data_ptr()));
  }
  raise_if_failed(nhwc ? "roi_align_backward_nhwc_assign" : "roi_align_backward_assign");
  return true;
}

bool nhwc_taken(bool backward, const Tensor& map, const RoiAlignArgs& a, int64_t rois) {
  return map.scalar_type() != at::kDouble &&
         mobula_hip_roialign_nhwc_supported(backward ? 1 : 0, static_cast<int>(map.element_size()), map.size(1),
                                            map.size(2), map.size(3), a.PH, a.PW, a.S, rois) != 0;
}

// dst = src where one is dense and the other channels-last (any other pair is torch's to copy).
void copy_format(const Tensor& src, const Tensor& dst) {
  const bool from_last = is_channels_last(src) && dst.is_contiguous();
  const int64_t bytes = src.element_size();
  const bool pair = from_last || (src.is_contiguous() && is_channels_last(dst));
  if (!pair || src.dim() != 4 || (bytes != 2 && bytes != 4) || src.is_neg() || src._is_zerotensor() ||
      src.size(0) >= (1ll << 28) || src.numel() >= (1ll << 38) || src.size(1) >= (1ll << 24) ||
      src.size(2) * src.size(3) >= (1ll << 24)) {   // (what the library's kernel takes)
    dst.copy_(src);
    return;
  }
  const int64_t channels = src.size(1), pixels = src.size(2) * src.size(3);
  begin(src, {});
  mobula_hip_transpose_planes(src.device().index(), src.size(0), from_last ? pixels : channels, from_last ? channels : pixels,
                              static_cast<int>(bytes), src.data_ptr(), dst.data_ptr());
  raise_if_failed("transpose_planes");
}
Tensor in_format(const Tensor& t, at::MemoryFormat format) {
  if (t.is_contiguous(format)) return t;
  const Tensor out = at::empty(t.sizes(), t.options().memory_format(format));
  copy_format(t, out);
  return out;
}

Tensor roi_align_forward(const Tensor& x, const Tensor& rois, const RoiAlignArgs& a) {
  const bool keeps_format = is_channels_last(x);
  const Tensor y = at::empty({rois.size(0), x.size(1), a.PH, a.PW},
                             x.options().memory_format(keeps_format ? at::MemoryFormat::ChannelsLast
                                                                    : at::MemoryFormat::Contiguous));
  const Tensor r = rois.contiguous();
  // (a pooled map of one bin is dense in both formats, and then not taken for a channels-last one)
  const bool nhwc = keeps_format && is_channels_last(y) && nhwc_taken(false, x, a, r.size(0));
  const Tensor xd = nhwc ? x : in_format(x, at::MemoryFormat::Contiguous);
  const Tensor yd = nhwc || y.is_contiguous() ? y : at::empty(y.sizes(), x.options());
  with_symbols(x.scalar_type(), [&](const auto& s) { call_forward(s, nhwc, xd, r, yd, a); });
  if (!yd.is_same(y)) copy_format(yd, y);
  return y;
}

struct RoiAlignBackward : public Node {
  RoiAlignArgs args;
  Tensor rois;
  Tensor like;   // the map: its format, type and place, not its values

  variable_list apply(variable_list&& grads) override {
    at::AutoDispatchBelowADInplaceOrView guard;
    variable_list out(2);
    if (!grads[0].defined()) return out;
    if (task_should_compute_output(0)) out[0] = data_gradient(with_values(grads[0]));
    if (task_should_compute_output(1)) out[1] = at::zeros_like(rois);   // no gradient flows to the boxes
    return out;
  }

  Tensor data_gradient(const Tensor& dy) const {
    const Tensor dx = at::empty_like(like);
    const Tensor r = rois.contiguous();
    if (is_channels_last(dx) && nhwc_taken(true, dx, args, r.size(0))) {
      const Tensor d = in_format(dy, at::MemoryFormat::ChannelsLast);
      bool taken = false;
      with_symbols(dx.scalar_type(), [&](const auto& s) { taken = call_assign(s, true, d, r, dx, args); });
      if (taken) return dx;
    }
    const Tensor d = in_format(dy, at::MemoryFormat::Contiguous);
    const Tensor dense = dx.is_contiguous() ? dx : at::empty(dx.sizes(), dx.options());
    with_symbols(dx.scalar_type(), [&](const auto& s) { call_assign(s, false, d, r, dense, args); });
    if (!dense.is_same(dx)) copy_format(dense, dx);
    return dx;
  }

  void release_variables() override {}
};

Tensor roi_align(const Tensor& x, const Tensor& rois, const RoiAlignArgs& a) {
  Tensor y;
  {
    at::AutoDispatchBelowADInplaceOrView guard;
    y = roi_align_forward(x, rois, a);
  }
  if (torch::autograd::compute_requires_grad(x, rois)) {
    std::shared_ptr<RoiAlignBackward> node(new RoiAlignBackward(), torch::autograd::deleteNode);
    node->args = a;
    node->rois = rois.detach();
    node->like = x.detach();
    node->set_next_edges(torch::autograd::collect_next_edges(x, rois));
    torch::autograd::set_history(y, node);
  }
  return y;
}

// ---- Conv2D -----------------------------------------------------------------

struct ConvArgs {
  int D, kernel[2], stride[2], pad[2], dil[2];
};

#define GEOMETRY_OF(x, a)                                                                                    \
  static_cast<int>((x).size(0)), static_cast<int>((x).size(1)), static_cast<int>((x).size(2)),              \
      static_cast<int>((x).size(3)), (a).D, (a).kernel[0], (a).kernel[1], (a).pad[0], (a).pad[1],           \
      (a).stride[0], (a).stride[1], (a).dil[0], (a).dil[1]

struct Conv2DBackward : public Node {
  ConvArgs args;
  Tensor x, weight, bias;

  variable_list apply(variable_list&& grads) override {
    at::AutoDispatchBelowADInplaceOrView guard;
    variable_list out(bias.defined() ? 3 : 2);
    if (!grads[0].defined()) return out;
    const Tensor dy = with_values(grads[0]).contiguous();
    const ConvArgs& a = args;
    const int dev = dy.device().index();
    const bool want_x = task_should_compute_output(0), want_w = task_should_compute_output(1);
    const bool want_b = bias.defined() && task_should_compute_output(2);
    if (want_x || want_w || want_b) {
      if (want_x) out[0] = at::empty_like(x);
      if (want_w) out[1] = at::empty_like(weight);
      if (want_b) out[2] = at::empty_like(bias);
      auto dense = [](const Tensor& t) { return !t.defined() || t.is_contiguous() ? t : at::empty(t.sizes(), t.options()); };
      const Tensor dx = dense(out[0]), dw = dense(out[1]), db = want_b ? dense(out[2]) : Tensor();
      // (x is read for the weights' gradient, the weights for that of x)
      const Tensor xd = want_w ? x.contiguous() : x, w = want_x ? weight.contiguous() : weight;
      begin(dy, {});
      mobula_hip_conv2d_gradients(dev, dy.data_ptr<float>(), xd.data_ptr<float>(), w.data_ptr<float>(), GEOMETRY_OF(x, a),
                                  want_x ? dx.data_ptr<float>() : nullptr, want_w ? dw.data_ptr<float>() : nullptr,
                                  want_b ? db.data_ptr<float>() : nullptr);
      raise_if_failed("conv2d_backward");
      if (want_x && !dx.is_same(out[0])) out[0].copy_(dx);
      if (want_w && !dw.is_same(out[1])) out[1].copy_(dw);
      if (want_b && !db.is_same(out[2])) out[2].copy_(db);
    }
    return out;
  }

  void release_variables() override {}
};

Tensor conv2d(const Tensor& x, const Tensor& weight, const Tensor& bias, const ConvArgs& a, int64_t OH, int64_t OW) {
  Tensor y;
  {
    at::AutoDispatchBelowADInplaceOrView guard;
    y = at::empty({x.size(0), a.D, OH, OW}, x.options().memory_format(at::MemoryFormat::Contiguous));
    const Tensor xd = x.contiguous(), w = weight.contiguous(), b = bias.defined() ? bias.contiguous() : w;
    begin(x, {-1, xd.numel(), w.numel(), b.numel(), -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, -1, y.numel()});
    conv2d_forward_c6a7aa85(x.device().index(), static_cast<int>(y.numel()), xd.data_ptr<float>(), w.data_ptr<float>(),
                            b.data_ptr<float>(), bias.defined() ? 1 : 0, GEOMETRY_OF(x, a), y.data_ptr<float>());
    raise_if_failed("conv2d_forward");
  }
  const bool has_bias = bias.defined();
  if (has_bias ? torch::autograd::compute_requires_grad(x, weight, bias)
               : torch::autograd::compute_requires_grad(x, weight)) {
    std::shared_ptr<Conv2DBackward> node(new Conv2DBackward(), torch::autograd::deleteNode);
    node->args = a;
    node->x = x.detach();
    node->weight = weight.detach();
    if (has_bias) node->bias = bias.detach();
    node->set_next_edges(has_bias ? torch::autograd::collect_next_edges(x, weight, bias)
                                  : torch::autograd::collect_next_edges(x, weight));
    torch::autograd::set_history(y, node);
  }
  return y;
}

// ---- arguments --------------------------------------------------------------

// The values of a vectorcall by parameter name; false: a name that is not there, a value given
// twice, too many of them.
bool by_name(const char* const* names, int count, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames,
             PyObject** out) {
  if (nargs > count) return false;
  for (int i = 0; i < count; ++i) out[i] = i < nargs ? args[i] : nullptr;
  const Py_ssize_t nkw = kwnames == nullptr ? 0 : PyTuple_GET_SIZE(kwnames);
  for (Py_ssize_t k = 0; k < nkw; ++k) {
    PyObject* const name = PyTuple_GET_ITEM(kwnames, k);
    int at = -1;
    for (int i = 0; i < count && at < 0; ++i)
      if (PyUnicode_CompareWithASCIIString(name, names[i]) == 0) at = i;
    if (at < 0 || out[at] != nullptr) return false;
    out[at] = args[nargs + k];
  }
  return true;
}

bool read_int(PyObject* o, int* out) {
  if (o == nullptr || !PyLong_CheckExact(o)) return false;
  int overflow = 0;
  const long v = PyLong_AsLongAndOverflow(o, &overflow);
  if (overflow != 0 || v < INT_MIN || v > INT_MAX) return false;
  *out = static_cast<int>(v);
  return true;
}

bool read_pair(PyObject* o, int (&out)[2]) {
  if (o == nullptr || !(PyTuple_CheckExact(o) || PyList_CheckExact(o)) || PySequence_Fast_GET_SIZE(o) != 2) return false;
  return read_int(PySequence_Fast_GET_ITEM(o, 0), &out[0]) && read_int(PySequence_Fast_GET_ITEM(o, 1), &out[1]);
}

// Hooks on every module's calls (torch.nn.modules.module.register_module_*_hook): the operator class's
// call is one, of an nn.Module.
bool has_module_hooks() {
  static PyObject* const module = PyImport_ImportModule("torch.nn.modules.module");
  static PyObject* const names[] = {
      PyUnicode_InternFromString("_global_forward_pre_hooks"), PyUnicode_InternFromString("_global_forward_hooks"),
      PyUnicode_InternFromString("_global_backward_pre_hooks"), PyUnicode_InternFromString("_global_backward_hooks")};
  if (module == nullptr) { PyErr_Clear(); return true; }
  PyObject* const scope = PyModule_GetDict(module);
  for (PyObject* const name : names) {
    PyObject* const hooks = name == nullptr ? nullptr : PyDict_GetItemWithError(scope, name);
    if (hooks == nullptr || !PyDict_Check(hooks) || PyDict_Size(hooks) != 0) {
      PyErr_Clear();
      return true;
    }
  }
  return false;
}

// A call that torch watches or transforms (torch.func, tracing, a dispatch mode, hooks): what it needs to
// see is the operator class's module and autograd function.
bool is_watched() {
  return at::tracer::impl::is_dispatch_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
         c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) || has_module_hooks();
}

// A plain tensor (or parameter) on a GPU, with memory of its own and no forward-mode tangent.
bool read_tensor(PyObject* o, Tensor* out) {
  if (o == nullptr || !THPVariable_CheckExact(o)) return false;
  const Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda() || t.layout() != at::kStrided || t.is_conj() || t.is_neg() || !t.has_storage() ||
      t.numel() > INT_MAX || t._fw_grad(0).defined())
    return false;
  *out = t;
  return true;
}

PyObject* not_taken() { Py_RETURN_NOTIMPLEMENTED; }

PyObject* py_roi_align(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
  HANDLE_TH_ERRORS
  static const char* const names[] = {"data", "rois", "pooled_size", "spatial_scale", "sampling_ratio"};
  PyObject* v[5];
  Tensor x, rois;
  RoiAlignArgs a;
  int pooled[2];
  if (is_watched() || !by_name(names, 5, args, nargs, kwnames, v) || !read_tensor(v[0], &x) || !read_tensor(v[1], &rois) ||
      !read_pair(v[2], pooled) || v[3] == nullptr || !(PyFloat_Check(v[3]) || PyLong_CheckExact(v[3])) ||
      !read_int(v[4], &a.S))
    return not_taken();
  a.scale = PyFloat_AsDouble(v[3]);
  if (a.scale == -1.0 && PyErr_Occurred() != nullptr) { PyErr_Clear(); return not_taken(); }
  a.PH = pooled[0]; a.PW = pooled[1];
  const at::ScalarType type = x.scalar_type();
  if ((type != at::kFloat && type != at::kHalf && type != at::kBFloat16 && type != at::kDouble) ||
      rois.scalar_type() != (type == at::kDouble ? at::kDouble : at::kFloat) || x.device() != rois.device() ||
      x.dim() != 4 || rois.dim() != 2 || rois.size(1) != 5 || a.PH <= 0 || a.PW <= 0 ||
      static_cast<double>(rois.size(0)) * x.size(1) * a.PH * a.PW > INT_MAX)
    return not_taken();
  Tensor y;
  {
    pybind11::gil_scoped_release no_gil;
    y = roi_align(x, rois, a);
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

PyObject* py_conv2d(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
  HANDLE_TH_ERRORS
  static const char* const names[] = {"x", "weight", "bias", "channels", "kernel_size", "strides", "padding",
                                      "dilation"};
  PyObject* v[8];
  // positional values are taken for the tensors only: how many of them are inputs is a question
  // for the operator class otherwise
  if (nargs > 3 || is_watched() || !by_name(names, 8, args, nargs, kwnames, v)) return not_taken();
  Tensor x, weight, bias;
  ConvArgs a;
  a.stride[0] = a.stride[1] = a.dil[0] = a.dil[1] = 1;
  a.pad[0] = a.pad[1] = 0;
  if (!read_tensor(v[0], &x) || !read_tensor(v[1], &weight) || (v[2] != nullptr && !read_tensor(v[2], &bias)) ||
      !read_int(v[3], &a.D) || !read_pair(v[4], a.kernel) || (v[5] != nullptr && !read_pair(v[5], a.stride)) ||
      (v[6] != nullptr && !read_pair(v[6], a.pad)) || (v[7] != nullptr && !read_pair(v[7], a.dil)))
    return not_taken();
  if (x.scalar_type() != at::kFloat || weight.scalar_type() != at::kFloat || x.device() != weight.device() ||
      x.dim() != 4 || weight.dim() != 4 || a.D <= 0 || weight.size(0) != a.D || weight.size(1) != x.size(1) ||
      weight.size(2) != a.kernel[0] || weight.size(3) != a.kernel[1])
    return not_taken();
  if (bias.defined() && (bias.scalar_type() != at::kFloat || bias.device() != x.device() || bias.dim() != 1 ||
                         bias.size(0) != a.D))
    return not_taken();
  int64_t out[2];
  for (int i = 0; i < 2; ++i) {
    const int64_t reach = static_cast<int64_t>(a.dil[i]) * (a.kernel[i] - 1) + 1;
    const int64_t room = x.size(2 + i) + 2ll * a.pad[i] - reach;
    if (a.kernel[i] <= 0 || a.stride[i] <= 0 || a.dil[i] <= 0 || a.pad[i] < 0 || room < 0) return not_taken();
    out[i] = room / a.stride[i] + 1;
  }
  if (static_cast<double>(x.size(0)) * a.D * out[0] * out[1] > INT_MAX) return not_taken();
  Tensor y;
  {
    pybind11::gil_scoped_release no_gil;
    y = conv2d(x, weight, bias, a, out[0], out[1]);
  }
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"ROIAlign", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_roi_align)),
     METH_FASTCALL | METH_KEYWORDS, "ROIAlign(data, rois, pooled_size, spatial_scale, sampling_ratio)"},
    {"Conv2D", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(py_conv2d)), METH_FASTCALL | METH_KEYWORDS,
     "Conv2D(x, weight, bias=None, channels, kernel_size, strides, padding, dilation)"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_direct", "The bundled operators for torch tensors on a GPU.", -1,
                      methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__torch_direct(void) { return PyModule_Create(&module); }
