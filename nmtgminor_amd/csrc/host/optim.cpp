// Gradient clipping and the Adam step over a model's parameter list: gathers the addresses and enqueues the multi-tensor
// passes. The interpreter took 0.9 ms for this with 193 tensors (an attribute, a check and a ctypes object per tensor and
// list), longer than the kernels for 60 M elements; here it is about 0.1 ms. What is not the plain case (several dtypes,
// moments that do not exist yet, layouts that need a copy) is left to the Python side, before anything is launched.
#include "host.h"
#include <torch/csrc/autograd/python_variable.h>

namespace nmtg_host {
namespace {

namespace py = pybind11;

bool supported(const Tensor& t, at::ScalarType type, at::Device device) {
  return t.defined() && t.layout() == at::kStrided && t.scalar_type() == type && t.device() == device && t.is_contiguous();
}

bool float_type(at::ScalarType t) { return t == at::kFloat || t == at::kHalf || t == at::kBFloat16; }

struct Lists {
  std::vector<void*> addr[4];
  std::vector<int64_t> size;
  Tensor first;
};

void* address(const Tensor& t) { return t.numel() ? t.data_ptr() : nullptr; }

optional<Tensor> clip_grad_norm(const py::list& params, double max_norm) {
  Lists l;
  for (py::handle h : params) {
    if (!THPVariable_Check(h.ptr())) return {};
    const Tensor& grad = THPVariable_Unpack(h.ptr()).grad();
    if (!grad.defined()) continue;
    if (!l.first.defined()) {
      if (!grad.is_cuda() || !float_type(grad.scalar_type())) return {};
      l.first = grad;
    }
    if (!supported(grad, l.first.scalar_type(), l.first.device())) return {};
    l.addr[0].push_back(address(grad));
    l.size.push_back(grad.numel());
  }
  if (l.size.empty()) return {};
  Launch on(l.first);
  const int n = static_cast<int>(l.size.size()), type = dtype_code(l.first);
  Tensor norm = empty_as(l.first, {}, at::kFloat);
  const Scratch ws(l.first, std::max<int64_t>(api.multi_tensor_l2norm_workspace_bytes(n, l.size.data()), 256));
  check(api.multi_tensor_l2norm(n, l.addr[0].data(), l.size.data(), norm.data_ptr<float>(), nullptr, ws.get(), ws.bytes, type, on.stream),
        "nmtg_multi_tensor_l2norm");
  if (max_norm > 0.0)
    check(api.multi_tensor_clip(n, l.addr[0].data(), l.size.data(), norm.data_ptr<float>(), static_cast<float>(max_norm), type, on.stream),
          "nmtg_multi_tensor_clip");
  return norm;
}

// state: the optimizer's, a dict from parameter to {exp_avg, exp_avg_sq}. One set of lists per dtype.
bool adam_step(const py::list& params, const py::dict& state, double lr, double beta1, double beta2, double eps, int64_t step, int64_t mode,
               bool bias_correction, double weight_decay) {
  const at::ScalarType types[3] = {at::kFloat, at::kHalf, at::kBFloat16};
  Lists lists[3];
  const py::str names[2] = {py::str("exp_avg"), py::str("exp_avg_sq")};

  optional<at::Device> device;
  for (py::handle h : params) {
    if (!THPVariable_Check(h.ptr())) return false;
    const Tensor& p = THPVariable_Unpack(h.ptr());
    const Tensor& grad = p.grad();
    if (!grad.defined()) continue;
    if (!device) device = p.device();
    const auto type = p.scalar_type();
    if (!p.is_cuda() || !float_type(type) || !supported(p, type, *device) || !supported(grad, type, *device)) return false;
    PyObject* entry = PyDict_GetItemWithError(state.ptr(), h.ptr());
    if (entry == nullptr || !PyDict_Check(entry)) {
      PyErr_Clear();
      return false;
    }
    Tensor moments[2];
    for (int i = 0; i < 2; ++i) {
      PyObject* m = PyDict_GetItemWithError(entry, names[i].ptr());
      if (m == nullptr || !THPVariable_Check(m)) {
        PyErr_Clear();
        return false;
      }
      moments[i] = THPVariable_Unpack(m);
      if (!supported(moments[i], type, *device) || moments[i].numel() != p.numel()) return false;
    }
    Lists& l = lists[type == types[0] ? 0 : type == types[1] ? 1 : 2];
    l.first = p;
    const Tensor* four[4] = {&grad, &p, &moments[0], &moments[1]};
    for (int i = 0; i < 4; ++i) l.addr[i].push_back(address(*four[i]));
    l.size.push_back(p.numel());
  }
  for (Lists& l : lists) {
    if (l.size.empty()) continue;
    Launch on(l.first);
    check(api.multi_tensor_adam(static_cast<int>(l.size.size()), l.addr[0].data(), l.addr[1].data(), l.addr[2].data(), l.addr[3].data(),
                                l.size.data(), static_cast<float>(lr), static_cast<float>(beta1), static_cast<float>(beta2),
                                static_cast<float>(eps), static_cast<int>(step), static_cast<int>(mode), bias_correction ? 1 : 0,
                                static_cast<float>(weight_decay), dtype_code(l.first), on.stream), "nmtg_multi_tensor_adam");
  }
  return true;
}

}  // namespace

void define_optim(pybind11::module_& m) {
  m.def("clip_grad_norm", &clip_grad_norm);
  m.def("adam_step", &adam_step);
}

}  // namespace nmtg_host
