// The autograd node of a small loss (_small.py), native.
//
// A backward pass over CUDA tensors runs on a thread of PyTorch's own, and a node written in Python needs the interpreter
// there: of a loss of 256 x 256 x 16 (one launch of 10 us behind it) the pass took 92 us, 42 of them in the node; with this one 28 to
// 50, and the forward pass behind it, whose thread has not lost the interpreter meanwhile, 64 for 100.  Loss and
// both gradients 194 -> 119 us.  What the node does not know (a graph of the gradient, weights that need
// one, points in double precision) it asks Python for, with the tensors it has saved.
#include <c10/core/SafePyObject.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/PyInterpreter.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>
#include <torch/csrc/utils/pybind.h>

#include <array>
#include <cstring>
#include <mutex>

#include "flash_sinkhorn_hip.h"

namespace {

namespace py = pybind11;
using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::Variable;
using torch::autograd::variable_list;

using GradFn = int (*)(const fs_small_problem*, void*, size_t, const float*, float*, float*, void*);

// x, y as the caller gave them; then what the solve read and left: points, weights, workspace, potentials
// (Solved.tensors).  Undefined where there is none.
constexpr int kGiven = 2, kSaved = kGiven + 6;

struct SmallLoss : public Node {
  SmallLoss(const fs_small_problem& problem, GradFn grad, py::object ask, std::array<Tensor, kSaved> tensors, at::IntArrayRef shape)
      : form(problem), grad(grad), ask(ask.release().ptr(), getPyInterpreter()), shape(shape.vec()) {
    for (int i = 0; i < kSaved; ++i) saved[i] = SavedVariable(tensors[i], false);
    plain = tensors[0].scalar_type() == at::kFloat || tensors[0].scalar_type() == at::kHalf ||
            tensors[0].scalar_type() == at::kBFloat16;
  }

  variable_list apply(variable_list&& grads) override {
    const std::array<Tensor, kSaved> t = unpacked();
    const Tensor out = grads[0].defined() ? grads[0] : at::zeros(shape, t[2].options().dtype(at::kFloat));
    std::array<bool, 4> need;
    for (int i = 0; i < 4; ++i) need[i] = edge[i] >= 0 && task_should_compute_output(edge[i]);
    variable_list result(num_outputs());
    auto give = [&](int i, Tensor v) { result[edge[i]] = std::move(v); };
    if (at::GradMode::is_enabled() || need[2] || need[3] || !plain) {
      ask_python(out, t, need, give);
      return result;
    }
    if (!need[0] && !need[1]) return result;
    std::array<Tensor, 2> g;
    for (int i = 0; i < 2; ++i)
      if (need[i]) g[i] = at::empty(t[2 + i].sizes(), t[2].options().dtype(at::kFloat));
    const Tensor scale = out.to(at::kFloat).contiguous();
    fs_small_problem p = form;
    p.x = t[2].data_ptr();
    p.y = t[3].data_ptr();
    p.a = t[4].defined() ? t[4].data_ptr<float>() : nullptr;
    p.b = t[5].defined() ? t[5].data_ptr<float>() : nullptr;
    const int rc = grad(&p, t[6].data_ptr(), t[6].nbytes(), scale.data_ptr<float>(), need[0] ? g[0].data_ptr<float>() : nullptr,
                        need[1] ? g[1].data_ptr<float>() : nullptr, c10::hip::getCurrentHIPStream(t[2].device().index()).stream());
    TORCH_CHECK(rc == FS_OK, "fs_small_grad failed (code ", rc, ")");
    for (int i = 0; i < 2; ++i)
      if (need[i]) give(i, g[i]);
    return result;
  }

  std::array<Tensor, kSaved> unpacked() {
    std::lock_guard<std::mutex> lock(mutex_);
    std::array<Tensor, kSaved> t;
    for (int i = 0; i < kSaved; ++i) t[i] = saved[i].unpack();
    return t;
  }

  template <typename Give>
  void ask_python(const Tensor& out, const std::array<Tensor, kSaved>& t, const std::array<bool, 4>& need, Give&& give) {
    py::gil_scoped_acquire gil;
    py::list tensors;
    for (const Tensor& v : t) tensors.append(v.defined() ? py::cast(v) : py::none());
    const py::tuple got = py::reinterpret_borrow<py::object>(ask.ptr(getPyInterpreter()))(
        out, tensors, py::make_tuple(need[0], need[1], need[2], need[3]));
    for (int i = 0; i < 4; ++i)
      if (need[i] && !got[i].is_none()) give(i, got[i].cast<Tensor>());
  }

  void release_variables() override {
    {
      std::lock_guard<std::mutex> lock(mutex_);
      for (SavedVariable& v : saved) v.reset_data();
    }
    std::shared_ptr<Node> gone;  // (with Python in it: not under the lock)
    std::lock_guard<std::mutex> lock(late_lock);
    gone.swap(late);
  }

  // Compiled autograd (PyTorch's, which records a backward pass as a graph): left to a node of a Python Function over the
  // same tensors, whose call it records as one operation.  It goes through the nodes of a pass one after the other, on one thread.
  void compiled_args(torch::dynamo::autograd::CompiledNodeArgs& args) const override {
    std::array<Tensor, kSaved> t;
    {
      py::gil_scoped_release release;  // (a hook that unpacks a tensor takes it, under the node's lock)
      t = const_cast<SmallLoss*>(this)->unpacked();
    }
    py::list tensors, given;
    for (const Tensor& v : t) tensors.append(v.defined() ? py::cast(v) : py::none());
    for (int i = 0; i < 4; ++i) {  // stand-ins: where the gradients go is this node's
      if (edge[i] < 0) {
        given.append(py::none());
        continue;
      }
      const torch::autograd::Edge& e = next_edge(edge[i]);
      if (!e.is_valid()) {
        given.append(py::cast(at::empty({0}, t[2].options().dtype(at::kFloat))));
        continue;
      }
      const torch::autograd::InputMetadata& m = e.function->input_metadata(e.input_nr);
      given.append(py::cast(at::empty_symint(m.shape_as_dim_vector(), m.options()).requires_grad_()));
    }
    const py::object out = py::reinterpret_borrow<py::object>(ask.ptr(getPyInterpreter())).attr("node")(tensors, shape, given);
    std::shared_ptr<Node> node = out.cast<Tensor>().grad_fn();
    if (node) node->compiled_args(args);
    std::lock_guard<std::mutex> lock(late_lock);
    late.swap(node);
  }
  variable_list apply_with_saved(const variable_list& inputs, torch::dynamo::autograd::SwapSavedVariables& saved) override {
    std::shared_ptr<Node> node;
    {
      std::lock_guard<std::mutex> lock(late_lock);
      node = late;
    }
    return node ? node->apply_with_saved(inputs, saved) : variable_list(num_outputs());
  }

  std::string name() const override { return "SmallLossBackward"; }

  fs_small_problem form;
  GradFn grad;
  c10::SafePyObject ask;
  std::vector<int64_t> shape;
  std::array<SavedVariable, kSaved> saved;
  std::array<int, 4> edge{-1, -1, -1, -1};  // of x, y and the weights that there are
  bool plain;
  mutable std::shared_ptr<Node> late;  // see compiled_args
  mutable std::mutex late_lock;
};

// Whether autograd sees nothing in these tensors but what a node of this kind serves: no transform of functorch, no
// tangents, no subclass (a Function refuses or serves those).
bool ordinary(const std::vector<std::optional<Tensor>>& tensors) {
  const c10::DispatchKeySet other({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                   c10::DispatchKey::Functionalize});
  for (const auto& t : tensors)
    if (t.has_value() && t->defined()) {
      if (t->key_set().has_any(other) || t->_fw_grad(0).defined()) return false;
    }
  return true;
}

Tensor attach(Tensor loss, std::optional<Tensor> a, std::optional<Tensor> b, const std::vector<std::optional<Tensor>>& tensors,
              uintptr_t form, size_t form_bytes, uintptr_t grad, py::object ask) {
  TORCH_CHECK(form_bytes == sizeof(fs_small_problem) && tensors.size() == kSaved, "the library and its binding differ");
  fs_small_problem p;
  std::memcpy(&p, reinterpret_cast<const void*>(form), sizeof(p));
  p.x = p.y = nullptr;
  p.a = p.b = p.eps_list = nullptr;
  std::array<Tensor, kSaved> t;
  for (int i = 0; i < kSaved; ++i) t[i] = tensors[i].value_or(Tensor());
  std::shared_ptr<SmallLoss> node(new SmallLoss(p, reinterpret_cast<GradFn>(grad), std::move(ask), t, loss.sizes()),
                                  torch::autograd::deleteNode);
  torch::autograd::edge_list edges;
  const std::array<Tensor, 4> given{t[0], t[1], a.value_or(Tensor()), b.value_or(Tensor())};
  for (int i = 0; i < 4; ++i)
    if (given[i].defined()) {
      node->edge[i] = (int)edges.size();
      edges.push_back(torch::autograd::impl::gradient_edge(given[i]));
    }
  node->set_next_edges(std::move(edges));
  torch::autograd::set_history(loss, node);
  return loss;
}

}  // namespace

PYBIND11_MODULE(_native, m) {
  m.def("ordinary", &ordinary);
  m.def("attach", &attach);
}
