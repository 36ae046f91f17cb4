// Shared by the sources of the _mpa_host extension: argument conversion and the operators that the
// layer code calls.
#pragma once

#include <torch/extension.h>

#include <ATen/core/grad_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <array>
#include <optional>

#include "../../include/mambapy_amd.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;
typedef std::optional<Tensor> Opt;

namespace mpa_host {

// launch-plan fields, in the order of scan.py: LaunchPlan.packed
struct Plan {
    int fwd_ns = 0, bwd_ns = 0, fwd_segments = 0, bwd_segments = 0, flags = 0, pscan_chunks = 0;
};
typedef std::array<int, 6> PackedPlan;
inline Plan unpack(const PackedPlan& p) { return Plan{p[0], p[1], p[2], p[3], p[4], p[5]}; }

inline Tensor val(const Opt& t) { return t.has_value() ? *t : Tensor(); }

inline int io_dtype(at::ScalarType t) {
    if (t == at::kFloat) return MPA_F32;
    TORCH_CHECK_TYPE(t == at::kBFloat16, "unsupported dtype ", t,
                     ": the kernels take float32 or bfloat16 tensors (state and accumulation are float32 in both cases)");
    return MPA_BF16;
}

inline void require_gpu(std::initializer_list<const Tensor*> ts) {
    for (const Tensor* t : ts)
        TORCH_CHECK(!t->defined() || t->is_cuda(),
                    "mambapy_amd ops need tensors on a ROCm device (there is no CPU implementation in this package)");
}

inline void check(int rc, const char* what) {
    TORCH_CHECK(rc == MPA_OK, what, " failed with status ", rc, ": ", mpa_status_string(rc));
}

inline void* ptr(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
inline float* fptr(const Tensor& t) { return static_cast<float*>(ptr(t)); }
inline void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

inline Tensor cast(const Tensor& t, at::ScalarType dt) { return t.defined() && t.scalar_type() != dt ? t.to(dt) : t; }
inline Tensor f32c(const Tensor& t) { return t.defined() ? cast(t, at::kFloat).contiguous() : t; }
inline Tensor dense(const Tensor& t) { return t.defined() ? t.contiguous() : t; }  // (a saved tensor may come back with other strides)
inline Tensor dense16(const Tensor& t) {  // ... and may start anywhere, as a view of a flat buffer does; for kernels with 16-byte loads
    const Tensor c = dense(t);
    return c.defined() && reinterpret_cast<uintptr_t>(c.const_data_ptr()) % 16 ? c.clone() : c;
}
inline Tensor unit_rows(const Tensor& t) { return t.stride(-1) == 1 ? t : t.contiguous(); }
inline Tensor empty(at::IntArrayRef shape, at::ScalarType dt, const Tensor& like) {
    return at::empty(shape, at::TensorOptions().dtype(dt).device(like.device()));
}
inline Tensor scratch(size_t bytes, const Tensor& like) { return empty({(int64_t)bytes}, at::kByte, like); }

inline bool tracked(std::initializer_list<const Tensor*> ts) {
    if (!at::GradMode::is_enabled()) return false;
    for (const Tensor* t : ts)
        if (t->defined() && t->requires_grad()) return true;
    return false;
}

// Forward-mode derivatives: the entry points run below autograd and have no rule for them.  Operators refuse a dual
// tensor; layers leave it to the composed path, whose operators do.  (functorch's wrapped tensors, of vmap and of its own
// grad and jvp, have no memory of their own and are refused with them.)
inline bool forward_mode() { return torch::autograd::ForwardADLevel::try_get_by_idx(0) != nullptr; }  // (no tangents outside of a level)
inline bool wrapped(const Tensor& t) {
    return t.defined() && (t.key_set().has(c10::DispatchKey::FuncTorchBatched) || t.key_set().has(c10::DispatchKey::FuncTorchGradWrapper));
}
inline void require_plain(std::initializer_list<const Tensor*> ts) {
    const bool tangents = forward_mode();
    for (const Tensor* t : ts) {
        TORCH_CHECK_NOT_IMPLEMENTED(!tangents || !t->defined() || !t->_fw_grad(/*level=*/0).defined(),
                                    "forward-mode derivatives are not implemented for the operators of mambapy_amd");
        TORCH_CHECK(!wrapped(*t), "functorch transforms (vmap, grad, jvp) are not implemented for the operators of mambapy_amd");
    }
}

inline SavedVariable keep(const Tensor& t) { return SavedVariable(t, false); }
inline Tensor grad_as(const Tensor& g, at::ScalarType dt) { return g.defined() ? cast(g, dt) : g; }

template <typename N>
std::shared_ptr<N> make_node(std::initializer_list<const Tensor*> inputs) {
    std::shared_ptr<N> n(new N(), torch::autograd::deleteNode);
    torch::autograd::edge_list edges;
    edges.reserve(inputs.size());
    for (const Tensor* t : inputs) edges.push_back(t->defined() ? torch::autograd::impl::gradient_edge(*t) : torch::autograd::Edge());
    n->set_next_edges(std::move(edges));
    return n;
}

void bind_model(py::module_& m);  // host_model.cpp
void bind_train(py::module_& m);  // host_train.cpp

}  // namespace mpa_host
