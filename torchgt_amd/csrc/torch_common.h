// What the translation units of the PyTorch-ROCm extension share: error and dtype translation, the current stream and the
// owner of a plan.
#pragma once
#include <torch/library.h>
#include <torch/custom_class.h>
#include <torch/autograd.h>
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/core/DeviceGuard.h>

#include "../../include/torchgt_hip.h"

namespace tgt_torch {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

inline void check(int rc, const char* what) {
    TORCH_CHECK(rc == TGT_OK, what, ": ", tgt_error_string(rc), " (", tgt_last_error(), ")");
}
inline int dtype_code(const Tensor& t) {
    if (t.scalar_type() == at::kFloat) return TGT_DTYPE_F32;
    if (t.scalar_type() == at::kBFloat16) return TGT_DTYPE_BF16;
    TORCH_CHECK(false, "torchgt: unsupported dtype ", t.scalar_type(), " (float32 or bfloat16)");
}
inline void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
inline const void* ptr(const c10::optional<Tensor>& t) { return (t.has_value() && t->defined()) ? t->data_ptr() : nullptr; }
inline void on_gpu(const Tensor& t, const char* op) {
    TORCH_CHECK(t.is_cuda(), op, " needs GPU tensors (there is no CPU implementation)");
}

// Whether an operator has to go through its autograd node: somebody wants gradients, or a tangent comes with the tensor (forward mode is
// refused there; passing the node by would drop the tangent without a word)
struct Wanted {
    bool gradients = false, tangents = false;
    void look(const Tensor& t) {
        gradients = gradients || t.requires_grad();
        tangents = tangents || t._fw_grad(0).defined();
    }
    bool node() const { return tangents || (gradients && at::GradMode::is_enabled()); }
};
// what a kernel reads has to be on the GPU of its first operand: a host pointer or another GPU's is a fault there
inline void same_gpu(const Tensor& t, const Tensor& first, const char* op, const char* name) {
    TORCH_CHECK(t.defined() && t.is_cuda() && t.device() == first.device(), op, ": ", name, " must be on the GPU ", first.device(), " like the other operands");
}

// Owner of a tgt_plan_t: the Python plan object holds one, and so does every autograd node that will need the plan
// in its backward - the plan lives until the last of them lets go.
struct PlanHolder : torch::CustomClassHolder {
    int64_t h;
    explicit PlanHolder(int64_t handle) : h(handle) {}
    ~PlanHolder() override {
        if (h) tgt_plan_destroy(reinterpret_cast<tgt_plan_t*>(h));
    }
    int64_t handle() const { return h; }
};

// the attention entry points take the number of rows from the plan: tensors of another length must not reach them
inline void rows_match_plan(const c10::intrusive_ptr<PlanHolder>& holder, int64_t N, const char* op) {
    int64_t info[16];
    check(tgt_plan_info(reinterpret_cast<const tgt_plan_t*>(holder->h), info), "tgt_plan_info");
    TORCH_CHECK(info[0] == N, op, ": ", N, " rows, but the plan was built for ", info[0], " nodes");
}

// A tensor of the given sizes on `base`'s memory from element `offset` (no dispatch, no autograd view: base is a plain
// buffer made here)
inline Tensor part_of(const Tensor& base, int64_t offset, at::IntArrayRef sizes) {
    auto impl = c10::make_intrusive<c10::TensorImpl>(c10::Storage(base.storage()), base.unsafeGetTensorImpl()->key_set(), base.dtype());
    impl->set_storage_offset(base.storage_offset() + offset);
    impl->set_sizes_contiguous(sizes);
    return Tensor(std::move(impl));
}
inline int64_t rounded(int64_t n) { return (n + 15) / 16 * 16; }      // parameter gradients start on their own 16 elements


// gradient buffers of a list of shapes in one allocation
struct FlatGrads {
    Tensor flat;
    std::vector<Tensor> t;
    FlatGrads(const std::vector<std::vector<int64_t>>& shapes, const at::TensorOptions& opt) {
        int64_t total = 0;
        std::vector<int64_t> off;
        for (const auto& s : shapes) {
            off.push_back(total);
            int64_t n = 1;
            for (int64_t d : s) n *= d;
            total += rounded(n);
        }
        flat = at::empty({total}, opt);
        t.reserve(shapes.size());
        for (size_t i = 0; i < shapes.size(); ++i) t.push_back(part_of(flat, off[i], shapes[i]));
    }
};

}  // namespace tgt_torch
