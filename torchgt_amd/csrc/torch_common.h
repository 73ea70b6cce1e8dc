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

}  // namespace tgt_torch
