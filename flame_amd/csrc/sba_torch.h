// Shared by the native host layer's sources (sba_torch*.cpp): the attention operator on tensors, below autograd.
#pragma once
#include <torch/extension.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>

#include "../../include/sba_mi355x.h"

namespace sba_torch {

using at::Tensor;

// What the kernels need of one packing (a cu_seqlens tensor): its row-block schedule and its sizes.  Built once per tensor and
// kept by plan_for(); a backward holds the one its forward used.
struct Plan : torch::CustomClassHolder {
    Tensor buffer;                       // int32 on the device: cu_seqlens (leading 0), then the schedule
    hipStream_t built_on = nullptr;      // the stream that `buffer` belongs to
    int64_t schedule_at = 0;             // first schedule int in `buffer`
    int n_docs = 0, n_jobs = 0, max_len = 0, total = 0;
    int64_t table_cols = 0;
    bool doc_major = false;
};

// One attention problem.  q, k, v: [B, H, T, D] or, with a plan, [H, N, D]; already of a head dim and of strides that the
// kernels take (see ready()).
struct Problem {
    Tensor q, k, v;
    c10::intrusive_ptr<Plan> plan;       // empty: dense
    double scale = 1.0;
    bool attend_current = false;
};

c10::intrusive_ptr<Plan> plan_for(const Tensor& cu_seqlens, int64_t n_heads, c10::Device device);
void check_plan(const Plan& plan, int64_t tokens, int64_t max_seqlens);

int64_t matrix_core_head_dim(const Tensor& t);
Tensor ready(const Tensor& t, int64_t head_dim);        // padded to `head_dim`, strides the kernels take

// o and rem are written; the result is the carry tables to hand to attention_backward() (undefined: nothing was kept).
Tensor attention_forward(const Problem& pr, const Tensor& o, const Tensor& rem, bool save);
void attention_backward(const Problem& pr, const Tensor& tables, const Tensor& d_o, const Tensor& d_rem, const Tensor& dq,
                        const Tensor& dk, const Tensor& dv);

void bind_model(py::module& m);          // sba_torch_model.cpp

// A dual tensor of forward-mode differentiation: the nodes here have no such derivative, and the kernels would drop it silently.
inline bool has_tangent(const Tensor& t) { return t._fw_grad(/*level=*/0).defined(); }

hipStream_t stream_of(const Tensor& t);
void check_status(int rc, const char* what);

}  // namespace sba_torch
