// The operator's host side in native code: argument checks, schedule cache, allocations, autograd.
//
// A forward + backward of a small problem is host time: through Python (an autograd.Function, a ctypes structure filled field
// by field, size queries) it took 170 us per pass where the three kernels take 21 (B=1, H=4, T=64, d=64).  What Python does in
// flame_amd/stickbreaking_attention/ is done here without the interpreter, and the backward runs on autograd's thread without
// asking for the interpreter lock.  Python's own version remains for torch.compile's tracing and for the per-kernel timer.
#include "sba_torch.h"

#include <ATen/ops/constant_pad_nd.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <ATen/ops/zeros_like.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <torch/csrc/autograd/custom_function.h>

#include <cstdlib>
#include <cstring>
#include <limits>
#include <mutex>
#include <unordered_map>
#include <vector>

namespace sba_torch {
namespace {

constexpr int64_t kMaxHeadDim = 256;

bool env_is_1(const char* name) {
    const char* e = std::getenv(name);
    return e && e[0] == '1' && e[1] == 0;
}

// Settings that Python holds (_lib.set_workspace_budget, _lib.check_gave_up); negative: not set, the environment decides.
std::atomic<double> g_budget{-1.0};
std::atomic<int> g_check_gave_up{-1};

// Whether the forward keeps nothing for the backward, which then recomputes the carries: under SBA_RECOMPUTE_CARRIES=1
// always, otherwise when the tables would exceed the budget (256 MiB unless set).
bool recompute_carries(size_t table_bytes) {
    if (env_is_1("SBA_RECOMPUTE_CARRIES")) return true;
    double budget = g_budget.load(std::memory_order_relaxed);
    if (budget < 0) {
        const char* e = std::getenv("SBA_WORKSPACE_BUDGET_MB");
        budget = (e && *e) ? std::atof(e) * (1 << 20) : 256.0 * (1 << 20);
    }
    return (double)table_bytes > budget;
}

bool gave_up_checked() {
    const int on = g_check_gave_up.load(std::memory_order_relaxed);
    return on >= 0 ? on != 0 : env_is_1("SBA_CHECK_GAVE_UP");
}

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return SBA_DTYPE_F32;
        case at::kBFloat16: return SBA_DTYPE_BF16;
        case at::kHalf: return SBA_DTYPE_F16;
        default: TORCH_CHECK_TYPE(false, "stick-breaking attention supports float32, bfloat16 and float16, got torch.", t);
    }
}

// 16-bit rows of 72, 80, 88 or 96 columns go to the matrix-core kernels as they are (SbaParams::columns)
bool rides_96(const Tensor& t) {
    const int64_t D = t.size(-1);
    return D > 64 && D <= 96 && D % 8 == 0 && t.scalar_type() != at::kFloat && !env_is_1("SBA_FORCE_GENERIC") &&
           !env_is_1("SBA_FORCE_GENERIC_BWD");
}

SbaTensor describe(const Tensor& t) {
    const auto s = t.strides();
    return t.dim() == 4 ? SbaTensor{t.data_ptr(), s[0], s[1], s[2]} : SbaTensor{t.data_ptr(), 0, s[0], s[1]};
}
SbaVector describe_rows(const Tensor& t) {
    const auto s = t.strides();
    return t.dim() == 3 ? SbaVector{t.data_ptr(), s[0], s[1]} : SbaVector{t.data_ptr(), 0, s[0]};
}

SbaParams params_of(const Problem& pr) {
    SbaParams p;
    std::memset(&p, 0, sizeof(p));
    p.struct_size = sizeof(SbaParams);
    p.dtype = dtype_code(pr.q.scalar_type());
    const auto sz = pr.q.sizes();
    const int64_t lead = pr.q.dim() - 3;                 // 1: dense, 0: packed
    p.n_heads = (int32_t)sz[lead];
    p.head_dim = (int32_t)sz[lead + 2];
    if (rides_96(pr.q)) {
        p.columns = p.head_dim;
        p.head_dim = 128;
    }
    p.total_tokens = (int32_t)sz[lead + 1];
    if (pr.plan) {
        p.n_seq = pr.plan->n_docs;
        // the library chooses its kernels from the longest sweep of the launch: the real longest document
        p.seq_len = std::max(pr.plan->max_len, 1);
        const int32_t* base = pr.plan->buffer.data_ptr<int32_t>();
        // a packing can leave the cache while a launch on a stream that did not build it still reads it
        const auto stream = c10::hip::getCurrentHIPStream(pr.q.device().index());
        if (stream.stream() != pr.plan->built_on) c10::hip::HIPCachingAllocator::recordStream(pr.plan->buffer.storage().data_ptr(), stream);
        p.cu_seqlens = base;
        p.schedule = base + pr.plan->schedule_at;
        p.n_schedule = pr.plan->n_jobs;
        p.table_cols = pr.plan->table_cols;
    } else {
        p.n_seq = (int32_t)sz[0];
        p.seq_len = (int32_t)sz[2];
    }
    p.attend_current = pr.attend_current ? 1 : 0;
    p.scale = (float)pr.scale;
    p.q = describe(pr.q);
    p.k = describe(pr.k);
    p.v = describe(pr.v);
    p.stream = stream_of(pr.q);
    return p;
}

Tensor bytes_like(const Tensor& t, size_t n) {
    return at::empty({(int64_t)n}, t.options().dtype(at::kByte));
}

// ---------------------------------------------------------------------------------------------------- packing plans
//
// One plan per cu_seqlens TENSOR and version (the layers of a model that receive the same tensor share one copy to the host),
// device and job order.  A weak reference keeps the tensor's address from being taken by another while its entry exists;
// entries of tensors that are gone leave when the next plan is built, so the cache holds the packings in use plus those that
// died since.
struct CacheKey {
    const void* tensor;
    int device;
    bool operator==(const CacheKey& o) const { return tensor == o.tensor && device == o.device; }
};
struct CacheHash {
    size_t operator()(const CacheKey& k) const { return std::hash<const void*>()(k.tensor) * 31 + k.device; }
};
struct CacheEntry {
    c10::weak_intrusive_ptr<c10::TensorImpl> tensor;
    int64_t version;
    c10::intrusive_ptr<Plan> plan;
};
std::mutex g_plans_mutex;
std::unordered_map<CacheKey, CacheEntry, CacheHash> g_plans;

c10::intrusive_ptr<Plan> build_plan(const Tensor& cu_seqlens, int64_t n_heads, c10::Device device) {
    // the copy waits for the stream: the program's other threads go on meanwhile
    std::optional<py::gil_scoped_release> unlocked;
    if (PyGILState_Check()) unlocked.emplace();
    // one copy to the host per new packing (none for a tensor that lives there)
    const Tensor host = cu_seqlens.detach().to(at::kCPU, at::kInt).contiguous();
    TORCH_CHECK_VALUE(host.dim() == 1 && host.numel() >= 2 && host.data_ptr<int32_t>()[0] == 0,
                      "cu_seqlens must be 1-D, start with 0 and hold at least one document");
    const int32_t* cu = host.data_ptr<int32_t>();
    auto plan = c10::make_intrusive<Plan>();
    plan->n_docs = (int)host.numel() - 1;
    for (int i = 0; i < plan->n_docs; ++i) {
        TORCH_CHECK_VALUE(cu[i + 1] >= cu[i], "cu_seqlens must be non-decreasing");
        plan->max_len = std::max(plan->max_len, cu[i + 1] - cu[i]);
    }
    plan->total = cu[plan->n_docs];
    plan->table_cols = sba_table_columns(cu, plan->n_docs);
    plan->n_jobs = sba_build_schedule(cu, plan->n_docs, (int)n_heads, nullptr, 0);
    plan->doc_major = plan->n_jobs * n_heads >= SBA_DOC_MAJOR_GRID;
    plan->schedule_at = (host.numel() + 7) & ~int64_t(7);       // rows of 32 bytes
    Tensor all = at::empty({plan->schedule_at + (int64_t)SBA_SCHEDULE_INTS * std::max(plan->n_jobs, 1)}, host.options());
    int32_t* out = all.data_ptr<int32_t>();
    std::memcpy(out, cu, host.numel() * sizeof(int32_t));
    const int got = sba_build_schedule(cu, plan->n_docs, (int)n_heads, out + plan->schedule_at, plan->n_jobs);
    TORCH_INTERNAL_ASSERT(got == plan->n_jobs);
    plan->buffer = all.to(device);
    if (device.is_cuda()) plan->built_on = stream_of(plan->buffer);
    return plan;
}

}  // namespace

hipStream_t stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

void check_status(int rc, const char* what) {
    TORCH_CHECK(rc == 0, what, " failed: ", sba_error_string(rc), " (code ", rc, ")");
}

c10::intrusive_ptr<Plan> plan_for(const Tensor& cu_seqlens, int64_t n_heads, c10::Device device) {
    // an inference tensor does not say whether it was written to since: nothing is kept for it
    if (cu_seqlens.is_inference()) return build_plan(cu_seqlens, n_heads, device);
    const CacheKey key{cu_seqlens.unsafeGetTensorImpl(), device.index()};
    const int64_t version = (int64_t)cu_seqlens._version();
    {
        std::lock_guard<std::mutex> lock(g_plans_mutex);
        auto it = g_plans.find(key);
        if (it != g_plans.end() && it->second.version == version && !it->second.tensor.expired()) {
            const auto& plan = it->second.plan;
            if ((plan->n_jobs * n_heads >= SBA_DOC_MAJOR_GRID) == plan->doc_major) return plan;
        }
    }
    auto plan = build_plan(cu_seqlens, n_heads, device);
    std::lock_guard<std::mutex> lock(g_plans_mutex);
    for (auto it = g_plans.begin(); it != g_plans.end();) it = it->second.tensor.expired() ? g_plans.erase(it) : std::next(it);
    CacheEntry entry{c10::weak_intrusive_ptr<c10::TensorImpl>(cu_seqlens.getIntrusivePtr()), version, plan};
    g_plans.insert_or_assign(key, std::move(entry));
    return plan;
}

void check_plan(const Plan& plan, int64_t tokens, int64_t max_seqlens) {
    TORCH_CHECK_VALUE(plan.total == tokens, "cu_seqlens ends at ", plan.total, " but q has ", tokens, " tokens");
    TORCH_CHECK_VALUE(plan.max_len <= max_seqlens, "max_seqlens=", max_seqlens, " is smaller than the longest document (",
                      plan.max_len, ")");
}

// Head dim that a problem's tensors are handed over with: 64, 128 and (16-bit types) 72 .. 96 and 256 have matrix-core kernels,
// others ride them zero-padded; float32 above 128 and everything under SBA_FORCE_GENERIC=1 keeps its own.
int64_t matrix_core_head_dim(const Tensor& t) {
    const int64_t D = t.size(-1);
    if (D == 64 || D == 128 || D > kMaxHeadDim || rides_96(t) || env_is_1("SBA_FORCE_GENERIC")) return D;
    if (D > 128) return t.scalar_type() == at::kFloat ? D : 256;
    return D < 64 ? 64 : 128;
}

Tensor ready(const Tensor& t, int64_t head_dim) {
    if (t.size(-1) != head_dim) return at::constant_pad_nd(t, {0, head_dim - t.size(-1)});
    bool ok = t.stride(-1) == 1 && ((uintptr_t)t.data_ptr() & 15) == 0;
    const int64_t per16 = 16 / t.element_size() - 1;
    for (int64_t i = 0; ok && i + 1 < t.dim(); ++i) ok = (t.stride(i) & per16) == 0;
    return ok ? t : t.contiguous();
}

Tensor attention_forward(const Problem& pr, const Tensor& o, const Tensor& rem, bool save) {
    SbaParams p = params_of(pr);
    p.o = describe(o);
    p.rem = describe_rows(rem);
    Tensor tables;
    if (save) {
        size_t n = std::max<size_t>(sba_workspace_bytes(&p), 16);
        p.save_for_backward = 1;
        if (recompute_carries(n)) {
            // half of it, where the backward makes the other half (its dQ pass takes 5 % longer; a sweep for the carries alone would
            // take half of a forward)
            p.save_for_backward = SBA_SAVE_ONE_TABLE;
            const size_t half = std::max<size_t>(sba_workspace_bytes(&p), 16);
            if (half >= n || recompute_carries(half)) p.save_for_backward = 0;
            n = half;
        }
        if (p.save_for_backward) {
            tables = bytes_like(pr.q, n);
            p.workspace = tables.data_ptr();
            p.workspace_bytes = n;
        }
    }
    check_status(sba_fwd(&p), "sba_fwd");
    return tables;
}

void attention_backward(const Problem& pr, const Tensor& tables, const Tensor& d_o, const Tensor& d_rem, const Tensor& dq,
                        const Tensor& dk, const Tensor& dv) {
    SbaParams p = params_of(pr);
    p.d_o = describe(d_o);
    if (d_rem.defined()) p.d_rem = describe_rows(d_rem);
    p.dq = describe(dq);
    p.dk = describe(dk);
    p.dv = describe(dv);
    if (tables.defined() && tables.numel() > 16) {
        if ((size_t)tables.numel() < sba_workspace_bytes(&p)) p.save_for_backward = SBA_SAVE_ONE_TABLE;
        p.workspace = tables.data_ptr();
        p.workspace_bytes = tables.numel();
    }
    // freed when this call returns: only the forward's tables live from one direction to the other
    const size_t n = std::max<size_t>(sba_bwd_scratch_bytes(&p), 16);
    const Tensor scratch = bytes_like(pr.q, n);
    p.bwd_scratch = scratch.data_ptr();
    p.bwd_scratch_bytes = n;
    check_status(sba_bwd(&p), "sba_bwd");
    if (gave_up_checked() && c10::hip::currentStreamCaptureStatusMayInitCtx() == c10::hip::CaptureStatus::None) {
        int flag = 0;
        check_status(sba_bwd_gave_up(&p, 0, &flag), "sba_bwd_gave_up");
        TORCH_CHECK(flag == 0, "stick-breaking attention backward: a kernel abandoned a bounded internal wait (error word "
                               "set); the gradients of this call are invalid");
    }
}

namespace {

// Uninitialised dq, dk, dv.  When q, k and v are the three column slices of one dense [.., 3*H*D] tensor (a stacked
// projection's output), the gradients are laid out the same way in ONE allocation, so that the caller's backward can hand the
// whole of it to the projection without concatenating.
std::array<Tensor, 3> empty_grads_like(const Tensor& q, const Tensor& k, const Tensor& v) {
    const int64_t step = k.storage_offset() - q.storage_offset(), n = q.numel();
    if (step > 0 && v.storage_offset() - k.storage_offset() == step && q.sizes() == k.sizes() && k.sizes() == v.sizes() &&
        q.strides() == k.strides() && k.strides() == v.strides() && q.storage().data() == k.storage().data() &&
        q.storage().data() == v.storage().data() && n > 0 && q.stride(-1) == 1) {
        int64_t span = 1;                                // elements from q's first to its last
        for (int64_t i = 0; i < q.dim(); ++i) span += (q.size(i) - 1) * q.stride(i);
        if (span + 2 * step == 3 * n) {
            const Tensor all = at::empty({3 * n}, q.options());
            return {all.as_strided(q.sizes(), q.strides(), 0), all.as_strided(q.sizes(), q.strides(), step),
                    all.as_strided(q.sizes(), q.strides(), 2 * step)};
        }
    }
    return {at::empty_like(q), at::empty_like(k), at::empty_like(v)};
}

Tensor cut(const Tensor& t, int64_t D) { return t.size(-1) == D ? t : t.narrow(-1, 0, D).contiguous(); }

struct Attention : torch::autograd::Function<Attention> {
    static torch::autograd::variable_list forward(torch::autograd::AutogradContext* ctx, const Tensor& q, const Tensor& k,
                                                  const Tensor& v, const std::optional<Tensor>& cu_seqlens,
                                                  c10::intrusive_ptr<Plan> plan, double scale, bool attend_current) {
        const int64_t D = q.size(-1), Dp = matrix_core_head_dim(q);
        Problem pr{ready(q, Dp), ready(k, Dp), ready(v, Dp), plan, scale, attend_current};
        Tensor o = at::empty_like(pr.q);
        Tensor rem = at::empty(pr.q.sizes().slice(0, pr.q.dim() - 1), pr.q.options());
        Tensor tables = attention_forward(pr, o, rem, true);
        ctx->save_for_backward({pr.q, pr.k, pr.v, tables, cu_seqlens ? *cu_seqlens : Tensor()});
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["options"] = (int64_t)(D * 2 + (attend_current ? 1 : 0));
        if (plan) ctx->saved_data["plan"] = c10::IValue::make_capsule(plan);
        ctx->set_materialize_grads(false);
        return {cut(o, D), rem};
    }

    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx,
                                                   torch::autograd::variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const int64_t options = ctx->saved_data["options"].toInt(), D = options / 2;
        Problem pr{saved[0], saved[1], saved[2], {}, ctx->saved_data["scale"].toDouble(), (options & 1) != 0};
        const auto plan = ctx->saved_data.find("plan");
        if (plan != ctx->saved_data.end()) pr.plan = c10::static_intrusive_pointer_cast<Plan>(plan->second.toCapsule());
        c10::DeviceGuard guard(pr.q.device());
        const Tensor d_o = grads[0].defined() ? ready(grads[0], pr.q.size(-1)) : at::zeros_like(pr.q);
        const Tensor d_rem = grads[1].defined() ? grads[1].contiguous() : Tensor();
        auto g = empty_grads_like(pr.q, pr.k, pr.v);
        attention_backward(pr, saved[3], d_o, d_rem, g[0], g[1], g[2]);
        return {cut(g[0], D), cut(g[1], D), cut(g[2], D), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

std::tuple<Tensor, Tensor> run(const Tensor& q, const Tensor& k, const Tensor& v, const std::optional<Tensor>& cu_seqlens,
                               int64_t max_seqlens, double scale, bool attend_current) {
    if (q.numel() == 0) return {q * 0, q.sum(-1) * 0};      // nothing to launch: empty results that stay in the graph
    TORCH_CHECK(q.is_cuda(), "stick-breaking attention runs on the GPU only (HIP kernels); there is no CPU path");
    TORCH_CHECK_TYPE(q.scalar_type() == k.scalar_type() && k.scalar_type() == v.scalar_type(), "q, k, v must share a dtype");
    TORCH_CHECK_VALUE(q.device() == k.device() && k.device() == v.device(), "q, k, v must be on the same device");
    TORCH_CHECK_VALUE(q.sizes() == k.sizes() && k.sizes() == v.sizes() && q.dim() == (cu_seqlens ? 3 : 4),
                      cu_seqlens ? "q, k, v must all be [H, total_tokens, D]" : "q, k, v must all be [B, H, T, D]");
    dtype_code(q.scalar_type());
    TORCH_CHECK_VALUE(q.size(-1) <= kMaxHeadDim, "head_dim ", q.size(-1), " is not supported (at most ", kMaxHeadDim, ")");
    TORCH_CHECK_NOT_IMPLEMENTED(!has_tangent(q) && !has_tangent(k) && !has_tangent(v),
                                "stick-breaking attention has no forward-mode derivative");
    c10::DeviceGuard guard(q.device());
    c10::intrusive_ptr<Plan> plan;
    if (cu_seqlens) {
        plan = plan_for(*cu_seqlens, q.size(0), q.device());
        check_plan(*plan, q.size(1), max_seqlens);
    }
    const bool train = at::GradMode::is_enabled() && (q.requires_grad() || k.requires_grad() || v.requires_grad());
    if (train) {
        auto out = Attention::apply(q, k, v, cu_seqlens, plan, scale, attend_current);
        return {out[0], out[1]};
    }
    // no backward can follow: nothing is kept
    at::AutoDispatchBelowADInplaceOrView below;
    const int64_t D = q.size(-1), Dp = matrix_core_head_dim(q);
    Problem pr{ready(q, Dp), ready(k, Dp), ready(v, Dp), plan, scale, attend_current};
    Tensor o = at::empty_like(pr.q);
    Tensor rem = at::empty(pr.q.sizes().slice(0, pr.q.dim() - 1), pr.q.options());
    attention_forward(pr, o, rem, false);
    return {cut(o, D), rem};
}

double scale_or_default(const std::optional<double>& inv_temp, const Tensor& q) {
    return inv_temp ? *inv_temp : 1.0 / std::sqrt((double)q.size(-1));
}

}  // namespace
}  // namespace sba_torch

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    using namespace sba_torch;
    m.def("attention", [](const Tensor& q, const Tensor& k, const Tensor& v, std::optional<double> inv_temp, bool attend_current) {
        return run(q, k, v, std::nullopt, 0, scale_or_default(inv_temp, q), attend_current);
    });
    m.def("attention_varlen", [](const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& cu_seqlens, int64_t max_seqlens,
                                 std::optional<double> inv_temp, bool attend_current) {
        return run(q, k, v, cu_seqlens, max_seqlens, scale_or_default(inv_temp, q), attend_current);
    });
    bind_model(m);
    m.def("set_workspace_budget", [](double bytes) { g_budget = bytes; });
    m.def("set_check_gave_up", [](int on) { g_check_gave_up = on; });
}
