// The language model's blocks as autograd nodes of their own: one node per transformer block instead of about forty framework
// operators, so that a block costs the host a dozen launches in each direction, the elementwise work around the matrix products
// runs in fused kernels (sba_model.hip), and the weights' gradients come out of their products in fp32.
//
// What a block computes is flame_amd/modeling_sba.py's SBABlock under autocast: fp32 weights and residual stream, 16-bit
// operands of every product, fp32 normalisation.
#include "sba_model.h"
#include "sba_torch.h"

#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <ATen/ops/mm.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/util/SmallVector.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>

#include <cstring>

namespace sba_torch {
namespace {

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;
using namespace sba_model;

void ok(int rc) { check_status(rc, "model kernel"); }
bool is_f16(at::ScalarType t) { return t == at::kHalf; }

// a 16-bit tensor of a caller's: dense, and from a 16-byte boundary on, as the kernels' loads of eight elements are meant to be
Tensor aligned(const Tensor& t) {
    const Tensor c = t.contiguous();
    return (uintptr_t)c.data_ptr() & 15 ? c.clone() : c;
}

Tensor empty(at::IntArrayRef sizes, const Tensor& like, at::ScalarType t) { return at::empty(sizes, like.options().dtype(t)); }

// fp32 weights as 16-bit ones, stacked along their rows in one buffer each; `groups` says how many weights share a buffer
std::vector<Tensor> cast_weights(at::ArrayRef<Tensor> w, at::IntArrayRef groups, at::ScalarType t) {
    CastList list = {};
    int64_t total = 0;
    for (const auto& x : w) {
        list.src[list.n] = x.data_ptr<float>();
        total += x.numel();
        list.end[list.n++] = total;
    }
    Tensor all = empty({total}, w[0], t);
    ok(cast_list(list, all.data_ptr(), is_f16(t), stream_of(all)));
    std::vector<Tensor> out;
    int64_t at = 0;
    int i = 0;
    for (int64_t g : groups) {
        int64_t rows = 0;
        const int64_t cols = w[i].size(1);
        for (int64_t j = 0; j < g; ++j) rows += w[i++].size(0);
        out.push_back(all.narrow(0, at, rows * cols).view({rows, cols}));
        at += rows * cols;
    }
    return out;
}

int compute_units() {
    static const int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess) n = 256;
        return n > 0 ? n : 256;
    }();
    return cus;
}

void check_on_gpu(const Tensor& x) { TORCH_CHECK_VALUE(x.is_cuda(), "the model's kernels run on the GPU only"); }

// d_weight = d_out^T . in, in fp32, of several products over the same rows at once
std::vector<Tensor> weight_grads(at::ArrayRef<std::pair<Tensor, Tensor>> pairs) {
    WeightGrads g = {};
    for (const auto& [d_out, in] : pairs) {
        auto& one = g.one[g.n++];
        one.a = d_out.data_ptr();
        one.b = in.data_ptr();
        one.lda = d_out.size(0) > 1 ? d_out.stride(0) : d_out.size(1);
        one.ldb = in.size(0) > 1 ? in.stride(0) : in.size(1);
        one.m = (int)d_out.size(1);
        one.n = (int)in.size(1);
        g.k = (int)in.size(0);
    }
    const Tensor& like = pairs[0].first;
    ok(weight_grads_fit(g) ? 0 : SBA_ERR_SHAPE);
    check_on_gpu(like);
    const int splits = weight_grad_splits(g, compute_units());
    const Tensor out = empty({g.total}, like, at::kFloat);
    Tensor partial;
    g.out = out.data_ptr<float>();
    if (splits > 1) {
        partial = empty({splits, g.total}, like, at::kFloat);
        g.partial = partial.data_ptr<float>();
    }
    ok(sba_model::weight_grads(g, splits, is_f16(like.scalar_type()), stream_of(like)));
    std::vector<Tensor> r;
    for (int i = 0; i < g.n; ++i)
        r.push_back(out.narrow(0, g.one[i].at, (int64_t)g.one[i].m * g.one[i].n).view({g.one[i].m, g.one[i].n}));
    return r;
}

struct Norm { Tensor y, rstd; };
Norm rms_norm(const Tensor& x, const Tensor& w, double eps, at::ScalarType t) {
    Norm r;
    const int64_t rows = x.size(0), cols = x.size(1);
    r.y = empty({rows, cols}, x, t);
    r.rstd = empty({rows}, x, at::kFloat);
    NormFwd a = {};
    a.x = x.data_ptr<float>();
    a.w = w.data_ptr<float>();
    a.y = r.y.data_ptr();
    a.rstd = r.rstd.data_ptr<float>();
    a.rows = (int)rows;
    a.cols = (int)cols;
    a.eps = (float)eps;
    ok(norm_fwd(a, is_f16(t), stream_of(x)));
    return r;
}

struct NormGrad { Tensor dx, dx16, part; };
// (the gradient of the weight is what norm_weight_grads() makes of `part`)
NormGrad rms_norm_grad(const Tensor& dy, const Tensor& x, const Tensor& w, const Tensor& rstd, const Tensor& dres, bool want16) {
    NormGrad r;
    const int64_t rows = x.size(0), cols = x.size(1);
    const int parts = norm_bwd_parts((int)rows);
    r.part = empty({parts, cols}, x, at::kFloat);
    r.dx = at::empty_like(x);
    NormBwd a = {};
    a.dy = dy.data_ptr();
    a.x = x.data_ptr<float>();
    a.w = w.data_ptr<float>();
    a.rstd = rstd.data_ptr<float>();
    a.dres = dres.defined() ? dres.data_ptr<float>() : nullptr;
    a.dx = r.dx.data_ptr<float>();
    if (want16) {
        r.dx16 = empty({rows, cols}, x, dy.scalar_type());
        a.dx16 = r.dx16.data_ptr();
    }
    a.dw_part = r.part.data_ptr<float>();
    a.rows = (int)rows;
    a.cols = (int)cols;
    ok(norm_bwd(a, is_f16(dy.scalar_type()), stream_of(x)));
    return r;
}

// out[i] = the gradient of weight[i] for each defined part, both in one launch (a launch of its own each is 5 us of a block's step)
void norm_weight_grads(const Tensor (&part)[2], const Tensor (&weight)[2], Tensor* const (&out)[2]) {
    const float* from[2] = {};
    float* to[2] = {};
    int n = 0, last = 0;
    for (int i = 0; i < 2; ++i) {
        if (!part[i].defined()) continue;
        *out[i] = at::empty_like(weight[i]);
        from[n] = part[i].data_ptr<float>();
        to[n++] = out[i]->data_ptr<float>();
        last = i;
    }
    if (n) ok(sum_parts(from, to, n, (int)part[last].size(0), (int)part[last].size(1), stream_of(part[last])));
}

Projection projection_of(const Tensor& x, const Tensor& w, bool rows_w, int epilogue, const Tensor& residual, const Tensor& pre, const Tensor& out) {
    Projection p = {};
    p.x = x.data_ptr();
    p.w = w.data_ptr();
    p.ldx = x.stride(0);
    p.ldw = w.stride(0);
    p.m = (int)x.size(0);
    p.k = (int)x.size(1);
    p.n = (int)w.size(rows_w ? 1 : 0);
    p.rows_w = rows_w;
    p.epilogue = epilogue;
    if (residual.defined()) p.residual = residual.data_ptr<float>();
    if (pre.defined()) p.pre = pre.data_ptr();
    p.out = out.data_ptr();
    return p;
}

// y = x w^T (rows_w: x w) into `out`, with what sba_model.h's epilogues do on the way; false where the kernels do not take it
bool try_project(const Tensor& x, const Tensor& w, bool rows_w, int epilogue, const Tensor& residual, const Tensor& pre, const Tensor& out) {
    Projection p = projection_of(x, w, rows_w, epilogue, residual, pre, out);
    if (!projects(p, compute_units())) return false;
    ProjectionTile tile;
    p.splits = projection_splits(p, compute_units(), tile);
    Tensor partial;
    if (p.splits > 1) {
        partial = empty({p.splits, p.m, p.n}, x, at::kFloat);
        p.partial = partial.data_ptr<float>();
    }
    ok(project_tile(p, tile, is_f16(x.scalar_type()), stream_of(x)));
    return true;
}

// What the kernels take for granted and the nodes see to before they call: the entries by themselves check it.
void check_operands(const Tensor& x, const Tensor& w, bool rows_w) {
    const auto t = x.scalar_type();
    TORCH_CHECK_TYPE((t == at::kBFloat16 || t == at::kHalf) && w.scalar_type() == t, "x and w must both be bfloat16 or both float16");
    TORCH_CHECK_VALUE(x.dim() == 2 && w.dim() == 2 && x.size(1) == w.size(rows_w ? 0 : 1), "x and w must be matrices that share k");
    TORCH_CHECK_VALUE(x.stride(1) == 1 && w.stride(1) == 1 && (x.size(0) < 2 || x.stride(0) >= x.size(1)) && (w.size(0) < 2 || w.stride(0) >= w.size(1)), "rows of x and w must be dense");
    TORCH_CHECK_VALUE(x.device() == w.device(), "x and w must be on the same device");
}
void check_dense(const Tensor& t, at::IntArrayRef sizes, at::ScalarType type, const Tensor& like, const char* name) {
    TORCH_CHECK_VALUE(t.defined() && t.sizes() == sizes && t.is_contiguous() && t.device() == like.device() && ((uintptr_t)t.data_ptr() & 15) == 0,
                      name, " must be a dense tensor of shape ", sizes, " on 16 bytes beside x");
    TORCH_CHECK_TYPE(t.scalar_type() == type, name, " must be ", type);
}
// The same with the tile of a caller's choice, where that tile's kernel takes the problem (tests of kernels that the rule picks elsewhere).
bool project_with(int64_t tile, const Tensor& x, const Tensor& w, bool rows_w, int64_t epilogue, const std::optional<Tensor>& residual,
                  const std::optional<Tensor>& pre, const Tensor& out, int64_t splits) {
    TORCH_CHECK(tile >= kTile256 && tile <= kTile64Halves && epilogue >= kStore && epilogue <= kSwigluBwd && splits >= 1, "project_with: no such tile, epilogue or share");
    check_operands(x, w, rows_w);
    const int64_t m = x.size(0), n = w.size(rows_w ? 1 : 0);
    const auto t = x.scalar_type();
    check_dense(out, {m, epilogue == kSwigluFwd ? n / 2 : epilogue == kSwigluBwd ? 2 * n : n}, epilogue == kAddResidual ? at::kFloat : t, x, "out");
    if (epilogue == kAddResidual) check_dense(residual.value_or(Tensor()), {m, n}, at::kFloat, x, "residual");
    if (epilogue == kSwigluBwd || (epilogue == kSwigluFwd && pre)) check_dense(pre.value_or(Tensor()), {m, epilogue == kSwigluBwd ? 2 * n : n}, t, x, "pre");
    check_on_gpu(x);
    c10::DeviceGuard guard(x.device());
    Projection p = projection_of(x, w, rows_w, (int)epilogue, residual.value_or(Tensor()), pre.value_or(Tensor()), out);
    TORCH_CHECK(addresses(p), "project_with: sizes or places that no tile takes");
    if (tile_time(p, (ProjectionTile)tile, compute_units()) >= 1e30) return false;
    Tensor partial;
    if (splits > 1) {
        const int64_t stages = p.k / 64, per = (stages + splits - 1) / splits;
        TORCH_CHECK(tile <= kTile128x256 && rows_w && epilogue == kStore && (splits - 1) * per < stages, "project_with: not shared out");
        partial = empty({splits, p.m, p.n}, x, at::kFloat);
        p.splits = (int)splits;
        p.partial = partial.data_ptr<float>();
    }
    ok(project_tile(p, (ProjectionTile)tile, is_f16(x.scalar_type()), stream_of(x)));
    return true;
}

// x w^T for w [n][k], x w for w [k][n]: 16-bit
Tensor project(const Tensor& x, const Tensor& w, bool rows_w) {
    Tensor out = empty({x.size(0), w.size(rows_w ? 1 : 0)}, x, x.scalar_type());
    if (!try_project(x, w, rows_w, kStore, Tensor(), Tensor(), out)) at::mm_out(out, x, rows_w ? w : w.t());
    return out;
}

// residual + x w^T: fp32, and the product's sum is not rounded to 16 bits before it is added, whichever way it is formed
Tensor project_add(const Tensor& x, const Tensor& w, const Tensor& residual) {
    Tensor out = at::empty_like(residual);
    // what the kernels do not take, contractions off 32 above all: 8192 x 1024, k = 2728 74 us, 71 with a 16-bit product and a pass
    // that adds; 84 with operands padded by zeros to 32 for the kernel, 89 with the last 8 of k in a product of their own
    if (!try_project(x, w, false, kAddResidual, residual, Tensor(), out)) return at::mm(x, w.t(), at::kFloat).add_(residual);
    return out;
}

// silu(x gate^T) * (x up^T) for w = gate rows | up rows; `pre`, if defined, receives the two products
Tensor project_swiglu(const Tensor& x, const Tensor& w, Tensor& pre, bool keep) {
    const int64_t rows = x.size(0), width = w.size(0) / 2;
    Tensor out = empty({rows, width}, x, x.scalar_type());
    if (keep) pre = empty({rows, 2 * width}, x, x.scalar_type());
    if (!try_project(x, w, false, kSwigluFwd, Tensor(), pre, out)) {
        pre = project(x, w, false);
        ok(swiglu_fwd(pre.data_ptr(), out.data_ptr(), rows, (int)width, is_f16(x.scalar_type()), stream_of(x)));
    }
    return out;
}

// the gradient of gate | up from d, the gradient of what silu(gate) * up was multiplied with: d w, then through the product
Tensor project_swiglu_grad(const Tensor& d, const Tensor& w, const Tensor& pre) {
    Tensor out = at::empty_like(pre);
    if (!try_project(d, w, true, kSwigluBwd, Tensor(), pre, out)) {
        const Tensor da = project(d, w, true);
        ok(swiglu_bwd(pre.data_ptr(), da.data_ptr(), out.data_ptr(), d.size(0), (int)w.size(1), is_f16(d.scalar_type()), stream_of(d)));
    }
    return out;
}

Tensor cast_to(const Tensor& x, at::ScalarType t) {
    Tensor out = empty(x.sizes(), x, t);
    ok(cast_one(x.data_ptr<float>(), out.data_ptr(), x.numel(), is_f16(t), stream_of(x)));
    return out;
}

// What a backward of these kernels returns under create_graph: its gradients, which say so if they are differentiated again (the
// kernels leave no graph, so they would pass for constants).
template <class F>
variable_list differentiable_once(const variable_list& in, F&& backward) {
    const bool graph = at::GradMode::is_enabled();
    variable_list grads;
    {
        at::AutoGradMode no_graph(false);
        grads = backward();
    }
    if (!graph) return grads;
    // they depend on what the node's inputs and its incoming gradients do
    torch::autograd::edge_list edges;
    if (const auto node = torch::autograd::get_current_node()) edges = node->next_edges();
    for (auto& e : torch::autograd::collect_next_edges(in)) edges.push_back(std::move(e));
    const auto error = std::make_shared<torch::autograd::Error>(
        "the language model's native nodes differentiate once: their gradients cannot be differentiated again", std::move(edges));
    for (auto& g : grads) {
        if (!g.defined()) continue;
        g = g.detach();
        torch::autograd::set_history(g, error);
    }
    return grads;
}

// -------------------------------------------------------------------------------------------------------- one block

struct BlockShape {
    int64_t B, T, hidden, heads, width;
    double eps1, eps2, scale;
    at::ScalarType t;
    c10::intrusive_ptr<Plan> plan;
};

// the three column slices of a [B*T, 3*hidden] product as the operator's q, k, v
Problem problem_of(const BlockShape& s, const Tensor& qkv) {
    const int64_t D = s.hidden / s.heads, row = 3 * s.hidden;
    auto view = [&](int64_t i) {
        return s.plan ? qkv.as_strided({s.heads, s.T, D}, {D, row, 1}, qkv.storage_offset() + i * s.hidden)
                      : qkv.as_strided({s.B, s.heads, s.T, D}, {s.T * row, D, row, 1}, qkv.storage_offset() + i * s.hidden);
    };
    return Problem{view(0), view(1), view(2), s.plan, s.scale, false};
}
// a dense [B*T, hidden] tensor as the operator's o
Tensor heads_of(const BlockShape& s, const Tensor& o) {
    const int64_t D = s.hidden / s.heads;
    return s.plan ? o.as_strided({s.heads, s.T, D}, {D, s.hidden, 1})
                  : o.as_strided({s.B, s.heads, s.T, D}, {s.T * s.hidden, D, s.hidden, 1});
}

// the operands have their types already: nothing for autocast to look at
struct NoAutocast {
    c10::impl::ExcludeDispatchKeyGuard guard{c10::DispatchKey::AutocastCUDA};
};

struct BlockState {
    Tensor x1, y1, rstd1, qkv, o, tables, y2, rstd2, gu, a;
    std::vector<Tensor> w;              // 16-bit: q|k|v stacked, o, gate|up stacked, down
};

// weights: norm1, q, k, v, o, norm2, gate, up, down
Tensor block_forward(const BlockShape& s, const Tensor& x, at::ArrayRef<Tensor> weights, bool train, BlockState& st) {
    const Tensor cast[] = {weights[1], weights[2], weights[3], weights[4], weights[6], weights[7], weights[8]};
    st.w = cast_weights(cast, {3, 1, 2, 1}, s.t);
    const int64_t N = s.B * s.T;
    auto n1 = rms_norm(x, weights[0], s.eps1, s.t);
    st.y1 = n1.y;
    st.rstd1 = n1.rstd;
    st.qkv = project(st.y1, st.w[0], false);
    Problem pr = problem_of(s, st.qkv);
    st.o = empty({N, s.hidden}, x, s.t);
    Tensor rem = s.plan ? empty({s.heads, s.T}, x, s.t) : empty({s.B, s.heads, s.T}, x, s.t);
    st.tables = attention_forward(pr, heads_of(s, st.o), rem, train);
    st.x1 = project_add(st.o, st.w[1], x);
    auto n2 = rms_norm(st.x1, weights[5], s.eps2, s.t);
    st.y2 = n2.y;
    st.rstd2 = n2.rstd;
    st.a = project_swiglu(st.y2, st.w[2], st.gu, train);
    return project_add(st.a, st.w[3], st.x1);
}

struct Block : torch::autograd::Function<Block> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& n1, const Tensor& wq, const Tensor& wk,
                          const Tensor& wv, const Tensor& wo, const Tensor& n2, const Tensor& wg, const Tensor& wu,
                          const Tensor& wd, const std::optional<Tensor>& cu_seqlens, const BlockShape& s) {
        const Tensor x = x_in.contiguous().view({s.B * s.T, s.hidden});
        BlockState st;
        const Tensor weights[] = {n1, wq, wk, wv, wo, n2, wg, wu, wd};
        Tensor out = block_forward(s, x, weights, true, st);
        ctx->save_for_backward({x, n1, n2, st.x1, st.y1, st.rstd1, st.qkv, st.o, st.tables, st.y2, st.rstd2, st.gu, st.a, st.w[0],
                                st.w[1], st.w[2], st.w[3], cu_seqlens ? *cu_seqlens : Tensor()});
        ctx->saved_data["scale"] = s.scale;
        ctx->saved_data["sizes"] = std::vector<int64_t>{s.B, s.T, s.hidden, s.heads, s.width};
        if (s.plan) ctx->saved_data["plan"] = c10::IValue::make_capsule(s.plan);
        return out.view(x_in.sizes());
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        return differentiable_once(grads, [&] { return gradients(ctx, grads); });
    }

    static variable_list gradients(AutogradContext* ctx, const variable_list& grads) {
        const auto sv = ctx->get_saved_variables();
        const Tensor &x = sv[0], &n1 = sv[1], &n2 = sv[2], &x1 = sv[3], &y1 = sv[4], &rstd1 = sv[5], &qkv = sv[6], &o = sv[7],
                     &tables = sv[8], &y2 = sv[9], &rstd2 = sv[10], &gu = sv[11], &a = sv[12], &w_qkv = sv[13], &w_o = sv[14],
                     &w_gu = sv[15], &w_d = sv[16];
        const auto z = ctx->saved_data["sizes"].toIntVector();
        BlockShape s{z[0], z[1], z[2], z[3], z[4], 0, 0, ctx->saved_data["scale"].toDouble(), qkv.scalar_type(), {}};
        const auto plan = ctx->saved_data.find("plan");
        if (plan != ctx->saved_data.end()) s.plan = c10::static_intrusive_pointer_cast<Plan>(plan->second.toCapsule());
        c10::DeviceGuard guard(x.device());
        const int64_t N = s.B * s.T;
        const Tensor dx2 = grads[0].contiguous().view({N, s.hidden});

        // what is asked for - x, norm1, q, k, v, o, norm2, gate, up, down -, and no further back than that leads
        auto asked = [&](int first, int last) {
            for (int i = first; i <= last; ++i)
                if (ctx->needs_input_grad(i)) return true;
            return false;
        };
        const Tensor dm = cast_to(dx2, s.t);
        Tensor dgu, dqkv, dy1;
        NormGrad g1, g2;
        if (asked(0, 8)) dgu = project_swiglu_grad(dm, w_d, gu);
        if (asked(0, 6)) g2 = rms_norm_grad(project(dgu, w_gu, true), x1, n2, rstd2, dx2, true);
        if (asked(0, 4)) {
            const Tensor d_o = project(g2.dx16, w_o, true);
            dqkv = at::empty_like(qkv);
            Problem pr = problem_of(s, qkv);
            const Problem g = problem_of(s, dqkv);
            attention_backward(pr, tables, heads_of(s, d_o), Tensor(), g.q, g.k, g.v);
        }
        if (asked(0, 1)) dy1 = project(dqkv, w_qkv, true);

        // weights first .. last lie stacked, `rows` of each: from the first asked one to the last
        c10::SmallVector<std::pair<Tensor, Tensor>, 4> products;
        c10::SmallVector<std::array<int64_t, 3>, 4> owners;
        auto want = [&](int first, int last, int64_t rows, const Tensor& d, const Tensor& in) {
            const int stacked = first;
            while (first <= last && !asked(first, first)) ++first;
            while (first < last && !asked(last, last)) --last;
            if (first > last) return;
            products.emplace_back(d.narrow(1, (first - stacked) * rows, (last - first + 1) * rows), in);
            owners.push_back({first, last, rows});
        };
        want(2, 4, s.hidden, dqkv, y1);
        want(5, 5, s.hidden, g2.dx16, o);
        want(7, 8, s.width, dgu, y2);
        want(9, 9, s.hidden, dm, a);
        variable_list out(12);
        if (!products.empty()) {
            const auto dw = weight_grads(products);
            for (size_t i = 0; i < dw.size(); ++i) {
                const auto [first, last, rows] = owners[i];
                for (int64_t w = first; w <= last; ++w)
                    if (asked(w, w)) out[w] = dw[i].narrow(0, (w - first) * rows, rows);
            }
        }
        if (asked(0, 1)) {
            g1 = rms_norm_grad(dy1, x, n1, rstd1, g2.dx, false);
            out[0] = g1.dx.view(grads[0].sizes());
        }
        norm_weight_grads({g1.part, g2.part}, {n1, n2}, {&out[1], &out[6]});
        return out;
    }
};

// block(), head() and next_token_loss() return nothing where the modules have to be called instead: they differentiate forward, too.
std::optional<Tensor> block(const Tensor& x, const std::vector<Tensor>& w, int64_t heads, double eps1, double eps2, py::object dtype,
                            const std::optional<Tensor>& cu_seqlens, int64_t max_seqlens) {
    bool dual = has_tangent(x);
    for (const auto& t : w) dual = dual || has_tangent(t);
    if (dual) return std::nullopt;
    BlockShape s;
    s.B = x.size(0);
    s.T = x.size(1);
    s.hidden = x.size(2);
    s.heads = heads;
    s.width = w[6].size(0);
    s.eps1 = eps1;
    s.eps2 = eps2;
    s.scale = 1.0 / std::sqrt((double)(s.hidden / heads));
    s.t = torch::python::detail::py_object_to_dtype(dtype);
    c10::DeviceGuard guard(x.device());
    NoAutocast no_autocast;
    if (cu_seqlens) {
        s.plan = plan_for(*cu_seqlens, heads, x.device());
        check_plan(*s.plan, s.T, max_seqlens);
    }
    bool train = x.requires_grad();
    for (const auto& t : w) train = train || t.requires_grad();
    if (at::GradMode::is_enabled() && train)
        return Block::apply(x, w[0], w[1], w[2], w[3], w[4], w[5], w[6], w[7], w[8], cu_seqlens, s);
    at::AutoDispatchBelowADInplaceOrView below;
    BlockState st;
    return block_forward(s, x.contiguous().view({s.B * s.T, s.hidden}), w, false, st).view(x.sizes());
}

// ---------------------------------------------------------------------------------- final norm, head and loss

struct Head : torch::autograd::Function<Head> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& n, const Tensor& w, double eps, at::ScalarType t) {
        const Tensor x = x_in.contiguous().view({-1, x_in.size(-1)});
        auto r = rms_norm(x, n, eps, t);
        const Tensor w16 = cast_to(w, t);
        Tensor logits = project(r.y, w16, false);
        ctx->save_for_backward({x, n, r.y, r.rstd, w16});
        auto sizes = x_in.sizes().vec();
        sizes.back() = w.size(0);
        return logits.view(sizes);
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        return differentiable_once(grads, [&] { return gradients(ctx, grads); });
    }
    static variable_list gradients(AutogradContext* ctx, const variable_list& grads) {
        const auto sv = ctx->get_saved_variables();
        c10::DeviceGuard guard(sv[0].device());
        const Tensor d = aligned(grads[0]).view({-1, grads[0].size(-1)});
        variable_list out(5);                                    // x, norm, weight
        if (ctx->needs_input_grad(2)) out[2] = weight_grads({{d, sv[2]}})[0];
        if (ctx->needs_input_grad(0) || ctx->needs_input_grad(1)) {
            auto g = rms_norm_grad(project(d, sv[4], true), sv[0], sv[1], sv[3], Tensor(), false);
            auto sizes = grads[0].sizes().vec();
            sizes.back() = sv[0].size(1);
            out[0] = g.dx.view(sizes);
            norm_weight_grads({g.part, Tensor()}, {sv[1], Tensor()}, {&out[1], &out[1]});
        }
        return out;
    }
};

std::optional<Tensor> head(const Tensor& x, const Tensor& n, const Tensor& w, double eps, py::object dtype) {
    if (has_tangent(x) || has_tangent(n) || has_tangent(w)) return std::nullopt;
    const at::ScalarType t = torch::python::detail::py_object_to_dtype(dtype);
    c10::DeviceGuard guard(x.device());
    NoAutocast no_autocast;
    if (at::GradMode::is_enabled() && (x.requires_grad() || n.requires_grad() || w.requires_grad()))
        return Head::apply(x, n, w, eps, t);
    at::AutoDispatchBelowADInplaceOrView below;
    const Tensor rows = x.contiguous().view({-1, x.size(-1)});
    auto r = rms_norm(rows, n, eps, t);
    auto sizes = x.sizes().vec();
    sizes.back() = w.size(0);
    return project(r.y, cast_to(w, t), false).view(sizes);
}

struct LossRows { Tensor mean, count, lse; };
LossRows loss_rows(const Tensor& logits, const Tensor& labels, int64_t ignore) {
    const int64_t rows = labels.numel();
    LossRows r{empty({}, logits, at::kFloat), empty({}, logits, at::kFloat), empty({2, rows}, logits, at::kFloat)};
    float* lse = r.lse.data_ptr<float>();
    ok(loss_fwd(logits.data_ptr(), labels.data_ptr<int64_t>(), lse, lse + rows, r.mean.data_ptr<float>(), r.count.data_ptr<float>(),
                (int)rows, (int)labels.size(-1), (int)logits.size(-1), ignore, is_f16(logits.scalar_type()), stream_of(logits)));
    return r;
}

// The loss's gradient from operators that leave a graph (create_graph).
Tensor differentiable_loss_grad(const Tensor& logits, const Tensor& labels, const Tensor& count, const Tensor& d_loss, int64_t ignore) {
    const Tensor target = at::cat({labels.narrow(1, 1, labels.size(1) - 1), at::full_like(labels.narrow(1, 0, 1), ignore)}, 1).unsqueeze(-1);
    const Tensor hit = target.eq(at::arange(logits.size(-1), labels.options())).to(at::kFloat);
    const Tensor scale = at::where(target.eq(ignore), at::zeros_like(count), d_loss / count);
    return ((at::softmax(logits.to(at::kFloat), -1) - hit) * scale).to(logits.scalar_type());
}

struct Loss : torch::autograd::Function<Loss> {
    static Tensor forward(AutogradContext* ctx, const Tensor& logits, const Tensor& labels_in, int64_t ignore) {
        const Tensor labels = labels_in.contiguous();
        auto r = loss_rows(aligned(logits), labels, ignore);
        ctx->save_for_backward({logits, labels, r.lse, r.count});
        ctx->saved_data["ignore"] = ignore;
        return r.mean;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const auto sv = ctx->get_saved_variables();
        const Tensor& labels = sv[1];
        c10::DeviceGuard guard(labels.device());
        if (at::GradMode::is_enabled())
            return {differentiable_loss_grad(sv[0], labels, sv[3], grads[0], ctx->saved_data["ignore"].toInt()), Tensor(), Tensor()};
        const Tensor logits = aligned(sv[0]), g = grads[0].contiguous();
        Tensor d = at::empty_like(logits);
        ok(loss_bwd(logits.data_ptr(), labels.data_ptr<int64_t>(), sv[2].data_ptr<float>(), sv[3].data_ptr<float>(),
                    g.data_ptr<float>(), d.data_ptr(), (int)labels.numel(), (int)labels.size(-1), (int)logits.size(-1),
                    ctx->saved_data["ignore"].toInt(), is_f16(logits.scalar_type()), stream_of(logits)));
        return {d, Tensor(), Tensor()};
    }
};

std::optional<Tensor> next_token_loss(const Tensor& logits, const Tensor& labels, int64_t ignore) {
    if (has_tangent(logits)) return std::nullopt;
    c10::DeviceGuard guard(logits.device());
    if (at::GradMode::is_enabled() && logits.requires_grad()) return Loss::apply(logits, labels, ignore);
    at::AutoDispatchBelowADInplaceOrView below;
    return loss_rows(aligned(logits), labels.contiguous(), ignore).mean;
}

// ---------------------------------------------------------------------------------------------- clip and step

// One pass of gradient clipping and AdamW over all weights; groups[group_of[i]]: {lr, weight_decay, beta1, beta2, eps} of
// weight i.  Returns the gradients' norm, or nothing, with nothing done, if a tensor is not one the kernels take or the stream
// captures a graph: the table of pointers and the step's settings leave from a host buffer of this call alone, which a replay would
// read after others have used it (an optimizer that is not `capturable` refuses to be captured for the like reason).
std::optional<Tensor> clip_and_step(const std::vector<Tensor>& p, const std::vector<Tensor>& g, const std::vector<Tensor>& m,
                                    const std::vector<Tensor>& v, const std::vector<Tensor>& step,
                                    const std::vector<int64_t>& group_of, const std::vector<std::vector<double>>& groups,
                                    double max_norm) {
    const int64_t n = (int64_t)p.size();
    if (n == 0) return std::nullopt;
    const c10::Device device = p[0].device();
    for (int64_t i = 0; i < n; ++i) {
        for (const Tensor* t : {&p[i], &g[i], &m[i], &v[i]})
            if (t->scalar_type() != at::kFloat || t->device() != device || !device.is_cuda() || t->layout() != at::kStrided ||
                !t->is_contiguous() || t->numel() != p[i].numel())
                return std::nullopt;
        if (step[i].scalar_type() != at::kFloat || step[i].device() != device || step[i].numel() != 1) return std::nullopt;
    }
    c10::DeviceGuard guard(device);
    if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return std::nullopt;
    Tensor host = at::empty({n * (int64_t)sizeof(OptTensor)}, at::TensorOptions().dtype(at::kByte).pinned_memory(true));
    auto* t = (OptTensor*)host.data_ptr();
    int64_t chunks = 0;
    for (int64_t i = 0; i < n; ++i) {
        const auto& h = groups[group_of[i]];
        OptTensor o = {};
        o.p = p[i].data_ptr<float>();
        o.g = g[i].data_ptr<float>();
        o.m = m[i].data_ptr<float>();
        o.v = v[i].data_ptr<float>();
        o.step = step[i].data_ptr<float>();
        o.n = p[i].numel();
        o.first_chunk = chunks;
        o.lr = h[0];
        o.decay = (float)(1.0 - h[0] * h[1]);
        o.beta1 = h[2];
        o.beta2 = h[3];
        o.one_minus_beta1 = (float)(1.0 - h[2]);
        o.beta2_f = (float)h[3];
        o.one_minus_beta2 = (float)(1.0 - h[3]);
        o.eps = (float)h[4];
        t[i] = o;
        chunks += (o.n + kOptChunk - 1) / kOptChunk;
    }
    const Tensor table = host.to(device, /*non_blocking=*/true);
    const Tensor work = empty({chunks + 1}, p[0], at::kFloat), norm = empty({}, p[0], at::kFloat);
    ok(clip_and_adamw((OptTensor*)table.data_ptr(), (int)n, chunks, (float)max_norm, work.data_ptr<float>(), norm.data_ptr<float>(),
                      stream_of(p[0])));
    for (const auto* list : {&p, &g, &m, &v, &step})       // written in place
        for (const auto& x : *list) x.unsafeGetTensorImpl()->bump_version();
    return norm;
}

}  // namespace

void bind_model(py::module& m) {
    m.def("block", &block);
    m.def("head", &head);
    m.def("next_token_loss", &next_token_loss);
    m.def("clip_and_step", &clip_and_step);
    m.def("project", [](const Tensor& x, const Tensor& w, bool rows_w) {
        check_operands(x, w, rows_w);
        check_on_gpu(x);
        c10::DeviceGuard guard(x.device());
        return project(x, w, rows_w);
    });
    m.def("project_with", &project_with, py::arg("tile"), py::arg("x"), py::arg("w"), py::arg("rows_w"), py::arg("epilogue"), py::arg("residual"),
          py::arg("pre"), py::arg("out"), py::arg("splits") = 1);
    m.attr("projection_tiles") = (int)kTile64Halves + 1;
    m.def("project_add", [](const Tensor& x, const Tensor& w, const Tensor& residual) {
        check_operands(x, w, false);
        check_dense(residual, {x.size(0), w.size(0)}, at::kFloat, x, "residual");
        check_on_gpu(x);
        c10::DeviceGuard guard(x.device());
        return project_add(x, w, residual);
    });
    m.def("project_swiglu", [](const Tensor& x, const Tensor& w) {
        check_operands(x, w, false);
        TORCH_CHECK_VALUE(w.size(0) % 16 == 0, "gate and up must have a multiple of 8 rows each");
        check_on_gpu(x);
        c10::DeviceGuard guard(x.device());
        Tensor pre;
        const Tensor out = project_swiglu(x, w, pre, true);
        return std::make_pair(out, pre);
    });
    m.def("project_swiglu_grad", [](const Tensor& d, const Tensor& w, const Tensor& pre) {
        check_operands(d, w, true);
        check_dense(pre, {d.size(0), 2 * w.size(1)}, d.scalar_type(), d, "pre");
        TORCH_CHECK_VALUE(w.size(1) % 8 == 0, "gate and up must have a multiple of 8 columns each");
        check_on_gpu(d);
        c10::DeviceGuard guard(d.device());
        return project_swiglu_grad(d, w, pre);
    });
    m.def("weight_grad", [](const Tensor& d_out, const Tensor& in) {
        const auto t = d_out.scalar_type();
        TORCH_CHECK_TYPE((t == at::kBFloat16 || t == at::kHalf) && in.scalar_type() == t, "d_out and in must both be bfloat16 or both float16");
        TORCH_CHECK_VALUE(d_out.dim() == 2 && in.dim() == 2 && d_out.size(0) == in.size(0) &&
                          (d_out.numel() == 0 || (d_out.stride(1) == 1 && in.stride(1) == 1)) && d_out.device() == in.device(),
                          "d_out and in must be matrices of the same rows, which are dense");
        c10::OptionalDeviceGuard guard(d_out.device());
        return weight_grads({{d_out, in}})[0];
    });
    m.attr("max_norm_width") = kMaxNormWidth;
}

}  // namespace sba_torch
