// Autograd nodes of the differentiable ops in native code: what autograd's device thread runs for a training step.
//
// A torch.autograd.Function's backward in Python holds that thread for some 50 us (interpreter, argument struct, allocations), an
// attention's as long as the kernels of a small step; a node takes 12.  Nodes keep what the backward needs as torch's own do
// (saved variables, so hooks on them work and a changed tensor is noticed) and call the entry points of libt5attn.so, whose
// addresses the binding passes in.  Attention's forward stays in Python, which hands over its result; norms and linear layers are
// native both ways.  Gradients that are differentiated in their turn, or come in batches, take formulas in torch's operations
// (norms and linear layers; the attention kernels have no second derivative, and asking for one raises).
//
// us, a pass of small training calls bound by the host, Python functions / nodes: attention B4 H8 L512 fp32 162 / 95; T5-small encoder,
// 60 to 500 tokens 3 780 to 4 600 / 2 800.
#include <torch/extension.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include "../../include/t5attn.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

struct Library {
    decltype(&t5a_bwd_dense) bwd_dense;
    decltype(&t5a_bwd_varlen) bwd_varlen;
    decltype(&t5a_bwd_workspace_bytes) bwd_bytes;
    decltype(&t5a_bwd_varlen_workspace_bytes) bwd_varlen_bytes;
    decltype(&t5a_bwd_table_workspace_bytes) table_bytes;
    decltype(&t5a_last_error) last_error;
    decltype(&t5a_gemm_f32) gemm;
    decltype(&t5a_gemm_f32_workspace_bytes) gemm_bytes;
    decltype(&t5a_rmsnorm_train) norm;
    decltype(&t5a_rmsnorm_bwd_workspace_bytes) norm_bytes;
} lib;
PyObject* switches = nullptr;      // the names of the Python module that binds this one, kept for good

void bind(pybind11::dict names, uintptr_t bwd_dense, uintptr_t bwd_varlen, uintptr_t bwd_bytes, uintptr_t bwd_varlen_bytes, uintptr_t table_bytes, uintptr_t last_error,
          uintptr_t gemm, uintptr_t gemm_bytes, uintptr_t norm, uintptr_t norm_bytes) {
    switches = names.release().ptr();
    lib.gemm = reinterpret_cast<decltype(lib.gemm)>(gemm);
    lib.gemm_bytes = reinterpret_cast<decltype(lib.gemm_bytes)>(gemm_bytes);
    lib.norm = reinterpret_cast<decltype(lib.norm)>(norm);
    lib.norm_bytes = reinterpret_cast<decltype(lib.norm_bytes)>(norm_bytes);
    lib.bwd_dense = reinterpret_cast<decltype(lib.bwd_dense)>(bwd_dense);
    lib.bwd_varlen = reinterpret_cast<decltype(lib.bwd_varlen)>(bwd_varlen);
    lib.bwd_bytes = reinterpret_cast<decltype(lib.bwd_bytes)>(bwd_bytes);
    lib.bwd_varlen_bytes = reinterpret_cast<decltype(lib.bwd_varlen_bytes)>(bwd_varlen_bytes);
    lib.table_bytes = reinterpret_cast<decltype(lib.table_bytes)>(table_bytes);
    lib.last_error = reinterpret_cast<decltype(lib.last_error)>(last_error);
}

// A plain tensor: no subclass, batch, functional or tracing wrapper, no forward-mode tangent.
bool plain_tensor(const Tensor& t) {
    constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::BatchedNestedTensor,
                                           c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched, c10::DispatchKey::Functionalize,
                                           c10::DispatchKey::ZeroTensor, c10::DispatchKey::Negative, c10::DispatchKey::Conjugate});
    return t.layout() == at::kStrided && !t.key_set().has_any(wrapped) && !t._fw_grad(0).defined();
}
bool plain_state() {
    return !torch::jit::tracer::isTracing() && !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
           c10::impl::TorchDispatchModeTLS::stack_len() == 0;
}

int type_code(const Tensor& t) {
    switch (t.scalar_type()) {
        case at::kBFloat16: return T5A_BF16;
        case at::kHalf: return T5A_F16;
        case at::kFloat: return T5A_F32;
        default: return -1;
    }
}

// head_dim contiguous, 16-byte aligned rows; a copy only where that fails
Tensor ready(const Tensor& t) {
    const int64_t unit = t.scalar_type() == at::kFloat ? 4 : 8;
    bool ok = t.stride(-1) == 1 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
    for (int64_t i = 0; ok && i + 1 < t.dim(); ++i) ok = t.stride(i) % unit == 0;
    return ok ? t : t.contiguous();
}
template <size_t N> void strides(const Tensor& t, int64_t (&out)[N]) {
    for (size_t i = 0; i < N; ++i) out[i] = t.stride(i);
}
t5a_bias bias_args(const Tensor& table, int buckets, int max_distance) {
    t5a_bias b = {};
    if (!table.defined()) return b;
    b.table = table.data_ptr();
    b.table_dtype = type_code(table);
    b.num_buckets = buckets;
    b.max_distance = max_distance;
    b.stride_bucket = table.stride(0);
    b.stride_head = table.stride(1);
    return b;
}
void check(int rc) { TORCH_CHECK(rc == T5A_OK, "libt5attn error ", rc, ": ", lib.last_error()); }
void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// `BACKWARD_FP32_MATH` of the Python module, as the Python backward reads it: when it runs
bool fp32_math() {
    pybind11::gil_scoped_acquire gil;
    PyObject* const value = PyDict_GetItemString(switches, "BACKWARD_FP32_MATH");
    const int on = value != nullptr ? PyObject_IsTrue(value) : 0;
    if (on < 0) throw pybind11::error_already_set();
    return on != 0;
}

template <typename N> std::shared_ptr<N> make_node() { return std::shared_ptr<N>(new N(), torch::autograd::deleteNode); }

// Gradients of an attention call whose graph is kept: good as they are, an error where one is differentiated in its turn (and not a
// derivative that silently lacks the terms through the attention).  `of`: what they depend on, so that the error lies on the way to it.
void first_order_only(variable_list& grads, const variable_list& of) {
    auto error = std::shared_ptr<torch::autograd::Error>(
        new torch::autograd::Error("the fused-bias attention has no second derivative", torch::autograd::collect_next_edges(of)), torch::autograd::deleteNode);
    for (const Tensor& g : grads)
        if (g.defined()) torch::autograd::set_history(g, error);
}

struct Params {
    bool causal; double scale; int buckets, max_distance, exact;
    int64_t max_q = 0, max_k = 0;
};

struct AttentionBackward : public Node {
    SavedVariable q_, k_, v_, o_, lse_, table_;
    Tensor cu_q, cu_k, len_q, len_k;      // packed batches: int32, on the device
    bool has_table = false, packed = false;
    Params p;

    std::string name() const override { return packed ? "FlashAttentionBiasVarlenBackward" : "FlashAttentionBiasBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable* s : {&q_, &k_, &v_, &o_, &lse_, &table_}) s->reset_data();
    }

    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(has_table ? 4 : 3);
        if (!grads[0].defined()) return out;
        const auto self = getptr();
        Tensor q0 = q_.unpack(), k0 = k_.unpack(), v0 = v_.unpack(), o0 = o_.unpack(self), lse = lse_.unpack(), table = has_table ? table_.unpack() : Tensor();
        const bool wide_math = fp32_math();
        TORCH_CHECK_NOT_IMPLEMENTED(q0.size(-1) != 128 || (q0.scalar_type() != at::kFloat && !wide_math),
                                    "backward at head_dim 128: bf16 / fp16 tensors only (the fp32 kernels cover head_dim 16, 32 and 64)");
        const bool graph_kept = at::GradMode::is_enabled();
        at::NoGradGuard no_grad;
        const c10::OptionalDeviceGuard device(q0.device());
        const Tensor g0 = grads[0];
        const Tensor q = ready(q0), k = ready(k0), v = ready(v0), o = ready(o0), g = ready(g0.scalar_type() == q0.scalar_type() ? g0 : g0.to(q0.scalar_type()));
        const bool pad_q = len_q.defined(), pad_k = len_k.defined();
        // (rows of padding get no gradient)
        const Tensor dq = pad_q ? at::zeros_like(q) : at::empty_like(q), dk = pad_k ? at::zeros_like(k) : at::empty_like(k),
                     dv = pad_k ? at::zeros_like(v) : at::empty_like(v);
        const Tensor wide = table.defined() && type_code(table) < 0 ? table.to(at::kFloat) : table;
        const int64_t H = q.size(1), B = packed ? cu_q.numel() - 1 : q.size(0), rows = packed ? p.max_q : q.size(2);
        const auto f32 = q.options().dtype(at::kFloat);
        const Tensor dtable = has_table ? at::empty({p.buckets, H}, f32) : Tensor();
        int64_t bytes = packed ? lib.bwd_varlen_bytes((int)q.size(0), (int)H) : lib.bwd_bytes((int)B, (int)H, (int)rows);
        bytes = std::max<int64_t>((bytes + 15) / 16 * 16, 16);
        if (has_table) bytes += lib.table_bytes((int)B, (int)H, (int)rows, p.buckets);
        const Tensor ws = at::empty({bytes}, q.options().dtype(at::kByte));
        auto fill = [&](auto& a) {
            a.q = q.data_ptr(); a.k = k.data_ptr(); a.v = v.data_ptr(); a.o = o.data_ptr(); a.dout = g.data_ptr(); a.lse = lse.data_ptr<float>();
            a.dq = dq.data_ptr(); a.dk = dk.data_ptr(); a.dv = dv.data_ptr(); a.dtable = has_table ? dtable.data_ptr<float>() : nullptr;
            a.workspace = ws.data_ptr(); a.workspace_bytes = bytes;
            strides(q, a.q_strides); strides(k, a.k_strides); strides(v, a.v_strides); strides(o, a.o_strides); strides(g, a.dout_strides);
            strides(dq, a.dq_strides); strides(dk, a.dk_strides); strides(dv, a.dv_strides);
            a.dtype = type_code(q); a.B = (int)B; a.H = (int)H; a.D = (int)q.size(-1);
            a.causal = p.causal; a.sm_scale = (float)p.scale; a.exact_scores = p.exact; a.fp32_math = wide_math;
            a.bias = bias_args(wide, p.buckets, p.max_distance);
        };
        if (packed) {
            t5a_varlen_bwd_args a = {};
            fill(a);
            a.cu_seqlens_q = cu_q.data_ptr<int>(); a.cu_seqlens_k = cu_k.data_ptr<int>();
            a.seq_lens_q = pad_q ? len_q.data_ptr<int>() : nullptr; a.seq_lens_k = pad_k ? len_k.data_ptr<int>() : nullptr;
            a.total_q = (int)q.size(0); a.total_k = (int)k.size(0); a.max_seqlen_q = (int)p.max_q; a.max_seqlen_k = (int)p.max_k;
            check(lib.bwd_varlen(&a, stream_of(q)));
        } else {
            t5a_dense_bwd_args a = {};
            fill(a);
            a.M = (int)q.size(2); a.N = (int)k.size(2);
            check(lib.bwd_dense(&a, stream_of(q)));
        }
        out[0] = dq; out[1] = dk; out[2] = dv;
        if (has_table && task_should_compute_output(3)) out[3] = dtable.scalar_type() == table.scalar_type() ? dtable : dtable.to(table.scalar_type());
        if (graph_kept) {
            variable_list of = {q0, k0, v0, g0};
            if (has_table) of.push_back(table);
            first_order_only(out, of);
        }
        return out;
    }
};

void attach(const Tensor& o, const Tensor& lse, const Tensor& q, const Tensor& k, const Tensor& v, const c10::optional<Tensor>& table,
            const c10::optional<Tensor>& cu_q, const c10::optional<Tensor>& cu_k, const c10::optional<Tensor>& len_q, const c10::optional<Tensor>& len_k,
            const Params& p) {
    auto node = make_node<AttentionBackward>();
    node->has_table = table.has_value();
    node->packed = cu_q.has_value();
    node->p = p;
    if (node->has_table) node->set_next_edges(torch::autograd::collect_next_edges(q, k, v, *table));
    else node->set_next_edges(torch::autograd::collect_next_edges(q, k, v));
    node->q_ = SavedVariable(q, false); node->k_ = SavedVariable(k, false); node->v_ = SavedVariable(v, false);
    if (node->has_table) node->table_ = SavedVariable(*table, false);
    if (node->packed) {
        node->cu_q = *cu_q; node->cu_k = *cu_k;
        if (len_q) node->len_q = *len_q;
        if (len_k) node->len_k = *len_k;
    }
    torch::autograd::set_history(o, node);
    node->o_ = SavedVariable(o, true);
    node->lse_ = SavedVariable(lse, false);
}

// --------------------------------------------------------------------------------------------- linear layers in fp32

// contiguous aligned rows, fp32 or bf16 (wide: fp32)
Tensor rows(const Tensor& t, bool wide = false) {
    Tensor r = t.scalar_type() == at::kHalf || (wide && t.scalar_type() != at::kFloat) ? t.to(at::kFloat) : t;
    r = r.contiguous();
    return reinterpret_cast<uintptr_t>(r.data_ptr()) % 16 == 0 ? r : r.clone();
}

// c[g] = alpha_g a[g] b[g]^T over contiguous matrices (t5attn.h)
struct Gemm { bool a_trans = false, b_trans = false, sum = false, relu = false; double alpha = 1.0; Tensor positive; };
void gemm(const variable_list& a, const variable_list& b, const variable_list& c, const Gemm& how) {
    t5a_gemm_f32_args g = {};
    for (size_t i = 0; i < a.size(); ++i) {
        g.a[i] = a[i].data_ptr(); g.b[i] = b[i].data_ptr();
        g.c[i] = c[how.sum ? 0 : i].data_ptr();
    }
    g.lda = a[0].size(1); g.ldb = b[0].size(1); g.ldc = c[0].size(1);
    if (how.positive.defined()) { g.positive = how.positive.data_ptr<float>(); g.ld_positive = how.positive.size(1); }
    g.M = (int)c[0].size(0); g.N = (int)c[0].size(1); g.K = (int)a[0].size(how.a_trans ? 0 : 1);
    g.groups = (int)a.size(); g.sum_groups = how.sum;
    g.a_dtype = type_code(a[0]); g.b_dtype = type_code(b[0]); g.c_dtype = type_code(c[0]);
    g.a_trans = how.a_trans; g.b_trans = how.b_trans; g.relu = how.relu; g.alpha = (float)how.alpha;
    const int64_t bytes = lib.gemm_bytes(&g);
    Tensor ws;
    if (bytes > 0) {
        ws = at::empty({bytes}, c[0].options().dtype(at::kByte));
        g.workspace = ws.data_ptr(); g.workspace_bytes = bytes;
    }
    check(lib.gemm(&g, stream_of(c[0])));
}

bool plain_all(const variable_list& ts) {
    if (!plain_state()) return false;
    for (const Tensor& t : ts)
        if (t.defined() && !plain_tensor(t)) return false;
    return true;
}

// x W_0^T factor, x W_1^T, ...: the same rows with up to three weights of one shape, rounded to one type once
struct ProjectionsBackward : public Node {
    SavedVariable x_;
    std::vector<SavedVariable> w_;
    double factor = 1.0;
    at::ScalarType dtype = at::kFloat;

    std::string name() const override { return "ProjectionsBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        x_.reset_data();
        for (auto& s : w_) s.reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        const size_t n = w_.size();
        variable_list out(1 + n);
        Tensor x = x_.unpack();
        variable_list w(n);
        bool any = false;
        for (size_t i = 0; i < n; ++i) { w[i] = w_[i].unpack(); any |= grads[i].defined(); }
        if (!any) return out;
        const c10::OptionalDeviceGuard device(x.device());
        for (size_t i = 0; i < n; ++i)
            if (!grads[i].defined()) grads[i] = at::zeros({x.size(0), w[i].size(0)}, x.options().dtype(dtype));
        variable_list all = grads;
        all.insert(all.end(), w.begin(), w.end());
        all.push_back(x);
        if (at::GradMode::is_enabled() || !plain_all(all)) {
            const Tensor wide = x.to(at::kFloat);
            for (size_t i = 0; i < n; ++i) {
                const Tensor g = i == 0 ? grads[i].to(at::kFloat) * factor : grads[i].to(at::kFloat);
                if (task_should_compute_output(0)) { const Tensor part = at::matmul(g, w[i]); out[0] = out[0].defined() ? out[0] + part : part; }
                if (task_should_compute_output(1 + i)) out[1 + i] = at::matmul(g.transpose(-1, -2), wide);
            }
            if (out[0].defined()) out[0] = out[0].to(x.scalar_type());
            return out;
        }
        at::NoGradGuard no_grad;
        variable_list g(n);
        for (size_t i = 0; i < n; ++i) g[i] = rows(grads[i]);
        if (task_should_compute_output(0)) {
            variable_list wr(n);
            for (size_t i = 0; i < n; ++i) wr[i] = rows(w[i]);
            out[0] = at::empty(x.sizes(), x.options());
            Gemm how; how.b_trans = true; how.sum = true; how.alpha = factor;
            gemm(g, wr, {out[0]}, how);
        }
        variable_list ga, xb, c;
        Gemm how; how.a_trans = how.b_trans = true;
        Tensor xr;
        for (size_t i = 0; i < n; ++i) {
            if (!task_should_compute_output(1 + i)) continue;
            if (!xr.defined()) xr = rows(x, g[0].scalar_type() == at::kBFloat16);
            if (c.empty() && i == 0) how.alpha = factor;
            out[1 + i] = at::empty(w[i].sizes(), w[i].options());
            ga.push_back(g[i]); xb.push_back(xr); c.push_back(out[1 + i]);
        }
        if (!c.empty()) gemm(ga, xb, c, how);
        return out;
    }
};

variable_list project(const Tensor& x, at::ScalarType dtype, double factor, const std::vector<Tensor>& w) {
    auto node = make_node<ProjectionsBackward>();
    variable_list out, inputs = {x};
    {
        at::NoGradGuard no_grad;
        const c10::OptionalDeviceGuard device(x.device());
        const Tensor xr = rows(x);
        variable_list a, b;
        for (const Tensor& t : w) {
            a.push_back(xr); b.push_back(rows(t)); inputs.push_back(t);
            out.push_back(at::empty({x.size(0), t.size(0)}, x.options().dtype(dtype)));
        }
        Gemm how; how.alpha = factor;
        gemm(a, b, out, how);
    }
    node->set_next_edges(torch::autograd::collect_next_edges(inputs));
    node->factor = factor; node->dtype = dtype;
    node->x_ = SavedVariable(x, false);
    for (const Tensor& t : w) node->w_.emplace_back(t, false);
    torch::autograd::set_history(out, node);
    return out;
}

// relu(x W_i^T) W_o^T: ReLU and its derivative are part of the products that make their operand
struct FeedForwardReluBackward : public Node {
    SavedVariable x_, wi_, wo_, mid_;
    std::string name() const override { return "FeedForwardReluBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable* s : {&x_, &wi_, &wo_, &mid_}) s->reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(3);
        const Tensor dy0 = grads[0];
        if (!dy0.defined()) return out;
        const Tensor x = x_.unpack(), wi = wi_.unpack(), wo = wo_.unpack(), mid0 = mid_.unpack();
        const c10::OptionalDeviceGuard device(x.device());
        const bool need_x = task_should_compute_output(0), need_wi = task_should_compute_output(1), need_wo = task_should_compute_output(2);
        if (at::GradMode::is_enabled() || !plain_all({x, wi, wo, dy0})) {
            const Tensor mid = at::relu(at::matmul(x, wi.t()));      // (differentiable in its turn)
            const Tensor dmid = at::matmul(dy0, wo) * (mid > 0);
            if (need_x) out[0] = at::matmul(dmid, wi);
            if (need_wi) out[1] = at::matmul(dmid.transpose(-1, -2), x);
            if (need_wo) out[2] = at::matmul(dy0.transpose(-1, -2), mid);
            return out;
        }
        at::NoGradGuard no_grad;
        const Tensor dy = rows(dy0), mid = rows(mid0);
        Gemm tt; tt.a_trans = tt.b_trans = true;
        Gemm nt; nt.b_trans = true;
        if (need_wo) { out[2] = at::empty(wo.sizes(), wo.options()); gemm({dy}, {mid}, {out[2]}, tt); }
        if (need_x || need_wi) {
            const Tensor dmid = at::empty_like(mid);
            Gemm masked = nt; masked.positive = mid;
            gemm({dy}, {rows(wo)}, {dmid}, masked);
            if (need_wi) { out[1] = at::empty(wi.sizes(), wi.options()); gemm({dmid}, {rows(x)}, {out[1]}, tt); }
            if (need_x) { out[0] = at::empty(x.sizes(), x.options()); gemm({dmid}, {rows(wi)}, {out[0]}, nt); }
        }
        return out;
    }
};

Tensor feed_forward_relu(const Tensor& x, const Tensor& wi, const Tensor& wo) {
    auto node = make_node<FeedForwardReluBackward>();
    Tensor mid, out;
    {
        at::NoGradGuard no_grad;
        const c10::OptionalDeviceGuard device(x.device());
        mid = at::empty({x.size(0), wi.size(0)}, x.options());
        out = at::empty({x.size(0), wo.size(0)}, x.options());
        Gemm how; how.relu = true;
        gemm({rows(x)}, {rows(wi)}, {mid}, how);
        gemm({mid}, {rows(wo)}, {out}, Gemm{});
    }
    node->set_next_edges(torch::autograd::collect_next_edges(x, wi, wo));
    node->x_ = SavedVariable(x, false); node->wi_ = SavedVariable(wi, false); node->wo_ = SavedVariable(wo, false);
    node->mid_ = SavedVariable(mid, false);
    torch::autograd::set_history(out, node);
    return out;
}

// ------------------------------------------------------------------------------------------- the norm of a training step

// y, or with dy (dx, dweight), over contiguous rows
void norm_call(const Tensor& x, const Tensor& weight, const Tensor& rstd, const Tensor& y, const Tensor& dy, const Tensor& dsum, const Tensor& dx, const Tensor& dw) {
    t5a_rmsnorm_train_args a = {};
    a.x = x.data_ptr(); a.weight = weight.data_ptr(); a.rstd = rstd.data_ptr<float>();
    a.rows = x.numel() / x.size(-1); a.dim = (int)x.size(-1);
    a.x_dtype = type_code(x); a.weight_dtype = type_code(weight);
    Tensor ws;
    if (y.defined()) {
        a.y = y.data_ptr();
    } else {
        a.dy = dy.data_ptr(); a.dsum = dsum.defined() ? dsum.data_ptr() : nullptr;
        a.dx = dx.data_ptr(); a.dweight = dw.data_ptr();
        a.workspace_bytes = lib.norm_bytes(a.rows, a.dim);
        ws = at::empty({a.workspace_bytes}, x.options().dtype(at::kByte));
        a.workspace = ws.data_ptr();
    }
    check(lib.norm(&a, stream_of(x)));
}
Tensor aligned(const Tensor& t) {
    const Tensor r = t.contiguous();
    return reinterpret_cast<uintptr_t>(r.data_ptr()) % 16 == 0 ? r : r.clone();
}
bool is_half(const Tensor& t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }

struct RmsNormBackward : public Node {
    SavedVariable total_, weight_, rstd_;
    bool stream = false, residual = false, saved_output = false;     // stream: the sum is an output with a gradient of its own
    double eps = 0.0;

    std::string name() const override { return "RmsNormBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (SavedVariable* s : {&total_, &weight_, &rstd_}) s->reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(residual ? 3 : 2);
        const Tensor dsum = stream ? grads[0] : Tensor(), dy = grads[stream ? 1 : 0];
        Tensor dx, dw;
        if (!dy.defined()) {
            dx = dsum;
        } else {
            const Tensor x = saved_output ? total_.unpack(getptr()) : total_.unpack(), weight = weight_.unpack(), rstd0 = rstd_.unpack();
            const c10::OptionalDeviceGuard device(x.device());
            if (at::GradMode::is_enabled() || !plain_all({x, weight, dy, dsum})) {
                // the kernel's backward in torch's operations
                const Tensor x32 = x.to(at::kFloat), rstd = at::rsqrt(x32.pow(2).mean(-1, true) + eps);
                Tensor n = x32 * rstd;
                if (is_half(weight)) n = n.to(weight.scalar_type());
                const Tensor g = (dy * weight).to(at::kFloat);
                dx = rstd * g - x32 * (rstd.pow(3) * (g * x32).mean(-1, true));
                if (dsum.defined()) dx = dx + dsum;
                std::vector<int64_t> outer(dy.dim() - 1);
                for (size_t i = 0; i < outer.size(); ++i) outer[i] = (int64_t)i;
                dw = dy.to(at::kFloat) * n;
                dw = (outer.empty() ? dw : dw.sum(outer)).to(weight.scalar_type());
                dx = dx.to(x.scalar_type());
            } else {
                at::NoGradGuard no_grad;
                const Tensor xr = aligned(x), w = weight.contiguous();
                dx = at::empty_like(xr);
                dw = at::empty_like(w);
                norm_call(xr, w, rstd0, Tensor(), aligned(dy), dsum.defined() ? aligned(dsum) : Tensor(), dx, dw);
            }
        }
        if (task_should_compute_output(0)) out[0] = dx;
        if (task_should_compute_output(1)) out[1] = dw;
        if (residual && task_should_compute_output(2)) out[2] = dx;
        return out;
    }
};

// (x + residual, norm of that sum), or without a residual (None, norm of x).  The mean square and the root are torch's own, so that a
// step's activations are bit for bit those of the expression in torch's operations.
pybind11::tuple rms_norm_train(const Tensor& x, const Tensor& weight, double eps, const c10::optional<Tensor>& residual) {
    auto node = make_node<RmsNormBackward>();
    Tensor total, rstd, y;
    {
        at::NoGradGuard no_grad;
        const c10::OptionalDeviceGuard device(x.device());
        total = residual ? x + *residual : x;
        rstd = at::rsqrt(total.to(at::kFloat).pow(2).mean(-1, true) + eps).contiguous();
        y = at::empty(x.sizes(), x.options().dtype(is_half(weight) ? weight.scalar_type() : at::kFloat));
        norm_call(aligned(total), weight.contiguous(), rstd, y, Tensor(), Tensor(), Tensor(), Tensor());
    }
    node->eps = eps;
    node->residual = residual.has_value();
    // (only the weight is trained: the residual stream carries no graph)
    node->stream = residual && (x.requires_grad() || residual->requires_grad());
    node->saved_output = node->stream;
    if (residual) node->set_next_edges(torch::autograd::collect_next_edges(x, weight, *residual));
    else node->set_next_edges(torch::autograd::collect_next_edges(x, weight));
    if (node->stream) torch::autograd::set_history(variable_list{total, y}, node);
    else torch::autograd::set_history(y, node);
    node->total_ = SavedVariable(total, node->stream);
    node->weight_ = SavedVariable(weight, false);
    node->rstd_ = SavedVariable(rstd, false);
    if (!residual) return pybind11::make_tuple(pybind11::none(), y);
    return pybind11::make_tuple(total, y);
}

// Whether a call takes a node: plain tensors (no subclass) and plain reverse-mode autograd.
bool takes(const pybind11::list& tensors) {
    if (!plain_state()) return false;
    for (const auto& o : tensors) {
        if (o.is_none()) continue;
        if (!THPVariable_CheckExact(o.ptr()) || !plain_tensor(THPVariable_Unpack(o.ptr()))) return false;
    }
    return true;
}

}  // namespace

PYBIND11_MODULE(_native, m) {
    m.attr("abi_version") = T5A_ABI_VERSION;
    m.def("bind", &bind);
    m.def("takes", &takes);
    m.def("first_order_only", [](const std::vector<c10::optional<Tensor>>& grads, const std::vector<c10::optional<Tensor>>& of) {
        auto defined = [](const std::vector<c10::optional<Tensor>>& ts) {
            variable_list out;
            for (const auto& t : ts)
                if (t) out.push_back(*t);
            return out;
        };
        variable_list g = defined(grads);
        first_order_only(g, defined(of));
    });
    m.def("gemm", [](const variable_list& a, const variable_list& b, const variable_list& c, bool a_trans, bool b_trans, bool sum, bool relu, double alpha,
                     const c10::optional<Tensor>& positive) {
        at::NoGradGuard no_grad;
        const c10::OptionalDeviceGuard device(c.at(0).device());
        Gemm how;
        how.a_trans = a_trans; how.b_trans = b_trans; how.sum = sum; how.relu = relu; how.alpha = alpha;
        if (positive) how.positive = *positive;
        gemm(a, b, c, how);
    });
    m.def("project", &project);
    m.def("feed_forward_relu", &feed_forward_relu);
    m.def("rms_norm_train", &rms_norm_train);
    m.def("attach_dense", [](const Tensor& o, const Tensor& lse, const Tensor& q, const Tensor& k, const Tensor& v, const c10::optional<Tensor>& table,
                             bool causal, double scale, int buckets, int max_distance, int exact) {
        attach(o, lse, q, k, v, table, {}, {}, {}, {}, Params{causal, scale, buckets, max_distance, exact});
    });
    m.def("attach_varlen", [](const Tensor& o, const Tensor& lse, const Tensor& q, const Tensor& k, const Tensor& v, const c10::optional<Tensor>& table,
                              const Tensor& cu_q, const Tensor& cu_k, int64_t max_q, int64_t max_k, const c10::optional<Tensor>& len_q,
                              const c10::optional<Tensor>& len_k, bool causal, double scale, int buckets, int max_distance, int exact) {
        attach(o, lse, q, k, v, table, cu_q, cu_k, len_q, len_k, Params{causal, scale, buckets, max_distance, exact, max_q, max_k});
    });
}
