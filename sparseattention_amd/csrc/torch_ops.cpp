// The hot calls of the Python layer in native code: argument checks, output allocation, the launch
// through the C ABI and, for the span attention, the autograd node.
//
// Why: at the sizes users call most the kernels take 20 to 70 us, and one call through ctypes, with
// its checks and allocations in Python, takes 12 to 20 us of host time; the backward of a Python
// autograd.Function additionally has to get the interpreter lock on the engine's thread.  Forward
// and backward at B8 H8 N2048 D64 (70 us of kernels): 115 us a call in Python, 69 us here (the kernels);
// tree build + attention of B2 H4 N256 D32 fp32 (18 us of kernels): 31.5 -> 16.4 us.
//
// Every function returns None when the arguments are not the plain case (all tensors on one GPU, of
// one type, shapes consistent): the Python layer then goes through its own checks, which raise the
// errors and handle the rest.
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/functions/basic_ops.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/utils/pybind.h>

#include <ATen/ATen.h>
#include <ATen/TracerMode.h>
#include <ATen/autocast_mode.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>

#include "../../include/hsa_gfx950.h"

namespace {

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

int type_code(at::ScalarType type) {
    switch (type) {
        case at::kFloat: return HSA_F32;
        case at::kHalf: return HSA_F16;
        case at::kBFloat16: return HSA_BF16;
        default: return -1;
    }
}
int type_code(const Tensor &t) { return type_code(t.scalar_type()); }

void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// what the library refuses: _lib.HsaError in Python
struct LibraryError : public std::runtime_error {
    using std::runtime_error::runtime_error;
};
void check(int rc, const char *what) {
    if (rc != HSA_OK) throw LibraryError(c10::str(what, " failed (", rc, "): ", hsa_last_error()));
}

bool same_kind(const Tensor &a, const Tensor &b) {
    return b.defined() && b.is_cuda() && a.device() == b.device() && a.scalar_type() == b.scalar_type();
}

// Nothing that watches or transforms torch's own calls: no tracing, no dispatch mode, no tensor subclass
// or functional transform, no forward-mode tangent; and nothing without strides (sparse).  Such calls go the general
// way, which either supports them or says that it does not.
bool ordinary(std::initializer_list<const Tensor *> ts) {
    constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::Batched,
                                           c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                           c10::DispatchKey::Functionalize});
    if (at::tracer::impl::is_dispatch_enabled() || c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Python))
        return false;
    for (const Tensor *t : ts)
        if (t->layout() != at::kStrided || t->key_set().has_any(wrapped) || t->_fw_grad(0).defined()) return false;
    return true;
}

// Whether a backward computes with torch's operations instead of the kernels: it is itself differentiated,
// or a transform watches the gradients (a batch of them under vmap).
bool composed(const variable_list &grads) {
    if (at::GradMode::is_enabled()) return true;
    for (const Tensor &g : grads)
        if (g.defined() && !ordinary({&g})) return true;
    return false;
}

bool aligned16(const Tensor &t) { return ((uintptr_t)t.data_ptr() & 15) == 0; }

int log2_exact(int64_t n) {
    int l = 0;
    while ((1ll << l) < n) ++l;
    return (1ll << l) == n ? l : -1;
}

Tensor workspace(const Tensor &like, size_t bytes) {
    return at::empty({(int64_t)((bytes + 3) / 4 + 1)}, like.options().dtype(at::kFloat));
}

// ------------------------------------------------------------------ span attention, canonical tables
struct Shape {
    int B, N, M, H, D, L, dtype;
};

Shape shape_of(const Tensor &Q, const Tensor &K) {
    return {(int)Q.size(0), (int)Q.size(1), (int)K.size(1), (int)Q.size(2), (int)Q.size(3), log2_exact(Q.size(1)),
            type_code(Q)};
}

Tensor attention_plain(const Tensor &Q, const Tensor &K, const Tensor &V, bool causal, int R) {
    const Shape s = shape_of(Q, K);
    Tensor out = at::empty_like(Q);
    c10::DeviceGuard guard(Q.device());
    check(hsa_attn_fwd(Q.data_ptr(), K.data_ptr(), V.data_ptr(), nullptr, nullptr, out.data_ptr(), nullptr, s.B, s.N,
                       s.M, s.H, s.D, s.L, R, causal, s.dtype, HSA_ATTN_AUTO, stream_of(Q)),
          "hsa_attn_fwd");
    return out;
}

// Forward keeps Q, K, V and, where the one-pass backward takes the problem, the output and one
// log-sum-exp per (query, head) (the reference keeps its Weights tensor,
// hierarchical_attention/ops/functional.py:116-264).
struct SpanAttention : public torch::autograd::Function<SpanAttention> {
    // one_pass: whether the one-pass backward is wanted where it is built for the head size
    static Tensor forward(AutogradContext *ctx, const Tensor &Qi, const Tensor &Ki, const Tensor &Vi, bool causal,
                          int64_t R, bool one_pass) {
        const Tensor Q = Qi.contiguous(), K = Ki.contiguous(), V = Vi.contiguous();
        const Shape s = shape_of(Q, K);
        ctx->saved_data["causal"] = causal;
        ctx->saved_data["R"] = R;
        if (one_pass && hsa_attn_bwd_saved_workspace_bytes(s.B, s.N, s.M, s.H, s.D, s.L, (int)R, causal, s.dtype) > 0 &&
            aligned16(Q) && aligned16(K) && aligned16(V)) {
            Tensor out = at::empty_like(Q);
            Tensor lse = at::empty({s.B, s.N, s.H}, Q.options().dtype(at::kFloat));
            c10::DeviceGuard guard(Q.device());
            const int rc = hsa_attn_fwd_lse(Q.data_ptr(), K.data_ptr(), V.data_ptr(), out.data_ptr(),
                                            (float *)lse.data_ptr(), s.B, s.N, s.M, s.H, s.D, s.L, (int)R, causal,
                                            s.dtype, stream_of(Q));
            if (rc != HSA_ERR_UNSUPPORTED) {  // unsupported: nothing was launched
                check(rc, "hsa_attn_fwd_lse");
                ctx->save_for_backward({Q, K, V, out, lse});
                return out;
            }
        }
        Tensor out = attention_plain(Q, K, V, causal, (int)R);
        ctx->save_for_backward({Q, K, V});
        return out;
    }

    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list saved = ctx->get_saved_variables();
        for (Tensor &t : saved) t = t.contiguous();  // (saved-tensor hooks may give back another layout)
        const Tensor &Q = saved[0], &K = saved[1], &V = saved[2];
        const bool causal = ctx->saved_data["causal"].toBool();
        const int R = (int)ctx->saved_data["R"].toInt();
        const Shape s = shape_of(Q, K);
        const Tensor G = grads[0].contiguous();
        Tensor dq = at::empty_like(Q), dk = at::empty_like(K), dv = at::empty_like(V);
        c10::DeviceGuard guard(Q.device());
        if (saved.size() == 5 && aligned16(G) && aligned16(Q) && aligned16(K) && aligned16(V) && aligned16(saved[3])) {
            const size_t bytes = hsa_attn_bwd_saved_workspace_bytes(s.B, s.N, s.M, s.H, s.D, s.L, R, causal, s.dtype);
            Tensor ws = workspace(Q, bytes);
            check(hsa_attn_bwd_saved(Q.data_ptr(), K.data_ptr(), V.data_ptr(), saved[3].data_ptr(),
                                     (const float *)saved[4].data_ptr(), G.data_ptr(), dq.data_ptr(), dk.data_ptr(),
                                     dv.data_ptr(), ws.data_ptr(), ws.nbytes(), s.B, s.N, s.M, s.H, s.D, s.L, R, causal,
                                     s.dtype, stream_of(Q)),
                  "hsa_attn_bwd_saved");
        } else {
            // the tile kernels move 16-byte pieces
            const int algo = aligned16(Q) && aligned16(K) && aligned16(V) && aligned16(G) ? HSA_ATTN_AUTO : HSA_ATTN_GATHER;
            Tensor ws = workspace(Q, hsa_attn_bwd_workspace_bytes(s.B, s.N, s.M, s.H, s.D, s.L, R, s.dtype, algo));
            check(hsa_attn_bwd(Q.data_ptr(), K.data_ptr(), V.data_ptr(), G.data_ptr(), dq.data_ptr(), dk.data_ptr(),
                               dv.data_ptr(), ws.data_ptr(), ws.nbytes(), s.B, s.N, s.M, s.H, s.D, s.L, R, causal,
                               s.dtype, algo, stream_of(Q)),
                  "hsa_attn_bwd");
        }
        if (at::GradMode::is_enabled()) {
            // the kernels have no derivative: differentiating these gradients again raises instead of leaving
            // the attention's terms out
            variable_list once;
            for (const Tensor &t : {dq, dk, dv}) once.push_back(t.detach().set_requires_grad(true));
            const auto error = std::make_shared<torch::autograd::DelayedError>(
                "the span attention cannot be differentiated twice", (int64_t)once.size());
            once = (*error)(std::move(once));
            return {once[0], once[1], once[2], Tensor(), Tensor(), Tensor()};
        }
        return {dq, dk, dv, Tensor(), Tensor(), Tensor()};
    }
};

// The tables are known to be build_tree_topology's for N = Q's rows with this causal flag.  part_one_pass:
// the one-pass backward for head sizes other than 32 / 64 / 128 channels too.
std::optional<Tensor> span_attention(const Tensor &Q, const Tensor &K, const Tensor &V, bool causal, int64_t R,
                                     bool part_one_pass) {
    if (!Q.is_cuda() || Q.dim() != 4 || K.dim() != 4 || !same_kind(Q, K) || !same_kind(Q, V) || type_code(Q) < 0 ||
        K.sizes() != V.sizes() || K.size(0) != Q.size(0) || K.size(2) != Q.size(2) || K.size(3) != Q.size(3) ||
        K.size(1) < 2 * Q.size(1) - 1 || Q.numel() == 0 || log2_exact(Q.size(1)) < 0 || R < 0 || R > (1 << 20) ||
        !ordinary({&Q, &K, &V}))
        return std::nullopt;
    if (at::GradMode::is_enabled() && (Q.requires_grad() || K.requires_grad() || V.requires_grad())) {
        const int64_t D = Q.size(3);
        return SpanAttention::apply(Q, K, V, causal, R, part_one_pass || D == 32 || D == 64 || D == 128);
    }
    return attention_plain(Q.contiguous(), K.contiguous(), V.contiguous(), causal, (int)R);
}

// ------------------------------------------------------------------------------------ tree build
bool dense_rows(const Tensor &t) {
    return t.stride(3) == 1 && t.stride(2) == t.size(3) && t.stride(1) == t.size(2) * t.size(3);
}
int64_t batch_stride(const Tensor &t) { return t.size(0) > 1 ? t.stride(0) : t.size(1) * t.size(2) * t.size(3); }

std::optional<Tensor> build_tree(const Tensor &Qp, const Tensor &Kp, const Tensor &Vp, const Tensor &Kl,
                                 const Tensor &Vl, const std::optional<Tensor> &out_, const std::optional<Tensor> &out2) {
    if (!Kl.is_cuda() || Kl.dim() != 4 || type_code(Kl) < 0 || Kl.numel() == 0 || Qp.dim() != 4) return std::nullopt;
    const int64_t B = Kl.size(0), N = Kl.size(1), H = Kl.size(2), D = Kl.size(3);
    if (N < 2 || log2_exact(N) < 0 || Qp.size(0) != B || Qp.size(1) != N - 1 || Qp.size(2) != H || Qp.size(3) != D ||
        Vl.sizes() != Kl.sizes())
        return std::nullopt;
    const Tensor *ins[5] = {&Qp, &Kp, &Vp, &Kl, &Vl};
    for (const Tensor *t : ins)
        if (!same_kind(Kl, *t) || !dense_rows(*t)) return std::nullopt;
    if (Kp.sizes() != Qp.sizes() || Vp.sizes() != Qp.sizes()) return std::nullopt;
    for (const std::optional<Tensor> *o : {&out_, &out2})
        if (*o && (!same_kind(Kl, **o) || (*o)->sizes() != Qp.sizes() || !dense_rows(**o))) return std::nullopt;
    const Tensor out = out_ ? *out_ : at::empty({B, N - 1, H, D}, Qp.options());
    c10::DeviceGuard guard(Kl.device());
    check(hsa_build_tree_fwd(Qp.data_ptr(), Kp.data_ptr(), Vp.data_ptr(), Kl.data_ptr(), Vl.data_ptr(), out.data_ptr(),
                             out2 ? out2->data_ptr() : nullptr, (int)B, (int)N, (int)H, (int)D, batch_stride(Qp),
                             batch_stride(Kp), batch_stride(Vp), batch_stride(Kl), batch_stride(Vl), batch_stride(out),
                             out2 ? batch_stride(*out2) : 0, type_code(Kl), stream_of(Kl)),
          "hsa_build_tree_fwd");
    return out;
}

// ------------------------------------------------------------------ residual sum and layer norm
struct NormShape {
    long rows;
    int C, dtype;
};
NormShape norm_shape(const Tensor &a) { return {(long)(a.numel() / a.size(-1)), (int)a.size(-1), type_code(a)}; }

// (sum, norm) of a and b, or (undefined, norm) of a alone; stats may be undefined
std::pair<Tensor, Tensor> add_norm_plain(const Tensor &a, const Tensor &b, const Tensor &gamma, const Tensor &beta,
                                         double eps, const Tensor &stats) {
    const NormShape s = norm_shape(a);
    Tensor sum = b.defined() ? at::empty_like(a) : Tensor(), norm = at::empty_like(a);
    c10::DeviceGuard guard(a.device());
    check(hsa_add_layer_norm_fwd(a.data_ptr(), b.defined() ? b.data_ptr() : nullptr, gamma.data_ptr(), beta.data_ptr(),
                                 b.defined() ? sum.data_ptr() : nullptr, norm.data_ptr(),
                                 stats.defined() ? (float *)stats.data_ptr() : nullptr, s.rows, s.C, (float)eps, s.dtype,
                                 stream_of(a)),
          "hsa_add_layer_norm_fwd");
    return {sum, norm};
}

// outputs: sum, norm (norm alone when there is nothing to add)
struct AddLayerNorm : public torch::autograd::Function<AddLayerNorm> {
    static variable_list forward(AutogradContext *ctx, const Tensor &a, const std::optional<Tensor> &b_,
                                 const Tensor &gamma, const Tensor &beta, double eps) {
        const Tensor b = b_ ? *b_ : Tensor();
        Tensor stats = at::empty({norm_shape(a).rows, 2}, a.options().dtype(at::kFloat));
        auto [sum, norm] = add_norm_plain(a, b, gamma, beta, eps, stats);
        ctx->set_materialize_grads(false);
        ctx->saved_data["add"] = b.defined();
        ctx->save_for_backward({b.defined() ? sum : a, stats, gamma, beta});
        if (b.defined()) return {sum, norm};
        return {norm};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const bool add = ctx->saved_data["add"].toBool();
        const Tensor dsum = add && grads[0].defined() ? grads[0].contiguous() : Tensor();
        if (!grads.back().defined() || (add && !grads[1].defined()))  // the norm was not used
            return {dsum, dsum, Tensor(), Tensor(), Tensor()};
        Tensor dnorm = grads.back().contiguous();
        if (composed(grads)) {  // torch's norm backward, which has a derivative and a batched form
            const variable_list saved = ctx->get_saved_variables();
            const Tensor &x = saved[0];
            std::vector<int64_t> row = x.sizes().vec();
            row.back() = 1;
            const Tensor st = saved[1].detach().t().contiguous();  // means, then reciprocal deviations
            auto [dx, dgamma, dbeta] = at::native_layer_norm_backward(dnorm, x, {x.size(-1)}, st[0].view(row),
                                                                      st[1].view(row), saved[2], saved[3],
                                                                      {true, true, true});
            if (dsum.defined()) dx = dx + dsum;
            return {dx, add ? dx : Tensor(), dgamma, dbeta, Tensor()};
        }
        auto aligned = [](const Tensor &t) { return !t.defined() || aligned16(t) ? t : t.clone(); };
        variable_list saved = ctx->get_saved_variables();
        for (Tensor &t : saved) t = aligned(t.contiguous());  // (saved-tensor hooks may give back another layout)
        const Tensor &x = saved[0], &stats = saved[1], &gamma = saved[2];
        const NormShape s = norm_shape(x);
        Tensor dx = at::empty_like(x), dgamma = at::empty_like(gamma), dbeta = at::empty_like(gamma);
        Tensor ws = workspace(x, hsa_add_layer_norm_bwd_workspace_bytes(s.rows, s.C));
        dnorm = aligned(dnorm);
        const Tensor ds = aligned(dsum);
        c10::DeviceGuard guard(x.device());
        check(hsa_add_layer_norm_bwd(dnorm.data_ptr(), ds.defined() ? ds.data_ptr() : nullptr, x.data_ptr(),
                                     (const float *)stats.data_ptr(), gamma.data_ptr(), dx.data_ptr(), dgamma.data_ptr(),
                                     dbeta.data_ptr(), ws.data_ptr(), ws.nbytes(), s.rows, s.C, s.dtype, stream_of(x)),
              "hsa_add_layer_norm_bwd");
        return {dx, add ? dx : Tensor(), dgamma, dbeta, Tensor()};
    }
};

// (a + b, layer_norm(a + b)), or (None, layer_norm(a)) without b; None where the kernel does not take it
std::optional<std::pair<Tensor, Tensor>> add_layer_norm(const Tensor &a_, const std::optional<Tensor> &b_,
                                                        const Tensor &gamma, const Tensor &beta, double eps) {
    // (before anything is asked for its data pointer)
    if (!ordinary({&a_, &gamma, &beta}) || (b_ && !ordinary({&*b_}))) return std::nullopt;
    if (!a_.is_cuda() || a_.numel() == 0 || !same_kind(a_, gamma) || !same_kind(a_, beta) || gamma.dim() != 1 ||
        gamma.size(0) != a_.size(-1) || beta.sizes() != gamma.sizes() || type_code(a_) < 0 ||
        !hsa_add_layer_norm_ok((int)a_.size(-1), type_code(a_)) || (b_ && (!same_kind(a_, *b_) || b_->sizes() != a_.sizes())) ||
        !gamma.is_contiguous() || !beta.is_contiguous() || !aligned16(gamma) || !aligned16(beta))
        return std::nullopt;
    const Tensor a = a_.contiguous(), b = b_ ? b_->contiguous() : Tensor();
    if (!aligned16(a) || (b.defined() && !aligned16(b))) return std::nullopt;
    if (at::GradMode::is_enabled() && (a.requires_grad() || (b.defined() && b.requires_grad()) || gamma.requires_grad() ||
                                       beta.requires_grad())) {
        variable_list r = AddLayerNorm::apply(a, b.defined() ? std::optional<Tensor>(b) : std::nullopt, gamma, beta, eps);
        return std::make_pair(r.size() == 2 ? r[0] : Tensor(), r.back());
    }
    return add_norm_plain(a, b, gamma, beta, eps, Tensor());
}

// ------------------------------------------------------------------------------- linear projections
// x [.., K] dense, w [N, K] (contract: [K, N]) with dense rows, of one 16-bit type; out: rows of N with the strides
// it has.  batches: x and out are [B, R, ..] whose batch elements lie apart.
bool projectable(const Tensor &x, const Tensor &w, const Tensor &b, bool contract) {
    return ordinary({&x, &w}) && x.is_cuda() && (x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16) && x.numel() > 0 &&
           x.dim() >= 2 && x.is_contiguous() && same_kind(x, w) && w.dim() == 2 && w.is_contiguous() && w.numel() > 0 &&
           x.size(-1) == w.size(contract ? 0 : 1) &&
           (!b.defined() || (same_kind(x, b) && b.dim() == 1 && b.is_contiguous() && b.size(0) == w.size(contract ? 1 : 0)));
}
hsa_linear_segment flat_rows(const Tensor &x, const Tensor &w, const Tensor &b, const Tensor &out, int64_t N) {
    const int64_t K = x.size(-1), rows = x.numel() / K;
    hsa_linear_segment s = {x.data_ptr(), w.data_ptr(), b.defined() ? b.data_ptr() : nullptr, out.data_ptr(), K,
                            w.size(1), N, 0, 0, 1, 0, (int)N};
    s.rows = rows < INT32_MAX ? (int)rows : 0;  // (0: refused)
    return s;
}
// the tile for the segments' products, or -1
int tile_for(const std::vector<hsa_linear_segment> &segs, const Tensor &like, int64_t K, bool contract) {
    return K > (1 << 20) ? -1 : hsa_linear_tile((int)segs.size(), segs.data(), (int)K, contract, type_code(like));
}
void launch_products(const std::vector<hsa_linear_segment> &segs, const Tensor &like, int64_t K, bool contract, int tile) {
    c10::DeviceGuard guard(like.device());
    check(hsa_linear((int)segs.size(), segs.data(), (int)K, contract, tile, type_code(like), stream_of(like)), "hsa_linear");
}

// x w^T + b, or x w + b with `contract`, without autograd: on this library's kernels where they are the faster
// ones, else by torch
Tensor project(const Tensor &x, const Tensor &w, const std::optional<Tensor> &b_, bool contract) {
    const Tensor b = b_ ? *b_ : Tensor();
    if (projectable(x, w, b, contract)) {
        const int64_t K = x.size(-1), N = w.size(contract ? 1 : 0), rows = x.numel() / K;
        const auto result = [&] {
            std::vector<int64_t> size = x.sizes().vec();
            size.back() = N;
            return at::empty(size, x.options());
        };
        // (the choice does not depend on where the result will lie: a tensor of its own begins aligned)
        std::vector<hsa_linear_segment> segs = {flat_rows(x, w, b, x, N)};
        const int tile = tile_for(segs, x, K, contract);
        if (tile >= 0) {
            Tensor out = result();
            segs[0].out = out.data_ptr();
            launch_products(segs, x, K, contract, tile);
            return out;
        }
        if (contract && !b.defined() && K >= 1024 && rows < INT32_MAX && K < INT32_MAX && N < INT32_MAX && N % 8 == 0 &&
            aligned16(w) && hsa_linear_long_pays((int)rows, (int)N, (int)K, type_code(x))) {
            Tensor out = result(), ws = workspace(x, hsa_linear_long_workspace_bytes((int)rows, (int)N, (int)K, type_code(x)));
            c10::DeviceGuard guard(x.device());
            check(hsa_linear_long(x.data_ptr(), K, w.data_ptr(), N, out.data_ptr(), N, (int)rows, (int)N, (int)K, ws.data_ptr(),
                                  ws.nbytes(), type_code(x), stream_of(x)),
                  "hsa_linear_long");
            return out;
        }
    }
    if (contract) return b.defined() ? at::linear(x, w.t(), b) : at::matmul(x, w);
    return at::linear(x, w, b_);
}

// The same of several (x, w), all without bias, in one launch where that pays.
variable_list project_all(const std::vector<std::pair<Tensor, Tensor>> &parts, bool contract) {
    const Tensor &like = parts[0].first;
    const int64_t K = like.size(-1);
    std::vector<hsa_linear_segment> segs;
    for (const auto &[x, w] : parts) {
        if (parts.size() > HSA_LINEAR_MAX_SEGMENTS || !projectable(x, w, Tensor(), contract) || x.size(-1) != K || !same_kind(x, like))
            break;
        segs.push_back(flat_rows(x, w, Tensor(), x, w.size(contract ? 1 : 0)));
    }
    const int tile = segs.size() == parts.size() ? tile_for(segs, like, K, contract) : -1;
    variable_list out;
    for (size_t i = 0; i < parts.size(); ++i) {
        const auto &[x, w] = parts[i];
        if (tile < 0) {
            out.push_back(project(x, w, std::nullopt, contract));
            continue;
        }
        std::vector<int64_t> size = x.sizes().vec();
        size.back() = segs[i].cols;
        out.push_back(at::empty(size, x.options()));
        segs[i].out = out.back().data_ptr();
    }
    if (tile >= 0) launch_products(segs, like, K, contract, tile);
    return out;
}

// ------------------------------------------------------------------ linear projections in training
bool rows_ok(const Tensor &t) {
    return t.dim() == 2 && t.stride(1) == 1 && t.stride(0) >= t.size(1) && t.stride(0) % 8 == 0 && aligned16(t);
}

using Segments = std::vector<std::tuple<Tensor, Tensor, int64_t>>;  // dY [rows, O], X [rows, I], first row of dW

// (dW [O, I], db [O] or undefined) of the sum over the segments of dY^T X, in `type`; nullopt where the
// kernel does not take the operands
std::optional<std::pair<Tensor, Tensor>> weight_grad(const Segments &segs, int64_t O, at::ScalarType type, bool bias) {
    if (segs.empty() || segs.size() > HSA_WEIGHT_GRAD_MAX_SEGMENTS || (bias && segs.size() != 1)) return std::nullopt;
    const Tensor &like = std::get<1>(segs[0]);
    if (!like.is_cuda() || (like.scalar_type() != at::kHalf && like.scalar_type() != at::kBFloat16) ||
        (type != at::kFloat && type != like.scalar_type()))
        return std::nullopt;
    const int64_t I = like.size(-1);
    hsa_weight_grad_segment seg[HSA_WEIGHT_GRAD_MAX_SEGMENTS];
    int n = 0;
    for (const auto &[dy, x, first] : segs) {
        if (!same_kind(like, dy) || !same_kind(like, x) || !rows_ok(dy) || !rows_ok(x) || x.size(1) != I ||
            x.size(0) != dy.size(0))
            return std::nullopt;
        if (x.size(0) == 0) continue;
        seg[n++] = {dy.data_ptr(), x.data_ptr(), dy.stride(0), x.stride(0), x.size(0), (int)dy.size(1), (int)first};
    }
    const size_t bytes = n ? hsa_weight_grad_workspace_bytes(n, seg, (int)I, bias) : 0;
    if (bytes == 0) return std::nullopt;
    Tensor ws = workspace(like, bytes);
    Tensor dw = at::empty({O, I}, like.options().dtype(type)), db = bias ? at::empty({O}, dw.options()) : Tensor();
    c10::DeviceGuard guard(like.device());
    check(hsa_weight_grad(n, seg, (int)O, (int)I, dw.data_ptr(), bias ? db.data_ptr() : nullptr, type_code(dw),
                          ws.data_ptr(), ws.nbytes(), type_code(like), stream_of(like)),
          "hsa_weight_grad");
    return std::make_pair(dw, db);
}

// whether a weight's gradient is small enough for the split-rows kernel to be the faster one
bool small_result(const Tensor &w) { return ((w.size(0) + 127) / 128) * ((w.size(1) + 127) / 128) <= 256; }

// A tensor that a node keeps for its backward without an edge of its own to it.
struct Kept {
    Tensor t;
};

// y = x w^T + b; backward: the weight's and the bias's gradients by the split-rows kernel, straight into the parameters' type.  `w`, `b` are the
// parameters in x's type (the casts that autocast makes); `w` keeps its graph, which a backward that is itself
// differentiated goes through.  The parameter is not saved: under autocast it may be written to before the
// backward.
struct Linear : public torch::autograd::Function<Linear> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &weight, const std::optional<Tensor> &bias,
                          const Kept &w, const std::optional<Tensor> &b) {
        ctx->save_for_backward({x, w.t});
        ctx->saved_data["bias"] = bias.has_value();
        ctx->saved_data["type"] = (int64_t)weight.scalar_type();
        return project(x, w.t, b, false);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const variable_list saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &w = saved[1];
        const bool bias = ctx->saved_data["bias"].toBool();
        const auto type = (at::ScalarType)ctx->saved_data["type"].toInt();  // the parameters'
        const Tensor &g = grads[0];
        Tensor dx, dw, db;
        if (!g.defined()) return {dx, dw, db, Tensor(), Tensor()};
        const Tensor g2 = g.reshape({-1, g.size(-1)}), x2 = x.reshape({-1, x.size(-1)});
        if (ctx->needs_input_grad(0)) dx = composed(grads) ? at::matmul(g, w) : project(g.contiguous(), w, std::nullopt, true);
        const bool need_w = ctx->needs_input_grad(1), need_b = bias && ctx->needs_input_grad(2);
        if (need_w && !composed(grads) && small_result(w)) {
            if (auto r = weight_grad({{g2, x2, 0}}, w.size(0), type, need_b)) {
                dw = r->first;
                db = r->second;
            }
        }
        if (need_w && !dw.defined()) dw = at::mm(g2.t(), x2).to(type);
        if (need_b && !db.defined()) db = g2.sum(0).to(type);
        return {dx, dw, db, Tensor(), Tensor()};
    }
};

// F.linear(x, weight, bias) under the current autocast state; nullopt where nothing is to be gained
// (types other than the 16-bit ones; in training no gradient of the weight or, unless `wide`, a result large
// enough to fill the chip by itself) or where the call is not a plain one.  wide: a vocabulary projection, whose
// input gradient is the long contraction.
std::optional<Tensor> linear(const Tensor &x, const Tensor &weight, const std::optional<Tensor> &bias, bool wide) {
    if (!ordinary({&x, &weight}) || (bias && !ordinary({&*bias}))) return std::nullopt;
    if (!x.is_cuda() || x.dim() < 2 || weight.dim() != 2 || x.numel() == 0 || x.size(-1) != weight.size(1) ||
        x.device() != weight.device() || !weight.is_contiguous())
        return std::nullopt;
    const bool train = at::GradMode::is_enabled() && (x.requires_grad() || weight.requires_grad() || (bias && bias->requires_grad()));
    const int64_t O = weight.size(0), I = weight.size(1);
    if (train && (!weight.requires_grad() || (!wide && (O % 8 || I % 8 || !small_result(weight))))) return std::nullopt;
    if (bias && (bias->dim() != 1 || bias->size(0) != O || !same_kind(weight, *bias))) return std::nullopt;
    const bool cast = at::autocast::is_autocast_enabled(at::kCUDA);
    const at::ScalarType type = cast ? at::autocast::get_autocast_dtype(at::kCUDA) : x.scalar_type();
    if (type != at::kHalf && type != at::kBFloat16) return std::nullopt;
    if (!cast && weight.scalar_type() != type) return std::nullopt;
    if (cast && ((weight.scalar_type() != at::kFloat && weight.scalar_type() != type) || type_code(x) < 0)) return std::nullopt;
    auto as = [&](const Tensor &t) { return cast ? at::autocast::cached_cast(type, t, at::kCUDA) : t; };
    const Kept w{as(weight)};
    if (!train) return project(as(x), w.t, bias ? std::optional<Tensor>(as(*bias)) : std::nullopt, false);
    const std::optional<Tensor> b = bias ? std::optional<Tensor>(as(*bias).detach()) : std::nullopt;
    return Linear::apply(as(x), weight, bias, w, b);
}

// ------------------------------------------------------- queries, keys and values of leaves and nodes
// The rows of x and y [B, N / M, C] converted and joined, as a node: what stands between the joined rows and their
// originals when a backward is itself differentiated.
struct JoinedRows : public torch::autograd::Node {
    int64_t N = 0;
    at::ScalarType x_type = at::kFloat, y_type = at::kFloat;
    variable_list apply(variable_list &&grads) override {
        const Tensor &g = grads[0];
        if (!g.defined()) return {Tensor(), Tensor()};
        return {g.narrow(1, 0, N).to(x_type), g.narrow(1, N, g.size(1) - N).to(y_type)};
    }
};
// where the gradients of x and y go, kept without their data
struct RowEdges : public torch::CustomClassHolder {
    torch::autograd::Edge x, y;
};

// q = x wq^T, k = cat([x, y]) wk^T, v = cat([x, y]) wv^T in the type of `w` (the parameters in the type
// that autocast computes in, with their graph).  The rows are converted once; the backward adds the
// three input gradients in fp32 and hands x and y theirs in their own types.  Only the converted rows are
// saved: the originals may be written to or freed.
struct QueryKeyValueRows : public torch::autograd::Function<QueryKeyValueRows> {
    static variable_list forward(AutogradContext *ctx, const Tensor &x, const Tensor &y, const Tensor &weight_q,
                                 const Tensor &weight_k, const Tensor &weight_v, const Kept &q, const Kept &k,
                                 const Kept &v) {
        const Tensor &wq = q.t, &wk = k.t, &wv = v.t;
        const int B = (int)x.size(0), N = (int)x.size(1), M = (int)y.size(1), C = (int)x.size(2);
        Tensor xy = at::empty({B, N + M, C}, wk.options());
        // rows of x by themselves: x itself where it has the type already
        Tensor xs = x.scalar_type() == xy.scalar_type() ? x : at::empty({B, N, C}, wk.options());
        c10::DeviceGuard guard(x.device());
        check(hsa_pack_rows(x.data_ptr(), y.data_ptr(), xy.data_ptr(), xs.is_same(x) ? nullptr : xs.data_ptr(), B, N, M, C,
                            type_code(x), type_code(y), type_code(xy), stream_of(x)),
              "hsa_pack_rows");
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({xs, xy, wq, wk, wv});
        auto edges = c10::make_intrusive<RowEdges>();
        if (x.requires_grad()) edges->x = torch::autograd::impl::gradient_edge(x);
        if (y.requires_grad()) edges->y = torch::autograd::impl::gradient_edge(y);
        ctx->saved_data["edges"] = c10::IValue::make_capsule(std::move(edges));
        ctx->saved_data["N"] = (int64_t)N;
        ctx->saved_data["types"] = std::vector<int64_t>{(int64_t)x.scalar_type(), (int64_t)y.scalar_type(), (int64_t)weight_k.scalar_type()};
        return project_all({{xs, wq}, {xy, wk}, {xy, wv}}, false);
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const variable_list saved = ctx->get_saved_variables();
        const Tensor *w = &saved[2];
        Tensor xs = saved[0].contiguous(), xy = saved[1].contiguous();
        const int64_t N = ctx->saved_data["N"].toInt(), B = xy.size(0), M = xy.size(1) - N, C = xy.size(2);
        const std::vector<int64_t> types = ctx->saved_data["types"].toIntVector();
        const auto x_type = (at::ScalarType)types[0], y_type = (at::ScalarType)types[1], w_type = (at::ScalarType)types[2];
        const bool by_torch = composed(grads);
        if (at::GradMode::is_enabled()) {  // itself differentiated: the rows' graph leads to x and y
            const auto edges = c10::static_intrusive_pointer_cast<RowEdges>(ctx->saved_data["edges"].toCapsule());
            xy = xy.detach();
            if (edges->x.is_valid() || edges->y.is_valid()) {
                auto join = std::shared_ptr<JoinedRows>(new JoinedRows(), torch::autograd::deleteNode);
                join->N = N;
                join->x_type = x_type;
                join->y_type = y_type;
                join->set_next_edges({edges->x, edges->y});
                torch::autograd::set_history(xy, join);
            }
            xs = xy.narrow(1, 0, N);
        }
        const bool need_x = ctx->needs_input_grad(0), need_y = ctx->needs_input_grad(1);
        Tensor dx, dy, dw[3], d[3];  // d: input gradients of the three projections
        if (!by_torch && need_x && grads[0].defined() && grads[1].defined() && grads[2].defined()) {
            const auto rows = [](const Tensor &g) { return g.reshape({-1, g.size(-1)}).contiguous(); };
            const variable_list r = project_all({{rows(grads[0]), w[0]}, {rows(grads[1]), w[1]}, {rows(grads[2]), w[2]}}, true);
            for (int i = 0; i < 3; ++i) d[i] = r[i];
        }
        for (int i = 0; i < 3; ++i) {
            const Tensor &g = grads[i];
            if (!g.defined()) continue;
            const Tensor g2 = g.reshape({-1, g.size(-1)}), r2 = (i == 0 ? xs : xy).reshape({-1, C});
            if (!d[i].defined() && (i == 0 ? need_x : need_x || need_y)) d[i] = at::mm(g2, w[i]);
            if (!ctx->needs_input_grad(2 + i)) continue;
            if (!by_torch)
                if (auto r = weight_grad({{g2, r2, 0}}, g2.size(1), w_type, false)) dw[i] = r->first;
            if (!dw[i].defined()) dw[i] = at::mm(g2.t(), r2).to(w_type);
        }
        if (!by_torch && d[1].defined() && d[2].defined()) {
            if (need_x) dx = at::empty({B, N, C}, xy.options().dtype(x_type));
            if (need_y) dy = at::empty({B, M, C}, xy.options().dtype(y_type));
            c10::DeviceGuard guard(xy.device());
            check(hsa_add_split_rows(d[1].data_ptr(), d[2].data_ptr(), d[0].defined() ? d[0].data_ptr() : nullptr,
                                     need_x ? dx.data_ptr() : nullptr, need_y ? dy.data_ptr() : nullptr, (int)B, (int)N,
                                     (int)M, (int)C, type_code(x_type), type_code(y_type), type_code(xy), stream_of(xy)),
                  "hsa_add_split_rows");
        } else {
            Tensor t;  // in fp32
            for (int i = 1; i < 3; ++i)
                if (d[i].defined()) t = t.defined() ? t + d[i].to(at::kFloat) : d[i].to(at::kFloat);
            if (t.defined()) {
                t = t.reshape({B, N + M, C});
                dx = t.narrow(1, 0, N);
                dy = t.narrow(1, N, M).to(y_type);
            }
            if (d[0].defined()) dx = dx.defined() ? dx + d[0].reshape({B, N, C}).to(at::kFloat) : d[0].reshape({B, N, C});
            if (dx.defined()) dx = dx.to(x_type);
        }
        return {dx, dy, dw[0], dw[1], dw[2], Tensor(), Tensor(), Tensor()};
    }
};

// The element type in which the three projections of the rows of x [B, N, C] and y [B, M, C] compute under the current
// autocast state; nullopt where the call is not a plain one on 16-bit types.
std::optional<at::ScalarType> rows_type(const Tensor &x, const Tensor &y, const Tensor &weight_q, const Tensor &weight_k,
                                        const Tensor &weight_v) {
    if (!ordinary({&x, &y, &weight_q, &weight_k, &weight_v})) return std::nullopt;
    if (x.dim() != 3 || y.dim() != 3 || x.numel() == 0 || y.numel() == 0 || x.device() != y.device() || y.size(0) != x.size(0) || y.size(2) != x.size(2) || weight_k.device() != x.device() ||
        weight_k.dim() != 2 || weight_k.size(1) != x.size(2))
        return std::nullopt;
    for (const Tensor *t : {&weight_q, &weight_k, &weight_v})
        if (!same_kind(weight_k, *t) || t->sizes() != weight_k.sizes() || !t->is_contiguous()) return std::nullopt;
    const int64_t O = weight_k.size(0), C = weight_k.size(1);
    if (O % 8 || C % 8 || ((O + 127) / 128) * ((C + 127) / 128) > 256 || x.numel() + y.numel() > (int64_t)1 << 40 ||
        x.size(1) + y.size(1) > (1 << 30))
        return std::nullopt;
    const bool cast = at::autocast::is_autocast_enabled(at::kCUDA);
    const at::ScalarType type = cast ? at::autocast::get_autocast_dtype(at::kCUDA) : x.scalar_type();
    if (type != at::kHalf && type != at::kBFloat16) return std::nullopt;
    for (const Tensor *t : {&x, &y, &weight_k})
        if (t->scalar_type() != type && !(cast && t->scalar_type() == at::kFloat)) return std::nullopt;
    return type;
}

// (queries of the rows of x [B, N, C]; keys, values of those and of y [B, M, C]) under the current autocast
// state; nullopt where the call is not a plain one in training on 16-bit types
std::optional<std::tuple<Tensor, Tensor, Tensor>> query_key_value_rows(const Tensor &x, const Tensor &y,
                                                                       const Tensor &weight_q, const Tensor &weight_k,
                                                                       const Tensor &weight_v) {
    if (!at::GradMode::is_enabled() || !x.is_cuda()) return std::nullopt;
    for (const Tensor *t : {&weight_q, &weight_k, &weight_v})
        if (!t->requires_grad()) return std::nullopt;
    const std::optional<at::ScalarType> type = rows_type(x, y, weight_q, weight_k, weight_v);
    if (!type) return std::nullopt;
    const Tensor xc = x.contiguous(), yc = y.contiguous();
    if (!aligned16(xc) || !aligned16(yc)) return std::nullopt;
    const bool cast = at::autocast::is_autocast_enabled(at::kCUDA);
    auto as = [&](const Tensor &t) { return Kept{cast ? at::autocast::cached_cast(*type, t, at::kCUDA) : t}; };
    variable_list r = QueryKeyValueRows::apply(xc, yc, weight_q, weight_k, weight_v, as(weight_q), as(weight_k), as(weight_v));
    return std::make_tuple(r[0], r[1], r[2]);
}

// The same without autograd: the rows stay where they are, every projection writes its part of the results, in one
// launch.  rows_plan: the products (their results to be filled in) and their tile, -1 where that does not pay; it
// depends on sizes and strides only.
using Three = std::optional<std::tuple<Tensor, Tensor, Tensor>>;
std::pair<std::vector<hsa_linear_segment>, int> rows_plan(const Tensor &x, const Tensor &y, const Tensor &wq, const Tensor &wk,
                                                          const Tensor &wv) {
    if (!projectable(x, wq, Tensor(), false) || !projectable(x, wk, Tensor(), false) || !projectable(x, wv, Tensor(), false) ||
        !projectable(y, wk, Tensor(), false))
        return {{}, -1};
    const int64_t B = x.size(0), N = x.size(1), M = y.size(1), O = wk.size(0);
    if (N + M > (1 << 28) || B > (1 << 24)) return {{}, -1};
    const auto rows = [&](const Tensor &in, const Tensor &w, int64_t out_rows) {
        hsa_linear_segment s = flat_rows(in, w, Tensor(), in, O);
        s.batches = (int)B;
        s.rows = (int)in.size(1);
        s.batch_x = in.stride(0);
        s.batch_out = out_rows * O;
        return s;
    };
    std::vector<hsa_linear_segment> segs = {rows(x, wq, N), rows(x, wk, N + M), rows(x, wv, N + M), rows(y, wk, N + M), rows(y, wv, N + M)};
    const int tile = O % 8 ? -1 : tile_for(segs, x, x.size(2), false);
    return {std::move(segs), tile};
}
Three query_key_value_plain(const Tensor &x, const Tensor &y, const Tensor &wq, const Tensor &wk, const Tensor &wv) {
    auto [segs, tile] = rows_plan(x, y, wq, wk, wv);
    if (tile < 0) return std::nullopt;
    const int64_t B = x.size(0), N = x.size(1), M = y.size(1), O = wk.size(0);
    Tensor q = at::empty({B, N, O}, x.options()), k = at::empty({B, N + M, O}, x.options()), v = at::empty_like(k);
    const int64_t nodes = N * O * q.element_size();
    segs[0].out = q.data_ptr();
    segs[1].out = k.data_ptr();
    segs[2].out = v.data_ptr();
    segs[3].out = (char *)k.data_ptr() + nodes;
    segs[4].out = (char *)v.data_ptr() + nodes;
    launch_products(segs, x, x.size(2), false, tile);
    return std::make_tuple(q, k, v);
}

Three query_key_value(const Tensor &x, const Tensor &y, const Tensor &weight_q, const Tensor &weight_k, const Tensor &weight_v) {
    if (!x.is_cuda()) return std::nullopt;
    if (at::GradMode::is_enabled())
        for (const Tensor *t : {&x, &y, &weight_q, &weight_k, &weight_v})
            if (t->requires_grad()) return std::nullopt;
    const std::optional<at::ScalarType> type = rows_type(x, y, weight_q, weight_k, weight_v);
    if (!type) return std::nullopt;
    const bool cast = at::autocast::is_autocast_enabled(at::kCUDA);
    auto as = [&](const Tensor &t) { return cast ? at::autocast::cached_cast(*type, t, at::kCUDA) : t; };
    return query_key_value_plain(x.to(*type).contiguous(), y.to(*type).contiguous(), as(weight_q), as(weight_k), as(weight_v));
}

// ------------------------------------------------------------------------------- one layer of the model
// the whole span-node update as one chain of fused levels, the norms on their kernel
bool layer_kind(const Tensor &x, int64_t heads) {
    if (at::GradMode::is_enabled() || at::autocast::is_autocast_enabled(at::kCUDA) || !x.is_cuda() || x.dim() != 3 || x.numel() == 0 ||
        (x.scalar_type() != at::kHalf && x.scalar_type() != at::kBFloat16) || heads < 1 || heads > (1 << 16))
        return false;
    const int64_t B = x.size(0), N = x.size(1), C = x.size(2);
    return B <= (1 << 20) && N >= 2 && N <= (1 << 24) && log2_exact(N) >= 0 && C % heads == 0 && C <= (1 << 16) &&
           hsa_cross_update_level_rows((int)B, (int)heads, (int)(C / heads), type_code(x)) >= N && hsa_add_layer_norm_ok((int)C, type_code(x));
}
// larger inputs whose rows' products do not go into one launch stay with the Python layer, which has a way without the
// copy for the largest and whose host time is small against their kernels'
bool layer_rows(const Tensor &x, const Tensor &y, const Tensor &wq, const Tensor &wk, const Tensor &wv) {
    return x.numel() < 1 << 20 || rows_plan(x, y, wq, wk, wv).second >= 0;
}
// Whether a layer of these sizes is one that decoder_layer takes, asked before its modules are looked at one by one (a
// forward of B2 N1024, two layers of 4 heads by 128 channels, which it does not take: 905 us when that is found out last,
// 845 here, 815 without the native layer; since then 818 -> 748 with the rows joined by a copy)
bool decoder_layer_takes(const Tensor &x, const Tensor &y, const Tensor &w, int64_t heads) {
    return layer_kind(x, heads) && ordinary({&x, &y, &w}) && y.dim() == 3 && y.numel() > 0 && y.size(0) == x.size(0) && layer_rows(x, y, w, w, w);
}

// A decoder layer without autograd, dropout and autocast on 16-bit tensors, launch for launch what the Python
// layer does: a short sequence's layer is 15 to 25 launches of a few us each, and through Python they take
// 170 us to enqueue (six layers of B1 N256: 1056 us a forward against 700 us of kernels).
//   x [B, N, C], y [B, N-1, C], nx = norm1(x), ny = norm_y(y); p: the parameters in the order of LayerParams
// Returns x, y and, with `following`, the next layer's norms of them; nullopt before anything is launched where
// the layer is not of this kind.
enum LayerParams { W_QKV_Y, W_KV_Y_PACKED, OUT_Y_W, OUT_Y_B, Q_X, K_X, V_X, OUT_X_W, OUT_X_B, NORM2_W, NORM2_B, FC1_W, FC1_B,
                   FC2_W, FC2_B, NORM_Y_W, NORM_Y_B, NORM1_W, NORM1_B };
std::optional<std::tuple<Tensor, Tensor, Tensor, Tensor>> decoder_layer(const Tensor &x, const Tensor &y, const Tensor &nx, const Tensor &ny,
                                                                        const std::vector<Tensor> &p, const std::vector<double> &eps,
                                                                        int64_t heads, int64_t window, bool causal, bool gelu,
                                                                        bool following) {
    if (!layer_kind(x, heads) || p.size() != (following ? NORM1_B + 1 : NORM_Y_W) || eps.size() != 3 || window < 0 || window > (1 << 20))
        return std::nullopt;
    const int64_t B = x.size(0), N = x.size(1), C = x.size(2);
    const int H = (int)heads, Dh = (int)(C / heads), code = type_code(x);
    if (!ordinary({&x, &y, &nx, &ny})) return std::nullopt;
    for (const Tensor *t : {&x, &y, &nx, &ny})
        if (!same_kind(x, *t) || t->dim() != 3 || !t->is_contiguous() || !aligned16(*t)) return std::nullopt;
    if (nx.sizes() != x.sizes() || y.size(0) != B || y.size(1) != N - 1 || y.size(2) != C || ny.sizes() != y.sizes()) return std::nullopt;
    for (const Tensor &t : p)
        if (!ordinary({&t}) || !same_kind(x, t) || !t.is_contiguous() || !aligned16(t)) return std::nullopt;
    const int64_t F = p[FC1_W].size(0);
    const auto matrix = [&](int i, int64_t rows, int64_t cols) { return p[i].dim() == 2 && p[i].size(0) == rows && p[i].size(1) == cols; };
    const auto row = [&](int i, int64_t n) { return p[i].dim() == 1 && p[i].size(0) == n; };
    if (!matrix(W_QKV_Y, 3 * C, C) || p[W_KV_Y_PACKED].numel() != 2 * C * C || !matrix(OUT_Y_W, C, C) || !row(OUT_Y_B, C) ||
        !matrix(Q_X, C, C) || !matrix(K_X, C, C) || !matrix(V_X, C, C) || !matrix(OUT_X_W, C, C) || !row(OUT_X_B, C) ||
        !row(NORM2_W, C) || !row(NORM2_B, C) || p[FC1_W].dim() != 2 || !matrix(FC1_W, F, C) || !row(FC1_B, F) || !matrix(FC2_W, C, F) ||
        !row(FC2_B, C))
        return std::nullopt;
    for (int i = NORM_Y_W; following && i <= NORM1_B; ++i)
        if (!row(i, C)) return std::nullopt;
    if (!layer_rows(nx, y, p[Q_X], p[K_X], p[V_X])) return std::nullopt;

    c10::DeviceGuard guard(x.device());
    // span nodes: the three projections, every level of the tree, the output projection, the residual
    const Tensor qkv = project(ny, p[W_QKV_Y], std::nullopt, false);
    Tensor nodes = at::empty({B, N - 1, C}, x.options());
    check(hsa_cross_update_top_fwd(x.data_ptr(), qkv.data_ptr(), p[W_KV_Y_PACKED].data_ptr(), nodes.data_ptr(), (int)B, (int)N, H, Dh, 0,
                                   (N - 1) * 3 * C, 3 * C, (N - 1) * C, C, code, stream_of(x)),
          "hsa_cross_update_top_fwd");
    const Tensor u = project(nodes, p[OUT_Y_W], p[OUT_Y_B], false);
    Tensor y2, ny2;
    if (following) std::tie(y2, ny2) = add_norm_plain(y, u, p[NORM_Y_W], p[NORM_Y_B], eps[1], Tensor());
    else y2 = at::add(y, u);
    // leaves: queries, keys and values of leaves and nodes, the attention, the output projection, the residual
    Tensor q, k, v;
    if (const Three r = query_key_value_plain(nx, y2, p[Q_X], p[K_X], p[V_X])) {
        std::tie(q, k, v) = *r;
    } else {
        q = project(nx, p[Q_X], std::nullopt, false);
        const Tensor xy = at::cat({nx, y2}, 1);
        k = project(xy, p[K_X], std::nullopt, false);
        v = project(xy, p[V_X], std::nullopt, false);
    }
    const auto split = [&](const Tensor &t) { return t.view({B, t.size(1), heads, Dh}); };
    const Tensor a = attention_plain(split(q), split(k), split(v), causal, (int)window).view({B, N, C});
    const Tensor o = project(a, p[OUT_X_W], p[OUT_X_B], false);
    auto [x2, n2] = add_norm_plain(x, o, p[NORM2_W], p[NORM2_B], eps[0], Tensor());
    // feed-forward
    const Tensor hidden = project(n2, p[FC1_W], p[FC1_B], false);
    const Tensor f = project(gelu ? at::gelu(hidden) : at::relu(hidden), p[FC2_W], p[FC2_B], false);
    if (!following) return std::make_tuple(at::add(x2, f), y2, Tensor(), Tensor());
    auto [x3, nx3] = add_norm_plain(x2, f, p[NORM1_W], p[NORM1_B], eps[2], Tensor());
    return std::make_tuple(x3, y2, nx3, ny2);
}

}  // namespace

PYBIND11_MODULE(_hsa_torch, m) {
    py::register_exception_translator([](std::exception_ptr p) {
        try {
            if (p) std::rethrow_exception(p);
        } catch (const LibraryError &e) {
            PyErr_SetString(py::module_::import("sparseattention_amd._lib").attr("HsaError").ptr(), e.what());
        }
    });
    m.def("span_attention", &span_attention);
    m.def("build_tree", &build_tree);
    m.def("add_layer_norm", &add_layer_norm);
    m.def("linear", &linear);
    m.def("project", &project);
    m.def("weight_grad", &weight_grad);
    m.def("query_key_value_rows", &query_key_value_rows);
    m.def("query_key_value", &query_key_value);
    m.def("decoder_layer_takes", &decoder_layer_takes);
    m.def("decoder_layer", &decoder_layer);
}
