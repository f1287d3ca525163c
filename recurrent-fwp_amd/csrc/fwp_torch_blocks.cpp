// The Delta-Net language model's blocks as C++ autograd functions over the C ABI: the feed-forward block, the
// Delta-Net layer's projections around the delta rule, LayerNorm, and the softmax's negative log-likelihood
// (reference: language_modeling/src/utils/model_utils.py:34-67, cuda_fast_weight_layer.py:57-188,
// model_main.py:1333-1361).  Biases, ReLU and its mask, residual additions and bias gradients happen inside the
// matrix products (fwp_matmul's epilogue), so a block is its products and nothing else.  Host code only.
//
// A backward pass that is itself to be differentiated (create_graph) recomputes the block from PyTorch's own
// operators and differentiates that.
#include "fwp_torch.hpp"

#include <optional>
#include <tuple>
#include <utility>
#include <vector>

namespace {

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

at::Tensor given(const std::optional<at::Tensor> &t) { return t.has_value() ? *t : at::Tensor(); }

float *ptr(const at::Tensor &t) { return t.defined() ? t.data_ptr<float>() : nullptr; }

// fp32, contiguous, 16-byte aligned
at::Tensor plain(const at::Tensor &t) {
    if (t.scalar_type() != at::kFloat) fail("fp32 tensors only");
    if (!t.is_contiguous()) return t.contiguous();
    return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 ? t.clone() : t;
}

// The kernels get addresses and sizes: every block compares its tensors' sizes before it hands them on.
bool optional_of(const at::Tensor &t, int64_t n) { return !t.defined() || same_shape(t, {n}); }
bool ends_in(const at::Tensor &x, int64_t n) { return x.dim() > 0 && x.size(-1) == n; }

// C = op(A) op(B) with an epilogue, shaped `shape` (M x N elements)
at::Tensor matmul(int layout, const at::Tensor &A, const at::Tensor &B, int64_t M, int64_t N, int64_t K, at::IntArrayRef shape,
                  const fwp_mm_epilogue &epi = {}) {
    at::Tensor C = at::empty(shape, A.options()), work;
    const int64_t n = fwp_product_workspace((int)M, (int)N, (int)K);
    if (n > 0) work = at::empty({n}, A.options());
    check(fwp_matmul(layout, ptr(A), layout == FWP_MM_TN ? M : K, ptr(B), layout == FWP_MM_NT ? K : N, ptr(C), N, (int)M,
                     (int)N, (int)K, &epi, ptr(work), stream_of(A)),
          "fwp_matmul");
    return C;
}

// Gradients of the weights of y = x W^T + bias from g = dy: g^T x, and the columns of g summed
at::Tensor weight_grad(const at::Tensor &g, const at::Tensor &x, int64_t rows, int64_t out, int64_t in, float *colsum) {
    fwp_mm_epilogue e{};
    e.colsum = colsum;
    return matmul(FWP_MM_TN, g, x, out, in, rows, {out, in}, e);
}

at::Tensor bias_like(int64_t n, const at::Tensor &x, bool want) { return want ? at::empty({n}, x.options()) : at::Tensor(); }

variable_list differentiate(const at::Tensor &y, const variable_list &inputs, const at::Tensor &g) {
    variable_list used, res(inputs.size());
    for (const at::Tensor &t : inputs)
        if (t.defined() && t.requires_grad()) used.push_back(t);
    if (used.empty()) return res;
    const variable_list grads = torch::autograd::grad({y}, used, {g}, std::nullopt, /*create_graph=*/true, /*allow_unused=*/true);
    for (size_t i = 0, j = 0; i < inputs.size(); i++)
        if (inputs[i].defined() && inputs[i].requires_grad()) res[i] = grads[j++];
    return res;
}

// ------------------------------------------------------------------ y = x W^T (+ bias) (relu)

struct LinearFn : torch::autograd::Function<LinearFn> {
    static at::Tensor forward(AutogradContext *ctx, const at::Tensor &x_in, const at::Tensor &W,
                              const std::optional<at::Tensor> &bias_in, bool relu) {
        const at::Tensor bias = given(bias_in);
        require_device(x_in);
        same_device(x_in, {W, bias});
        require(W.dim() == 2 && W.numel() > 0 && x_in.numel() > 0 && ends_in(x_in, W.size(1)) && optional_of(bias, W.size(0)),
                "x, weight and bias do not fit one another");
        const int64_t in = W.size(1), out = W.size(0), rows = x_in.numel() / in;
        const at::Tensor x = plain(x_in);
        std::vector<int64_t> shape = x.sizes().vec();
        shape.back() = out;
        LaunchGuard guard(x);
        fwp_mm_epilogue e{};
        e.bias = ptr(bias);
        e.relu = relu;
        at::Tensor y;
        if (rows <= 64 && in >= 64 && in % 64 == 0) {       // few rows: latency counts (fwp_decode.hip)
            y = at::empty(shape, x.options());
            const at::Tensor w = plain(W);
            check(fwp_rows_matmul(ptr(x), nullptr, nullptr, 0.f, nullptr, ptr(w), ptr(bias), nullptr, relu, ptr(y), (int)rows, (int)out,
                                  (int)in, stream_of(x)),
                  "fwp_rows_matmul");
        } else {
            y = matmul(FWP_MM_NT, x, W, rows, out, in, shape, e);
        }
        if (ctx) {
            ctx->save_for_backward({x_in, W, bias, relu ? y : at::Tensor()});
            ctx->set_materialize_grads(false);
        }
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const at::Tensor &W = saved[1], &bias = saved[2], &y = saved[3];
        if (!grads[0].defined()) return variable_list(4);
        if (at::GradMode::is_enabled()) {
            at::Tensor z = at::linear(saved[0], W, bias.defined() ? std::optional<at::Tensor>(bias) : std::nullopt);
            variable_list res = differentiate(y.defined() ? at::relu(z) : z, {saved[0], W, bias}, grads[0]);
            res.resize(4);
            return res;
        }
        const at::Tensor x = plain(saved[0]);
        at::Tensor g = plain(grads[0]);
        if (y.defined()) g = at::threshold_backward(g, y, 0);
        const int64_t in = W.size(1), out = W.size(0), rows = x.numel() / in;
        LaunchGuard guard(x);
        variable_list res(4);
        if (ctx->needs_input_grad(0)) res[0] = matmul(FWP_MM_NN, g, W, rows, in, out, saved[0].sizes());
        const bool want_bias = bias.defined() && ctx->needs_input_grad(2);
        res[2] = bias_like(out, x, want_bias);
        if (ctx->needs_input_grad(1) || want_bias) res[1] = weight_grad(g, x, rows, out, in, ptr(res[2]));
        return res;
    }
};

// ------------------------------------------------------------------ s = relu(x W1^T + b1) W2^T + b2 (+ residual)

struct FeedForwardFn : torch::autograd::Function<FeedForwardFn> {
    // residual: undefined, or added; `same`: it is x (its gradient then joins x's inside the last product)
    static at::Tensor forward(AutogradContext *ctx, const at::Tensor &x_in, const at::Tensor &W1, const at::Tensor &b1,
                              const at::Tensor &W2, const at::Tensor &b2, const std::optional<at::Tensor> &residual_in,
                              bool same) {
        const at::Tensor residual = given(residual_in);
        require_device(x_in);
        same_device(x_in, {W1, b1, W2, b2, residual});
        require(W1.dim() == 2 && W1.numel() > 0 && x_in.numel() > 0 && ends_in(x_in, W1.size(1)) && same_shape(b1, {W1.size(0)}) &&
                    same_shape(W2, {W1.size(1), W1.size(0)}) && same_shape(b2, {W1.size(1)}) &&
                    (!residual.defined() || residual.sizes() == x_in.sizes()),
                "x, weights, biases and residual do not fit one another");
        const int64_t d = W1.size(1), inner = W1.size(0), rows = x_in.numel() / d;
        const at::Tensor x = plain(x_in), res = same ? x : residual.defined() ? plain(residual) : residual;
        LaunchGuard guard(x);
        fwp_mm_epilogue e{};
        e.bias = ptr(b1);
        e.relu = 1;
        const at::Tensor hid = matmul(FWP_MM_NT, x, W1, rows, inner, d, {rows, inner}, e);
        e = {};
        e.bias = ptr(b2);
        e.residual = ptr(res);
        const at::Tensor s = matmul(FWP_MM_NT, hid, W2, rows, d, inner, x_in.sizes(), e);
        if (ctx) {
            ctx->save_for_backward({x_in, W1, b1, W2, b2, hid});
            ctx->saved_data["same"] = same;
            ctx->saved_data["residual"] = residual.defined();
            ctx->set_materialize_grads(false);
        }
        return s;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list res(7);
        if (!grads[0].defined()) return res;
        const auto saved = ctx->get_saved_variables();
        const at::Tensor &W1 = saved[1], &b1 = saved[2], &W2 = saved[3], &b2 = saved[4], &hid = saved[5];
        const bool same = ctx->saved_data["same"].toBool();
        if (ctx->saved_data["residual"].toBool() && !same) res[5] = grads[0];
        if (at::GradMode::is_enabled()) {
            at::Tensor s = at::linear(at::relu(at::linear(saved[0], W1, b1)), W2, b2);
            const variable_list g = differentiate(same ? s + saved[0] : s, {saved[0], W1, b1, W2, b2}, grads[0]);
            std::copy(g.begin(), g.end(), res.begin());
            return res;
        }
        const at::Tensor x = plain(saved[0]), g = plain(grads[0]);
        const int64_t d = W1.size(1), inner = W1.size(0), rows = x.numel() / d;
        LaunchGuard guard(x);
        res[4] = bias_like(d, x, ctx->needs_input_grad(4));
        if (ctx->needs_input_grad(3) || res[4].defined()) res[3] = weight_grad(g, hid, rows, d, inner, ptr(res[4]));
        if (!(ctx->needs_input_grad(0) || ctx->needs_input_grad(1) || ctx->needs_input_grad(2))) return res;
        fwp_mm_epilogue e{};
        e.gate = ptr(hid);      // the ReLU's gradient: where the activation is positive
        const at::Tensor gh = matmul(FWP_MM_NN, g, W2, rows, inner, d, {rows, inner}, e);
        res[2] = bias_like(inner, x, ctx->needs_input_grad(2));
        if (ctx->needs_input_grad(1) || res[2].defined()) res[1] = weight_grad(gh, x, rows, inner, d, ptr(res[2]));
        if (ctx->needs_input_grad(0)) {
            e = {};
            e.residual = same ? ptr(g) : nullptr;
            res[0] = matmul(FWP_MM_NN, gh, W1, rows, d, inner, saved[0].sizes(), e);
        }
        return res;
    }
};

// ------------------------------------------------------------------ s = (x +) o_net(delta rule(qkvb_net(x)))

// The gradient of the projection qkvb from that of the delta rule's read-out, go [T,B,H,D]
at::Tensor projection_grad(const at::Tensor &go, const at::Tensor &qkvb, const at::Tensor &q, const at::Tensor &k, const at::Tensor &beta,
                           const at::Tensor &buf, double scale) {
    const int64_t B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3), rows = T * B;
    void *const s = stream_of(go);
    Parts parts({rows * H * D, rows * H * D, rows * H * D, rows * H}, go.options());
    const at::Tensor gq = parts.take(B, H, T, D), gk = parts.take(B, H, T, D), gv = parts.take(B, H, T, D), gb = parts.take(B, H, T, 1);
    const float *vdiff = ptr(buf), *ckpt = vdiff + rows * H * D;
    const fwp_view gov = {ptr(go), H * D, D, B * H * D};
    const int chunk = fwp_query(FWP_Q_DEFAULT_CHUNK);
    const at::Tensor work = segment_work(B, H, T, D, D, chunk, go.options(), true);
    check(fwp_delta_bwd_segments(view_of(q), view_of(k), view_of(beta), vdiff, gov, ckpt, ptr(gq), ptr(gk), ptr(gv), ptr(gb), ptr(work), (int)B,
                                 (int)H, (int)T, (int)D, (int)D, chunk, s),
          "fwp_delta_bwd_segments");
    const at::Tensor gp = at::empty_like(qkvb);
    check(fwp_deltanet_prep_bwd(ptr(qkvb), ptr(gq), ptr(gk), ptr(gv), ptr(gb), ptr(gp), (int)T, (int)B, (int)H, (int)D, (float)scale, s),
          "fwp_deltanet_prep_bwd");
    return gp;
}

// The read-out [T,B,H,D] that a DeltaBlockFn's forward pass left, as a function of its x and Wqkvb again: with create_graph the
// gradient of Wo is a product with it.
struct DeltaReadOutFn : torch::autograd::Function<DeltaReadOutFn> {
    static at::Tensor forward(AutogradContext *ctx, const at::Tensor &x, const at::Tensor &Wqkvb, const at::Tensor &qkvb, const at::Tensor &q,
                              const at::Tensor &k, const at::Tensor &beta, const at::Tensor &buf, const at::Tensor &out, double scale) {
        ctx->save_for_backward({x, Wqkvb, qkvb, q, k, beta, buf});
        ctx->saved_data["scale"] = scale;
        return out.detach();
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const at::Tensor &x = saved[0], &Wqkvb = saved[1], go = plain(grads[0]);
        LaunchGuard guard(go);
        const at::Tensor gp = projection_grad(go, saved[2], saved[3], saved[4], saved[5], saved[6], ctx->saved_data["scale"].toDouble());
        variable_list res(9);
        if (ctx->needs_input_grad(0)) res[0] = at::matmul(gp, Wqkvb);
        if (ctx->needs_input_grad(1)) res[1] = at::matmul(gp.flatten(0, 1).t(), x.reshape({-1, x.size(2)}));
        return res;
    }
};

struct DeltaBlockFn : torch::autograd::Function<DeltaBlockFn> {
    // x [T,B,d]; Wqkvb [H (3D+1), d]; Wo [d, H D]; state [B,H,D,D] in/out (fresh: out, from zeros)
    static at::Tensor forward(AutogradContext *ctx, const at::Tensor &x_in, const at::Tensor &Wqkvb, const at::Tensor &Wo,
                              const at::Tensor &state, int64_t H, int64_t D, double scale, bool residual, bool fresh) {
        require_device(x_in);
        same_device(x_in, {Wqkvb, Wo, state});
        require(x_in.dim() == 3, "expected [len, bsz, d_model]");
        const int64_t T = x_in.size(0), B = x_in.size(1), d = x_in.size(2), rows = T * B, width = H * (3 * D + 1);
        require(x_in.numel() > 0 && same_shape(Wqkvb, {width, d}) && same_shape(Wo, {d, H * D}) && same_shape(state, {B, H, D, D}),
                "projections and state do not fit the heads");
        require_state(state, "W");
        const at::Tensor x = plain(x_in);
        const auto opts = x.options();
        LaunchGuard guard(x);
        void *const s = stream_of(x);
        const at::Tensor qkvb = matmul(FWP_MM_NT, x, Wqkvb, rows, width, d, {T, B, width});
        Parts parts({rows * H * D, rows * H * D, rows * H * D, rows * H}, opts);
        const at::Tensor q = parts.take(B, H, T, D), k = parts.take(B, H, T, D), v = parts.take(B, H, T, D),
                         beta = parts.take(B, H, T, 1);
        if (fresh)
            check(fwp_deltanet_prep_start(ptr(qkvb), ptr(q), ptr(k), ptr(v), ptr(beta), ptr(state), (int)T, (int)B, (int)H, (int)D, (float)scale, s),
                  "fwp_deltanet_prep_start");
        else
            check(fwp_deltanet_prep_fwd(ptr(qkvb), ptr(q), ptr(k), ptr(v), ptr(beta), (int)T, (int)B, (int)H, (int)D, (float)scale, s),
                  "fwp_deltanet_prep_fwd");
        const at::Tensor out = at::empty({T, B, H, D}, opts);
        const fwp_out_view ov = {ptr(out), H * D, D, B * H * D};
        const int chunk = fwp_query(FWP_Q_DEFAULT_CHUNK);
        at::Tensor saved;
        float *vdiff = nullptr, *ckpt = nullptr;
        if (ctx) {
            const int64_t n_vdiff = rows * H * D, n_ckpt = fwp_delta_ckpt_floats((int)B, (int)H, (int)T, (int)D, (int)D, chunk);
            if (n_ckpt < 0) fail("invalid dimensions");
            saved = at::empty({n_vdiff + n_ckpt}, opts);
            vdiff = ptr(saved);
            ckpt = vdiff + n_vdiff;
        }
        const at::Tensor work = segment_work(B, H, T, D, D, chunk, opts, false);
        check(fwp_delta_fwd_segments(view_of(q), view_of(k), view_of(v), view_of(beta), ptr(state), ov, vdiff, ckpt, ptr(work), (int)B,
                                     (int)H, (int)T, (int)D, (int)D, chunk, s),
              "fwp_delta_fwd_segments");
        fwp_mm_epilogue e{};
        e.residual = residual ? ptr(x) : nullptr;
        const at::Tensor y = matmul(FWP_MM_NT, out, Wo, rows, d, H * D, x_in.sizes(), e);
        if (ctx) {
            ctx->save_for_backward({x_in, Wqkvb, Wo, qkvb, q, k, beta, saved, out});
            ctx->saved_data["scale"] = scale;
            ctx->saved_data["residual"] = residual;
            ctx->set_materialize_grads(false);
        }
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list res(9);
        if (!grads[0].defined()) return res;
        const auto saved = ctx->get_saved_variables();
        const at::Tensor x = plain(saved[0]), g = plain(grads[0]), &Wqkvb = saved[1], &Wo = saved[2], &qkvb = saved[3],
                         &q = saved[4], &k = saved[5], &beta = saved[6], &buf = saved[7], &out = saved[8];
        const int64_t B = q.size(0), H = q.size(1), T = q.size(2), D = q.size(3), rows = T * B, d = Wqkvb.size(1),
                      width = Wqkvb.size(0);
        LaunchGuard guard(x);
        // create_graph: the projections' products from PyTorch's operators (the delta rule's own gradients, as from
        // fast_weight_delta, carry no graph)
        const bool graph = at::GradMode::is_enabled();
        if (ctx->needs_input_grad(2))
            res[2] = graph ? at::matmul(grads[0].reshape({rows, d}).t(),
                                        DeltaReadOutFn::apply(saved[0], Wqkvb, qkvb, q, k, beta, buf, out, ctx->saved_data["scale"].toDouble())
                                            .reshape({rows, H * D}))
                           : weight_grad(g, out, rows, d, H * D, nullptr);
        const at::Tensor go = matmul(FWP_MM_NN, g, Wo, rows, H * D, d, {T, B, H, D});
        const at::Tensor gp = projection_grad(go, qkvb, q, k, beta, buf, ctx->saved_data["scale"].toDouble());
        if (ctx->needs_input_grad(1))
            res[1] = graph ? at::matmul(gp.reshape({rows, width}).t(), saved[0].reshape({rows, d}))
                           : weight_grad(gp, x, rows, width, d, nullptr);
        if (ctx->needs_input_grad(0) && graph) {
            res[0] = at::matmul(gp, Wqkvb);
            if (ctx->saved_data["residual"].toBool()) res[0] = res[0] + grads[0];
        } else if (ctx->needs_input_grad(0)) {
            fwp_mm_epilogue e{};
            e.residual = ctx->saved_data["residual"].toBool() ? ptr(g) : nullptr;
            res[0] = matmul(FWP_MM_NN, gp, Wqkvb, rows, d, width, saved[0].sizes(), e);
        }
        return res;
    }
};

// ------------------------------------------------------------------ LayerNorm over the last axis

struct LayerNormFn : torch::autograd::Function<LayerNormFn> {
    static at::Tensor forward(AutogradContext *ctx, const at::Tensor &x_in, const at::Tensor &gamma, const at::Tensor &beta, double eps) {
        require_device(x_in);
        same_device(x_in, {gamma, beta});
        require(gamma.dim() == 1 && beta.sizes() == gamma.sizes() && x_in.numel() > 0 && ends_in(x_in, gamma.size(0)),
                "rows, weight and bias do not fit one another");
        const at::Tensor x = plain(x_in), g = plain(gamma), b = plain(beta);
        const int64_t cols = gamma.numel(), rows = x.numel() / cols;
        LaunchGuard guard(x);
        at::Tensor y = at::empty(x.sizes(), x.options()), stats;
        if (ctx) stats = at::empty({rows, 2}, x.options());
        check(fwp_layer_norm_fwd(ptr(x), ptr(g), ptr(b), ptr(y), ptr(stats), (int)rows, (int)cols, (float)eps, stream_of(x)),
              "fwp_layer_norm_fwd");
        if (ctx) {
            ctx->save_for_backward({x_in, gamma, beta, stats});
            ctx->saved_data["eps"] = eps;
            ctx->set_materialize_grads(false);
        }
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list res(4);
        if (!grads[0].defined()) return res;
        const auto saved = ctx->get_saved_variables();
        const at::Tensor &gamma = saved[1], &stats = saved[3];
        if (at::GradMode::is_enabled()) {
            res = differentiate(at::layer_norm(saved[0], gamma.sizes(), gamma, saved[2], ctx->saved_data["eps"].toDouble()),
                                {saved[0], gamma, saved[2]}, grads[0]);
            res.resize(4);
            return res;
        }
        const at::Tensor x = plain(saved[0]), g = plain(gamma), gy = plain(grads[0]);
        const int64_t cols = gamma.numel(), rows = x.numel() / cols;
        LaunchGuard guard(x);
        res[0] = at::empty(x.sizes(), x.options());
        res[1] = at::empty({cols}, x.options());
        res[2] = at::empty({cols}, x.options());
        const at::Tensor work = at::empty({fwp_layer_norm_workspace((int)rows, (int)cols)}, x.options());
        check(fwp_layer_norm_bwd(ptr(gy), ptr(x), ptr(stats), ptr(g), ptr(res[0]), ptr(res[1]), ptr(res[2]), ptr(work), (int)rows,
                                 (int)cols, stream_of(x)),
              "fwp_layer_norm_bwd");
        return res;
    }
};

// ------------------------------------------------------------------ negative log-likelihood under softmax(x W^T + bias)

struct NllFn : torch::autograd::Function<NllFn> {
    // x [rows, dim], target [rows] int64
    static at::Tensor forward(AutogradContext *ctx, const at::Tensor &x_in, const at::Tensor &W, const at::Tensor &bias,
                              const at::Tensor &target_in) {
        require_device(x_in);
        same_device(x_in, {W, bias, target_in});
        require(x_in.dim() == 2 && target_in.dim() == 1 && target_in.size(0) == x_in.size(0) && target_in.scalar_type() == at::kLong,
                "hidden [rows, d_model] and int64 targets [rows]");
        require(x_in.numel() > 0 && W.dim() == 2 && W.numel() > 0 && W.size(1) == x_in.size(1) && same_shape(bias, {W.size(0)}),
                "hidden, weight and bias do not fit one another");
        const at::Tensor x = plain(x_in), target = target_in.contiguous();
        const int64_t rows = x.size(0), dim = x.size(1), vocab = W.size(0);
        LaunchGuard guard(x);
        const at::Tensor loss = at::empty({rows}, x.options()),
                         work = at::empty({fwp_nll_workspace((int)rows, (int)vocab)}, x.options());
        at::Tensor logits, stats;
        if (ctx) {
            logits = at::empty({rows, vocab}, x.options());
            stats = at::empty({rows, 2}, x.options());
            check(fwp_nll_stats_fwd(ptr(x), ptr(W), ptr(bias), target.data_ptr<int64_t>(), ptr(logits), ptr(loss), ptr(stats),
                                    ptr(work), (int)rows, (int)vocab, (int)dim, stream_of(x)),
                  "fwp_nll_stats_fwd");
            ctx->save_for_backward({x_in, W, bias, target, logits, stats});
            ctx->set_materialize_grads(false);
        } else {
            check(fwp_nll_fwd(ptr(x), ptr(W), ptr(bias), target.data_ptr<int64_t>(), nullptr, ptr(loss), nullptr, ptr(work), (int)rows,
                              (int)vocab, (int)dim, stream_of(x)),
                  "fwp_nll_fwd");
        }
        return loss;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list res(4);
        if (!grads[0].defined()) return res;
        const auto saved = ctx->get_saved_variables();
        const at::Tensor &W = saved[1], &bias = saved[2], &target = saved[3], &logits = saved[4], &stats = saved[5];
        if (at::GradMode::is_enabled()) {
            res = differentiate(at::cross_entropy_loss(at::linear(saved[0], W, bias), target, {}, at::Reduction::None),
                                {saved[0], W, bias}, grads[0]);
            res.resize(4);
            return res;
        }
        const at::Tensor x = plain(saved[0]), g = plain(grads[0]);
        const int64_t rows = x.size(0), dim = x.size(1), vocab = W.size(0);
        LaunchGuard guard(x);
        if (ctx->needs_input_grad(0)) res[0] = at::empty({rows, dim}, x.options());
        if (ctx->needs_input_grad(1) || ctx->needs_input_grad(2)) {
            res[1] = at::empty({vocab, dim}, x.options());
            res[2] = at::empty({vocab}, x.options());
        }
        at::Tensor work;
        const int64_t n = std::max(fwp_matmul_workspace((int)rows, (int)dim, (int)vocab),
                                   fwp_matmul_workspace((int)vocab, (int)dim, (int)rows));
        if (n > 0) work = at::empty({n}, x.options());
        check(fwp_nll_stats_bwd(ptr(x), ptr(W), ptr(logits), ptr(stats), target.data_ptr<int64_t>(), ptr(g), ptr(res[0]), ptr(res[1]),
                                ptr(res[2]), ptr(work), (int)rows, (int)vocab, (int)dim, stream_of(x)),
              "fwp_nll_stats_bwd");
        return res;
    }
};

// ------------------------------------------------------------------ decoding

// A layer's parameters: qkvb_net.weight, o_net.weight, dec_attn.layer_norm weight and bias, CoreNet.0 weight and
// bias, CoreNet.3 weight and bias, pos_ff.layer_norm weight and bias.
constexpr size_t kPerLayer = 10;

// One token per sequence through the layers: x [1,B,d], states [B,H,D,D] per layer (empty: zeros) ->
// (hidden [1,B,d], the states after the token), or nothing for parameters that fwp_rows_matmul does not take (the layers
// one by one do).  Nothing is recorded.
std::optional<std::tuple<at::Tensor, std::vector<at::Tensor>>> decode_layers(const at::Tensor &x_in, const std::vector<at::Tensor> &params,
                                                              const std::vector<at::Tensor> &states, int64_t H, int64_t D,
                                                              double eps, bool pre_norm, double scale) {
    at::AutoDispatchBelowADInplaceOrView below;
    require_device(x_in);
    const size_t layers = params.size() / kPerLayer;
    require(params.size() == layers * kPerLayer && (states.empty() || states.size() == layers) && x_in.dim() == 3 && x_in.size(0) == 1,
            "one token per sequence, ten parameters and one state per layer");
    const at::Tensor x = plain(x_in);
    const int64_t B = x.size(1), d = x.size(2), width = H * (3 * D + 1);
    const auto opts = x.options();
    LaunchGuard guard(x);
    void *const s = stream_of(x);
    int64_t inner_most = 0;
    for (size_t l = 0; l < layers; l++) {
        const at::Tensor *p = &params[kPerLayer * l];
        const int64_t inner = p[4].dim() == 2 ? p[4].size(0) : 0;
        bool ok = inner > 0 && inner % 64 == 0 && same_shape(p[0], {width, d}) && same_shape(p[1], {d, H * D}) && same_shape(p[4], {inner, d}) &&
                  same_shape(p[5], {inner}) && same_shape(p[6], {d, inner});
        for (size_t i : {2, 3, 7, 8, 9}) ok = ok && same_shape(p[i], {d});
        for (size_t i = 0; i < kPerLayer; i++) {
            ok = ok && p[i].device() == x.device() && p[i].scalar_type() == at::kFloat && p[i].is_contiguous() &&
                 reinterpret_cast<uintptr_t>(p[i].data_ptr()) % 16 == 0;
        }
        if (!ok) return std::nullopt;
        inner_most = std::max(inner_most, inner);
    }
    // one buffer for everything in between; the states, which the caller keeps or drops one by one, on their own
    const int64_t rows_d = (B * d + 3) & ~int64_t(3);
    const at::Tensor work = at::empty({B * width + 4 + B * H * D + 4 * rows_d + B * inner_most}, opts);
    float *const a = ptr(work), *const b = a + rows_d, *const y = b + rows_d, *const h2 = y + rows_d, *const out = h2 + rows_d,
                *const hid = out + B * H * D, *const qkvb = hid + B * inner_most;
    const at::Tensor result = at::empty({1, B, d}, opts);
    std::vector<at::Tensor> after(layers);
    const float *const none = nullptr;
    const auto product = [&](const float *in, const at::Tensor *g, const at::Tensor *be, float *norm, const at::Tensor &W,
                             const at::Tensor *bias, const float *residual, int relu, float *to) {
        check(fwp_rows_matmul(in, g ? ptr(*g) : none, be ? ptr(*be) : none, (float)eps, norm, ptr(W), bias ? ptr(*bias) : none, residual,
                              relu, to, (int)B, (int)W.size(0), (int)W.size(1), s),
              "fwp_rows_matmul");
    };
    const float *in = ptr(x);       // the layer's input, before the last layer's LayerNorm (post-norm)
    for (size_t l = 0; l < layers; l++) {
        const at::Tensor *p = &params[kPerLayer * l], *before = pre_norm ? p + 2 : l ? p - 2 : nullptr;
        at::Tensor from;
        if (!states.empty()) {
            from = plain(states[l]);
            same_device(x, {from});
            require(same_shape(from, {B, H, D, D}), "a state does not fit [bsz, n_head, d_head, d_head]");
        }
        after[l] = at::empty({B, H, D, D}, opts);
        // post-norm: LN of the previous layer's sum on the way in, that is also the residual; pre-norm: this layer's
        product(in, before, before ? before + 1 : nullptr, before ? y : nullptr, p[0], nullptr, none, 0, qkvb);
        check(fwp_deltanet_step(qkvb, ptr(from), ptr(after[l]), out, (int)B, (int)H, (int)D,
                                (float)scale, s),
              "fwp_deltanet_step");
        product(out, nullptr, nullptr, nullptr, p[1], nullptr, before ? y : in, 0, a);
        // feed-forward: post-norm adds the normalised rows back, pre-norm the rows themselves
        const at::Tensor *norm = pre_norm ? p + 8 : p + 2;
        product(a, norm, norm + 1, pre_norm ? nullptr : h2, p[4], &p[5], none, 1, hid);
        float *const to = pre_norm && l + 1 == layers ? ptr(result) : b;
        product(hid, nullptr, nullptr, nullptr, p[6], &p[7], pre_norm ? a : h2, 0, to);
        in = to;
    }
    if (!pre_norm) {
        const at::Tensor *p = &params[kPerLayer * (layers - 1)];
        check(fwp_layer_norm_fwd(in, ptr(p[8]), ptr(p[9]), ptr(result), nullptr, (int)B, (int)d, (float)eps, s), "fwp_layer_norm_fwd");
    }
    return std::make_tuple(result, std::move(after));
}

// word embedding times scale plus the positions' sinusoids, for ids [T,B]; nothing is recorded
at::Tensor embed(const at::Tensor &table, const at::Tensor &ids, const at::Tensor &inv_freq, double scale, double clamp) {
    at::AutoDispatchBelowADInplaceOrView below;
    require_device(table);
    same_device(table, {ids, inv_freq});
    require(table.dim() == 2 && ids.dim() == 2, "a table [n_token, d_model] and ids [len, bsz]");
    const int64_t T = ids.size(0), B = ids.size(1), d = table.size(1);
    require(ids.scalar_type() == at::kLong && inv_freq.numel() * 2 == d, "int64 ids [len, bsz] and d_model/2 frequencies");
    const at::Tensor t = plain(table), i = ids.contiguous(), f = plain(inv_freq), out = at::empty({T, B, d}, t.options());
    LaunchGuard guard(t);
    check(fwp_embed(ptr(t), i.data_ptr<int64_t>(), ptr(f), ptr(out), (int)T, (int)B, (int)d, t.size(0), (float)scale, (float)clamp,
                    stream_of(t)),
          "fwp_embed");
    return out;
}

bool records(std::initializer_list<const at::Tensor *> ts) {
    if (!at::GradMode::is_enabled()) return false;
    for (const at::Tensor *t : ts)
        if (t->defined() && t->requires_grad()) return true;
    return false;
}

at::Tensor linear(const at::Tensor &x, const at::Tensor &W, const std::optional<at::Tensor> &bias_, bool relu) {
    const at::Tensor bias = given(bias_);
    if (records({&x, &W, &bias})) return LinearFn::apply(x, W, bias_, relu);
    at::AutoDispatchBelowADInplaceOrView below;
    return LinearFn::forward(nullptr, x, W, bias_, relu);
}

at::Tensor feed_forward(const at::Tensor &x, const at::Tensor &W1, const at::Tensor &b1, const at::Tensor &W2, const at::Tensor &b2,
                        const std::optional<at::Tensor> &residual_) {
    const at::Tensor residual = given(residual_);
    const bool same = residual.defined() && residual.is_same(x);
    if (records({&x, &W1, &b1, &W2, &b2, &residual}))
        return FeedForwardFn::apply(x, W1, b1, W2, b2, same ? std::nullopt : residual_, same);
    at::AutoDispatchBelowADInplaceOrView below;
    return FeedForwardFn::forward(nullptr, x, W1, b1, W2, b2, residual_, same);
}

at::Tensor delta_block(const at::Tensor &x, const at::Tensor &Wqkvb, const at::Tensor &Wo, const at::Tensor &state, int64_t n_head,
                       int64_t d_head, double scale, bool residual, bool fresh) {
    if (records({&x, &Wqkvb, &Wo})) return DeltaBlockFn::apply(x, Wqkvb, Wo, state, n_head, d_head, scale, residual, fresh);
    at::AutoDispatchBelowADInplaceOrView below;
    return DeltaBlockFn::forward(nullptr, x, Wqkvb, Wo, state, n_head, d_head, scale, residual, fresh);
}

at::Tensor layer_norm(const at::Tensor &x, const at::Tensor &gamma, const at::Tensor &beta, double eps) {
    if (records({&x, &gamma, &beta})) return LayerNormFn::apply(x, gamma, beta, eps);
    at::AutoDispatchBelowADInplaceOrView below;
    return LayerNormFn::forward(nullptr, x, gamma, beta, eps);
}

at::Tensor nll(const at::Tensor &x, const at::Tensor &W, const at::Tensor &bias, const at::Tensor &target) {
    if (records({&x, &W, &bias})) return NllFn::apply(x, W, bias, target);
    at::AutoDispatchBelowADInplaceOrView below;
    return NllFn::forward(nullptr, x, W, bias, target);
}

// ------------------------------------------------------------------ does a block apply?

// One call per block instead of a dozen attributes looked up from Python, which costs as much as a small layer's kernels.
// The two Python types, held for good from bind_blocks on.
PyObject *g_tensor_type, *g_parameter_type;

// An ordinary tensor or parameter (no subclass, no tracer's stand-in), or nothing
const at::Tensor *ordinary(py::handle h) {
    const PyObject *const type = reinterpret_cast<PyObject *>(Py_TYPE(h.ptr()));
    return type == g_tensor_type || type == g_parameter_type ? &THPVariable_Unpack(h.ptr()) : nullptr;
}

bool on_gpu(const at::Tensor &t) {
#ifdef FWP_HOST_STUB
    return true;
#else
    return t.is_cuda();
#endif
}

// fp32 on the GPU, with something in it
const at::Tensor *fp32(py::handle h) {
    const at::Tensor *const t = ordinary(h);
    return t && t->scalar_type() == at::kFloat && t->numel() > 0 && on_gpu(*t) ? t : nullptr;
}

// The kernels' offsets reach rows of 2^21 floats, their launches 2^24 rows.
const at::Tensor *input(py::handle h) {
    const at::Tensor *const t = fp32(h);
    return t && t->dim() > 0 && t->numel() / t->size(-1) <= (int64_t(1) << 24) ? t : nullptr;
}
const at::Tensor *parameter(py::handle h) {
    const at::Tensor *const t = fp32(h);
    if (!t || !t->is_contiguous()) return nullptr;
    for (const int64_t n : t->sizes())
        if (n > (int64_t(1) << 21)) return nullptr;
    return t;
}

bool takes_all(py::handle x_, const py::list &params) {
    if (!input(x_)) return false;
    for (py::handle p : params)
        if (!parameter(p)) return false;
    return true;
}

bool takes_linear(py::handle x_, py::handle W_, py::handle b_) {
    const at::Tensor *const x = input(x_), *const W = parameter(W_), *const b = parameter(b_);
    return x && W && b && W->dim() == 2 && x->size(-1) == W->size(1) && same_shape(*b, {W->size(0)});
}

bool takes_feed_forward(py::handle x_, py::handle W1_, py::handle b1_, py::handle W2_, py::handle b2_) {
    const at::Tensor *const x = input(x_), *const W1 = parameter(W1_), *const b1 = parameter(b1_), *const W2 = parameter(W2_),
                     *const b2 = parameter(b2_);
    if (!(x && W1 && b1 && W2 && b2)) return false;
    const int64_t d = x->size(-1), inner = b1->numel();
    return same_shape(*W1, {inner, d}) && same_shape(*b1, {inner}) && same_shape(*W2, {d, inner}) && same_shape(*b2, {d});
}

bool takes_layer_norm(py::handle x_, py::handle g_, py::handle b_, int64_t d) {
    const at::Tensor *const x = input(x_), *const g = parameter(g_), *const b = parameter(b_);
    return x && g && b && d % 4 == 0 && d <= 1024 && x->size(-1) == d && same_shape(*g, {d}) && same_shape(*b, {d});
}

bool takes_delta_block(py::handle x_, py::handle Wqkvb_, py::handle Wo_, int64_t H, int64_t D) {
    const at::Tensor *const x = input(x_), *const Wqkvb = parameter(Wqkvb_), *const Wo = parameter(Wo_);
    return x && Wqkvb && Wo && (D == 16 || D == 32 || D == 64) && same_shape(*Wqkvb, {H * (3 * D + 1), x->size(-1)}) &&
           same_shape(*Wo, {x->size(-1), H * D});
}

bool takes_nll(py::handle x_, py::handle W_, py::handle b_, py::handle target_) {
    const at::Tensor *const x = input(x_), *const W = parameter(W_), *const b = parameter(b_), *const target = ordinary(target_);
    return x && W && b && target && x->dim() == 2 && W->dim() == 2 && x->size(1) == W->size(1) && same_shape(*b, {W->size(0)}) &&
           target->scalar_type() == at::kLong && target->device() == x->device() && same_shape(*target, {x->size(0)});
}

}  // namespace

void bind_blocks(py::module_ &m) {
    g_tensor_type = py::object(py::module_::import("torch").attr("Tensor")).release().ptr();
    g_parameter_type = py::object(py::module_::import("torch.nn").attr("Parameter")).release().ptr();
    m.def("takes_all", &takes_all, "may an input and parameters of any sizes go to the kernels?");
    m.def("takes_linear", &takes_linear, "does linear apply?");
    m.def("takes_feed_forward", &takes_feed_forward, "does feed_forward apply?");
    m.def("takes_layer_norm", &takes_layer_norm, "does layer_norm apply?");
    m.def("takes_delta_block", &takes_delta_block, "does delta_block apply?");
    m.def("takes_nll", &takes_nll, "does nll apply?");
    m.def("linear", &linear, py::arg("x"), py::arg("W"), py::arg("bias") = py::none(), py::arg("relu") = false,
          "x W^T (+ bias) (relu)");
    m.def("feed_forward", &feed_forward, py::arg("x"), py::arg("W1"), py::arg("b1"), py::arg("W2"), py::arg("b2"),
          py::arg("residual") = py::none(), "relu(x W1^T + b1) W2^T + b2 (+ residual)");
    m.def("decode_layers", &decode_layers, "one token per sequence through the layers -> (hidden, states); records nothing");
    m.def("embed", &embed, "the model's input from token ids; records nothing");
    m.def("layer_norm", &layer_norm, "LayerNorm over the last axis (a multiple of 4 up to 1024)");
    m.def("nll", &nll, "per-row negative log-likelihood of the targets under softmax(x W^T + bias); a target of -100 counts 0");
    m.def("delta_block", &delta_block, py::arg("x"), py::arg("Wqkvb"), py::arg("Wo"), py::arg("state"), py::arg("n_head"), py::arg("d_head"),
          py::arg("scale"), py::arg("residual"), py::arg("fresh") = false,
          "the Delta-Net layer between its input and its LayerNorm; the state is updated in place, from zeros whatever it holds if it is fresh");
}
