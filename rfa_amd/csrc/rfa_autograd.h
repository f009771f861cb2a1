// The package's autograd functions as C++ nodes, and the chains of them that one call of a module is.
//
// The Python autograd functions (rfa_amd/rfa.py, utils.py, projection.py, causal_attention.py,
// cross_attention.py) are the general form: any dtype, either binding, tracing, dispatch modes,
// functorch's errors.  What a training or serving step does -- plain fp16 tensors on one HIP
// device -- comes here instead: the same launches in the same order, without an interpreter between
// them.  Each entry point returns nothing when a tensor or the mode is not plain (see plain()), and
// the caller then goes its general way; errors in shapes are raised by the same checks as there.
//
// What bounds a layer without this is the host.  The Python functions over the same kernels (input gradients by the
// library there) / these nodes, us: a layer of 8 heads of 64, 8192 tokens, forward + backward, 212 of kernels, 487 / 237;
// 128 tokens of 4 heads, the scan alone, 125 / 75; an encoder-decoder layer, 16384 + 8192 rows, 611 / 324; a decoding step of
// 64 sequences 71 / 23.
#pragma once
#include <ATen/autocast_mode.h>
#include <ATen/hip/HIPContextLight.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPException.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <algorithm>

namespace {

using OptTensor = c10::optional<Tensor>;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// ---- which calls are plain ------------------------------------------------------------
// Tracing must record the Python functions, dispatch modes and tensor subclasses must see them, and
// functorch's wrappers and forward-mode tangents must meet the errors that those raise.
bool plain_mode() {
    return !torch::jit::tracer::isTracing() && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

bool plain(const Tensor& t, torch::ScalarType type, int64_t dim) {
    static const c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                          c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched,
                                          c10::DispatchKey::Functionalize, c10::DispatchKey::Negative,
                                          c10::DispatchKey::Conjugate});
    return t.defined() && t.is_cuda() && t.scalar_type() == type && t.dim() == dim && t.layout() == c10::kStrided &&
           !t.key_set().has_any(odd) && !t._fw_grad(0).defined();
}

bool node_plain(const Tensor& t) { return plain_mode() && plain(t, t.scalar_type(), t.dim()); }

bool plain_half(const Tensor& t, int64_t dim) { return plain(t, torch::kFloat16, dim); }
bool plain_half(const OptTensor& t, int64_t dim) { return !t.has_value() || plain(*t, torch::kFloat16, dim); }

template <typename... T>
bool wants_grad(const T&... t) {
    return at::GradMode::is_enabled() && (... || (t.defined() && t.requires_grad()));
}
bool wants_grad_opt(const OptTensor& t) { return t.has_value() && t->requires_grad(); }

bool aligned16(const Tensor& t) { return reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0; }
// A saved tensor comes back through the hooks that the program may have set.  Other strides are theirs to choose, and
// a hook may get type or device wrong: all three are looked at again before a pointer is used.
void check_saved(const char* name, const Tensor& t, const Tensor& like) {
    TORCH_CHECK(t.is_cuda() && t.device() == like.device(), name, " must be on ", like.device(), " (got ", t.device(), ")");
    TORCH_CHECK_TYPE(t.scalar_type() == torch::kFloat16, name, " must be float16 (got ", t.scalar_type(), ")");
}

// and the shapes, where launches take them together: layers w [e_out, E] over x [.., E] whose outputs have `rows` rows
void check_saved_layers(const Tensor& x, const Tensor* w, int64_t n, int64_t rows, int64_t e_out) {
    const int64_t e_in = x.dim() > 0 ? x.size(-1) : 0;
    bool ok = x.dim() > 0 && x.numel() == rows * e_in;
    for (int64_t p = 0; p < n; ++p) ok = ok && w[p].dim() == 2 && w[p].size(0) == e_out && w[p].size(1) == e_in;
    TORCH_CHECK_VALUE(ok, "saved x ", x.sizes(), " and weight ", w[0].sizes(), " do not fit the gradient of ", rows, " rows of ", e_out);
}

Tensor opt(const OptTensor& t) { return t.has_value() ? *t : Tensor(); }
OptTensor opt(const Tensor& t) { return t.defined() ? OptTensor(t) : c10::nullopt; }

// ---- random matrices --------------------------------------------------------------------
struct BuildNode : public torch::autograd::Function<BuildNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& w, const OptTensor& sigma, double tau) {
        const Tensor wc = w.contiguous();
        const OptTensor sg = sigma.has_value() ? OptTensor(sigma->contiguous()) : c10::nullopt;
        ctx->saved_data["tau"] = tau;
        ctx->saved_data["need_w"] = w.requires_grad();
        ctx->saved_data["need_sigma"] = wants_grad_opt(sigma);
        ctx->save_for_backward({wc, opt(sg)});
        return build_random_matrices(wc, sg, tau);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto saved = ctx->get_saved_variables();
        auto [dsigma, dw] = build_random_matrices_backward(saved[0], opt(saved[1]), g[0].contiguous(),
                                                           ctx->saved_data["tau"].toDouble(),
                                                           ctx->saved_data["need_sigma"].toBool(),
                                                           ctx->saved_data["need_w"].toBool());
        return {opt(dw), opt(dsigma), Tensor()};
    }
};

Tensor build_matrices(const Tensor& w, const OptTensor& sigma, double tau) {
    if (at::GradMode::is_enabled() && (w.requires_grad() || wants_grad_opt(sigma))) return BuildNode::apply(w, sigma, tau);
    return build_random_matrices(w.contiguous(), sigma.has_value() ? OptTensor(sigma->contiguous()) : c10::nullopt, tau);
}

// tau = 0 or matrices that are not fp16 [H, D, d] with sigma [H, 1, d] take the ATen chain
bool plain_matrices(const Tensor& w, const OptTensor& sigma, double tau) {
    return plain_half(w, 3) && tau != 0 &&
           (!sigma.has_value() || (plain_half(*sigma, 3) && sigma->size(0) == w.size(0) && sigma->size(1) == 1 &&
                                   sigma->size(2) == w.size(2)));
}

// ---- feature map ------------------------------------------------------------------------
void check_feature_grad(const Tensor& x, const Tensor& x0, const Tensor& w, const Tensor& g) {
    check_feature_args(x, w);
    check_half("grad_phi", g, 4);
    TORCH_CHECK_VALUE(x.sizes() == x0.sizes() && g.size(0) == x0.size(0) && g.size(1) == x0.size(1) && g.size(2) == x0.size(2) &&
                          g.size(3) == 2 * w.size(1), "grad_phi ", g.sizes(), " does not fit x ", x0.sizes(), " and ", w.size(1),
                      " features");
}

// dx of one or two tensors through the same w, or the packed gradient [dx0 | dx1 | third] in `packed`; returns dW'
// in fp16, undefined where w takes no gradient
Tensor feature_grads(const Tensor& x0, const Tensor* x1, const Tensor& w, const Tensor& g0, const Tensor* g1,
                     const Tensor* third, Tensor& dx0, Tensor* dx1, bool packed, double scale, bool need_dw) {
    if (!need_dw) {
        if (packed) dx0 = std::get<0>(feature_map_backward_pair_packed(x0, *x1, w, g0, *g1, opt(*third), scale, false));
        else if (x1) std::tie(dx0, *dx1, std::ignore) = feature_map_backward_pair(x0, *x1, w, g0, *g1, scale, false);
        else dx0 = std::get<0>(feature_map_backward(x0, w, g0, scale, false));
        return Tensor();
    }
    const int64_t R = x0.size(0) * x0.size(1);
    const int H = (int)x0.size(2), d = (int)x0.size(3), D = (int)w.size(1);
    check_feature_grad(x0, x0, w, g0);
    if (x1) check_feature_grad(*x1, x0, w, *g1);
    if (third) TORCH_CHECK_VALUE(third->numel() == x0.numel() && third->is_contiguous(), "third must hold the rows of x");
    dx0 = packed ? torch::empty({R, 3 * (int64_t)H * d}, x0.options()) : torch::empty_like(x0);
    if (x1 && !packed) *dx1 = torch::empty_like(*x1);
    Tensor dw = torch::empty({H, D, d}, x0.options());
    Launch l(x0);
    const size_t nbytes = x1 ? rfa_feature_map_backward_pair_workspace_bytes(R, H, D, d)
                             : rfa_feature_map_backward_workspace_bytes(R, H, D, d);
    Tensor ws = workspace(nbytes, x0);
    check_rc(rfa_feature_map_backward_half(ptr(x0), x1 ? ptr(*x1) : nullptr, ptr(w), ptr(g0), g1 ? ptr(*g1) : nullptr,
                                           third ? ptr(*third) : nullptr, packed ? nullptr : ptr(dx0),
                                           x1 && !packed ? ptr(*dx1) : nullptr, packed ? ptr(dx0) : nullptr, ptr(dw), R, H, D,
                                           d, (float)scale, ptr(ws), nbytes, l.stream));
    return dw;
}

struct FeatureNode : public torch::autograd::Function<FeatureNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, double scale) {
        const Tensor xc = x.contiguous(), wc = w.contiguous();
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["need_w"] = w.requires_grad();
        ctx->save_for_backward({xc, wc});
        return feature_map_forward(xc, wc, scale);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto saved = ctx->get_saved_variables();
        Tensor dx;
        const Tensor dw = feature_grads(saved[0], nullptr, saved[1], g[0].contiguous(), nullptr, nullptr, dx, nullptr, false,
                                        ctx->saved_data["scale"].toDouble(), ctx->saved_data["need_w"].toBool());
        return {dx, dw, Tensor()};
    }
};

OptTensor node_random_project(const Tensor& x, const Tensor& w, double scale) {
    if (!plain_mode() || !plain_half(x, 4) || !plain_half(w, 3)) return c10::nullopt;
    if (wants_grad(x, w)) return FeatureNode::apply(x, w, scale);
    return feature_map_forward(x.contiguous(), w.contiguous(), scale);
}

// ---- projections to heads, with the feature map where a bit of `phi` is set ----------------------
// The weights and biases of up to three Linear layers over one input; the first, or the first two, through the
// feature map.
struct Layers {
    std::vector<Tensor> w;
    std::vector<OptTensor> b;
    bool phi[3] = {false, false, false};
};

std::vector<bool> phi_flags(const Layers& l) { return std::vector<bool>(l.phi, l.phi + l.w.size()); }

// (dW, db) of Linear layers that share the input x2: one row-split launch where the widths allow it
std::pair<std::vector<Tensor>, std::vector<OptTensor>> param_grads(const Tensor& x2, const std::vector<Tensor>& dys,
                                                                   const std::vector<bool>& bias) {
    if (dys[0].size(1) % 128 == 0 && x2.size(1) % 128 == 0) {
        std::vector<Tensor> c;
        for (const Tensor& dy : dys) c.push_back(dy.contiguous());
        auto [dws, dbs] = linear_weight_grad(x2.contiguous(), c, bias);
        return {dws, dbs};
    }
    std::vector<Tensor> dws;
    std::vector<OptTensor> dbs;
    for (size_t p = 0; p < dys.size(); ++p) {
        dws.push_back(at::mm(dys[p].t(), x2));
        dbs.push_back(bias[p] ? OptTensor(dys[p].sum(0)) : c10::nullopt);
    }
    return {dws, dbs};
}

// Products through the framework's own kernels: a library product costs 19 us of host time, these 4 to 5, and
// two of them in a backward need a second pass over dx, three a stack of the weights.  Up to 7 * 2^30
// multiply-adds they are level on the device where there are rows enough, us own / library: 8192 rows of 512 -> 512
// 11.6 / 12.3 (dx), 10.3 / 11.3 (y); three of them 25 / 21.5 + 3.0 for the stack.  Past that the library's larger tiles
// win (8192 rows of 1024 -> 1024 28.5 / 23.4, 26.7 / 22.6; three 69 / 57 + 7.8), for two layers without a packed
// gradient, where it takes two products, later (16384 rows of 512 28.4 / 35.6; of 1024 82.5 / 75).  Few rows of a
// wide layer lose device time to it (the contraction is walked by one workgroup per tile: 512 rows of 1024 -> 1024
// 12.6 / 8.0 dx, 10.8 / 8.6 y; three 32 / 16.5 + 4.5), which is given for the host time: a step of that size waits
// for the host by far.
bool own_product(int64_t rows, int64_t e_out, int64_t e_in, int64_t n) {
    return rows > 0 && rows * e_out * e_in * n <= (n == 2 ? (int64_t)1 << 34 : (int64_t)7 << 30);
}

// dx = sum_p dy_p W_p for dy_p [rows, E_out] that lie ld halves a row from dys[p] on.  Not where the backward pass
// itself is recorded (create_graph): the library's products are differentiable, a launch is not.
bool own_input_grad(int64_t rows, const Tensor* w, int64_t n) {
    const int64_t widest = (int64_t)1 << 22;      // what the launch addresses
    bool ok = !at::GradMode::is_enabled() && own_product(rows, w[0].size(0), w[0].size(1), n) && w[0].size(0) % 32 == 0 &&
              w[0].size(1) % 128 == 0 && w[0].size(1) <= widest && n * w[0].size(0) <= widest;
    for (int64_t p = 0; p < n; ++p) ok = ok && w[p].is_contiguous() && aligned16(w[p]);
    return ok;
}

Tensor input_grad(const std::vector<const void*>& dys, int64_t ld, const Tensor* w, const Tensor& x) {
    const int64_t n = (int64_t)dys.size(), e_out = w[0].size(0), e_in = w[0].size(1), rows = x.numel() / e_in;
    std::array<const void*, 3> wp{};
    for (int64_t p = 0; p < n; ++p) wp[p] = ptr(w[p]);
    Tensor dx = torch::empty(x.sizes(), x.options());
    Launch l(x);
    check_rc(rfa_linear_input_grad(dys.data(), ld, wp.data(), (int)n, ptr(dx), rows, (int)e_out, (int)e_in, l.stream));
    return dx;
}

// dx (of x's shape), dW and db of layers over one input in one launch where the library takes them so.  dys as for
// input_grad; `dw` and `db` [n] get the gradients, db those whose flag is set.
bool linear_grads(const std::vector<const void*>& dys, int64_t ld, const Tensor* w, const Tensor& x, const Tensor& x2,
                  const std::vector<bool>& bias, Tensor& dx, std::vector<Tensor>& dw, std::vector<OptTensor>& db) {
    const int64_t n = (int64_t)dys.size(), e_out = w[0].size(0), e_in = w[0].size(1), rows = x2.size(0);
    const size_t nbytes = rfa_linear_grads_workspace_bytes(rows, (int)e_out, (int)e_in, (int)n);
    if (nbytes == 0) return false;
    const Tensor xc = x2.contiguous();
    if (!aligned16(xc)) return false;
    std::array<const void*, 3> wp{};
    std::array<void*, 3> dwp{}, dbp{};
    for (int64_t p = 0; p < n; ++p) {
        wp[p] = ptr(w[p]);
        dw.push_back(torch::empty({e_out, e_in}, x.options()));
        db.push_back(bias[p] ? OptTensor(torch::empty({e_out}, x.options())) : c10::nullopt);
        dwp[p] = ptr(dw[p]);
        dbp[p] = ptr(db[p]);
    }
    dx = torch::empty(x.sizes(), x.options());
    Launch l(x);
    Tensor ws = workspace(nbytes, x);
    check_rc(rfa_linear_grads(ptr(xc), dys.data(), ld, wp.data(), (int)n, ptr(dx), dwp.data(), dbp.data(), rows, (int)e_out,
                              (int)e_in, ptr(ws), nbytes, l.stream));
    return true;
}

// Those gradients and the feature map's where the library takes all of it: the first nphi layers went through the feature
// map (outputs y), g their gradients, else those of the layers' outputs.  dwf as feature_grads.
bool project_grads(const variable_list& g, const Tensor* y, int64_t nphi, const Tensor& wf, const Tensor* w, int64_t n, const Tensor& x,
                   const std::vector<bool>& bias, double scale, bool need_wf, Tensor& dx, std::vector<Tensor>& dw,
                   std::vector<OptTensor>& db, Tensor& dwf) {
    const int64_t e_out = w[0].size(0), e_in = w[0].size(1), rows = x.size(0) * x.size(1);
    const int H = (int)y[0].size(2), d = (int)y[0].size(3), D = (int)wf.size(1);
    const size_t nbytes = rfa_project_grads_workspace_bytes(rows, H, D, d, (int)e_in, (int)n, (int)nphi);
    if (nbytes == 0 || !aligned16(x) || !x.is_contiguous()) return false;
    std::array<Tensor, 3> gc;
    for (int64_t p = 0; p < n; ++p) {
        gc[p] = g[p].contiguous();
        if (!aligned16(gc[p])) return false;
    }
    for (int64_t p = 0; p < nphi; ++p) check_feature_grad(y[p], y[0], wf, gc[p]);
    std::array<const void*, 3> wp{}, gp{}, yp{};
    std::array<void*, 3> dwp{}, dbp{};
    for (int64_t p = 0; p < n; ++p) {
        wp[p] = ptr(w[p]);
        gp[p] = ptr(gc[p]);
        if (p < nphi) yp[p] = ptr(y[p]);
        dw.push_back(torch::empty({e_out, e_in}, x.options()));
        db.push_back(bias[p] ? OptTensor(torch::empty({e_out}, x.options())) : c10::nullopt);
        dwp[p] = ptr(dw[p]);
        dbp[p] = ptr(db[p]);
    }
    dx = torch::empty(x.sizes(), x.options());
    if (need_wf) dwf = torch::empty({H, D, d}, x.options());
    Launch l(x);
    Tensor ws = workspace(nbytes, x);
    check_rc(rfa_project_grads(ptr(x), yp.data(), ptr(wf), gp.data(), wp.data(), (int)n, (int)nphi, ptr(dx), dwp.data(), dbp.data(),
                               need_wf ? ptr(dwf) : nullptr, rows, H, D, d, (int)e_in, (float)scale, ptr(ws), nbytes, l.stream));
    return true;
}

struct ProjectNode : public torch::autograd::Function<ProjectNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& x, const OptTensor& wf, double scale, int64_t heads,
                                 int64_t phi, const OptTensor& w0, const OptTensor& b0, const OptTensor& w1,
                                 const OptTensor& b1, const OptTensor& w2, const OptTensor& b2) {
        Layers l;
        for (const auto& [w, b] : {std::pair(&w0, &b0), std::pair(&w1, &b1), std::pair(&w2, &b2)}) {
            if (!w->has_value()) break;
            l.phi[l.w.size()] = (phi >> l.w.size()) & 1;
            l.w.push_back((*w)->contiguous());
            l.b.push_back(*b);
        }
        const OptTensor wfc = wf.has_value() ? OptTensor(wf->contiguous()) : c10::nullopt;
        auto [ys, phis] = project_feature_map(x.contiguous(), l.w, l.b, phi_flags(l), wfc, heads, scale, true);
        int64_t bias = 0;
        variable_list keep{x, opt(wfc)}, out;
        for (const OptTensor& w : {w0, w1, w2})
            if (w.has_value()) keep.push_back(*w);
        for (size_t p = 0; p < l.w.size(); ++p) {
            bias |= (int64_t)l.b[p].has_value() << p;
            if (l.phi[p]) keep.push_back(*ys[p]);
            out.push_back(l.phi[p] ? *phis[p] : *ys[p]);
        }
        ctx->saved_data["scale"] = scale;
        ctx->saved_data["phi"] = phi;
        ctx->saved_data["bias"] = bias;
        ctx->saved_data["n"] = (int64_t)l.w.size();
        ctx->saved_data["need_x"] = x.requires_grad();
        ctx->saved_data["need_wf"] = wants_grad_opt(wf);
        ctx->save_for_backward(keep);
        return out;
    }

    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto saved = ctx->get_saved_variables();
        const int64_t n = ctx->saved_data["n"].toInt(), phi = ctx->saved_data["phi"].toInt();
        const int64_t bias_bits = ctx->saved_data["bias"].toInt();
        const double scale = ctx->saved_data["scale"].toDouble();
        const bool need_x = ctx->saved_data["need_x"].toBool(), need_wf = ctx->saved_data["need_wf"].toBool();
        const Tensor &x = saved[0], &wf = saved[1];
        const Tensor* const w = &saved[2];
        const Tensor* const y = &saved[2 + n];
        check_saved("x", x, g[0]);
        for (int64_t p = 0; p < n; ++p) check_saved("weight", w[p], g[0]);
        for (int64_t p = 0, i = 0; p < n; ++p)
            if ((phi >> p) & 1) check_saved("y", y[i++], g[0]);
        const int64_t rows = g[0].size(0) * g[0].size(1), e_out = w[0].size(0);
        TORCH_CHECK_VALUE(x.dim() == 3 && x.size(0) == g[0].size(0) && x.size(1) == g[0].size(1), "saved x ", x.sizes(),
                          " does not fit the gradient ", g[0].sizes());
        check_saved_layers(x, w, n, rows, e_out);
        for (int64_t p = 0, i = 0; p < n; ++p) {
            const Tensor& like = (phi >> p) & 1 ? y[i++] : g[p];
            TORCH_CHECK_VALUE(like.dim() == 4 && like.size(0) == x.size(0) && like.size(1) == x.size(1) && like.size(2) == g[0].size(2) &&
                                  like.size(2) * like.size(3) == e_out, "saved output ", like.sizes(), " does not fit ", rows, " rows of ", e_out);
        }
        const Tensor x2 = x.reshape({rows, x.size(2)});
        variable_list out(11);                    // x, wf, scale, heads, phi, w0, b0, w1, b1, w2, b2
        std::vector<bool> bias;
        for (int64_t p = 0; p < n; ++p) bias.push_back((bias_bits >> p) & 1);
        Tensor dwf;
        const bool own_x = need_x && own_input_grad(rows, w, n);
        std::vector<Tensor> dw;
        std::vector<OptTensor> db;
        if (own_x && (phi == 1 || phi == 3) &&
            project_grads(g, y, phi == 3 ? 2 : 1, wf, w, n, x, bias, scale, need_wf, out[0], dw, db, dwf)) {
            for (int64_t p = 0; p < n; ++p) {
                out[5 + 2 * p] = dw[p];
                out[6 + 2 * p] = opt(db[p]);
            }
        } else if (n == 3 && phi == 3 && need_x) {
            // [dy_q | dy_k | dv] side by side, written by the feature-map backward launch itself: one
            // GEMM for dx and one contraction for the three weight gradients
            Tensor packed;
            const Tensor g0 = g[0].contiguous(), g1 = g[1].contiguous(), g2 = g[2].contiguous();
            dwf = feature_grads(y[0], &y[1], wf, g0, &g1, &g2, packed, nullptr, true, scale, need_wf);
            const char* base = static_cast<const char*>(packed.data_ptr());
            const std::vector<const void*> dyp{base, base + 2 * e_out, base + 4 * e_out};
            out[0] = own_x ? input_grad(dyp, 3 * e_out, w, x) : at::mm(packed, at::cat({w[0], w[1], w[2]}, 0)).view(x.sizes());
            auto [dws, dbs] = param_grads(x2, {packed}, {bias_bits != 0});
            for (int64_t p = 0; p < n; ++p) {
                out[5 + 2 * p] = dws[0].narrow(0, p * e_out, e_out);
                if (bias[p]) out[6 + 2 * p] = dbs[0]->narrow(0, p * e_out, e_out);
            }
        } else {
            std::vector<Tensor> dys(n);
            if (phi == 3) {              // two of them: one launch
                const Tensor g0 = g[0].contiguous(), g1 = g[1].contiguous();
                dwf = feature_grads(y[0], &y[1], wf, g0, &g1, nullptr, dys[0], &dys[1], false, scale, need_wf);
            }
            for (int64_t p = 0; p < n; ++p) {
                if (!dys[p].defined()) {
                    dys[p] = g[p].contiguous();
                    if ((phi >> p) & 1) {        // the only one
                        const Tensor gp = dys[p];
                        dwf = feature_grads(y[0], nullptr, wf, gp, nullptr, nullptr, dys[p], nullptr, false, scale, need_wf);
                    }
                }
                dys[p] = dys[p].reshape({rows, -1});
            }
            bool own = own_x;
            for (const Tensor& dy : dys) own = own && aligned16(dy);
            std::vector<const void*> dyp;
            for (Tensor& dy : dys) dyp.push_back(ptr(dy));
            if (!own || !linear_grads(dyp, w[0].size(0), w, x, x2, bias, out[0], dw, db)) {
                if (own) out[0] = input_grad(dyp, w[0].size(0), w, x);
                for (int64_t p = 0; p < n && need_x && !own; ++p) {
                    out[0] = out[0].defined() ? out[0].addmm_(dys[p], w[p]) : at::mm(dys[p], w[p]);
                }
                std::tie(dw, db) = param_grads(x2, dys, bias);
            }
            for (int64_t p = 0; p < n; ++p) {
                out[5 + 2 * p] = dw[p];
                out[6 + 2 * p] = opt(db[p]);
            }
            if (out[0].defined()) out[0] = out[0].view(x.sizes());
        }
        out[1] = dwf;
        return out;
    }
};

constexpr int64_t kMaxProjectWidth = (int64_t)1 << 25;       // rfa_project_feature_map: 32-bit offsets within a row tile

// what the fused launch takes (rfa_amd/projection.py: fused_projection_supported)
bool plain_layers(const Tensor& x, const OptTensor& wf, const Layers& l, int64_t heads) {
    if (!plain_half(x, 3)) return false;
    const Tensor& w0 = l.w[0];
    for (size_t p = 0; p < l.w.size(); ++p)
        if (!plain_half(l.w[p], 2) || l.w[p].sizes() != w0.sizes() || !plain_half(l.b[p], 1)) return false;
    const int64_t out = w0.size(0), in = w0.size(1);
    if (in != x.size(2) || in % 64 != 0 || in > kMaxProjectWidth || out % heads != 0 || (out / heads != 64 && out / heads != 128)) return false;
    return !wf.has_value() ||
           (plain_half(*wf, 3) && (wf->size(1) == 32 || wf->size(1) == 64 || wf->size(1) == 128));
}

std::vector<Tensor> project(const Tensor& x, const OptTensor& wf, double scale, int64_t heads, const Layers& l) {
    bool grad = x.requires_grad() || wants_grad_opt(wf);
    int64_t phi = 0;
    for (size_t p = 0; p < l.w.size(); ++p) {
        grad = grad || l.w[p].requires_grad() || wants_grad_opt(l.b[p]);
        phi |= (int64_t)l.phi[p] << p;
    }
    auto w = [&](size_t p) { return p < l.w.size() ? OptTensor(l.w[p]) : c10::nullopt; };
    auto b = [&](size_t p) { return p < l.w.size() ? l.b[p] : c10::nullopt; };
    if (grad && at::GradMode::is_enabled())
        return ProjectNode::apply(x, wf, scale, heads, phi, w(0), b(0), w(1), b(1), w(2), b(2));
    std::vector<Tensor> wc, out;
    for (const Tensor& t : l.w) wc.push_back(t.contiguous());
    auto [ys, phis] = project_feature_map(x.contiguous(), wc, l.b, phi_flags(l),
                                          wf.has_value() ? OptTensor(wf->contiguous()) : c10::nullopt, heads, scale, false);
    for (size_t p = 0; p < l.w.size(); ++p) out.push_back(l.phi[p] ? *phis[p] : *ys[p]);
    return out;
}

// ---- one Linear layer by the projection kernel ------------------------------------------------
// heads of 64 columns and no feature map: the plain product
bool own_linear(const Tensor& x, const Tensor& w, const OptTensor& b) {
    const int64_t e_in = w.size(1), e_out = w.size(0), rows = e_in ? x.numel() / e_in : 0;
    return own_product(rows, e_out, e_in, 1) && e_in <= kMaxProjectWidth && e_in % 64 == 0 && e_out % 64 == 0 && e_in > 0 && e_out > 0 &&
           x.size(-1) == e_in && x.is_contiguous() && w.is_contiguous() && aligned16(x) && aligned16(w) &&
           w.device() == x.device() &&
           (!b.has_value() || (b->size(0) == e_out && b->is_contiguous() && aligned16(*b) && b->device() == x.device()));
}

Tensor projection(const Tensor& x, const Tensor& w, const OptTensor& b) {
    auto shape = x.sizes().vec();
    shape.back() = w.size(0);
    Tensor y = torch::empty(shape, x.options());
    std::array<const void*, 1> wp{ptr(w)}, bp{ptr(b)};
    std::array<void*, 1> yp{ptr(y)};
    Launch l(x);
    check_rc(rfa_project_feature_map(ptr(x), wp.data(), bp.data(), yp.data(), nullptr, 1, nullptr, x.numel() / w.size(1),
                                     (int)w.size(1), (int)(w.size(0) / 64), 32, 64, 0.f, l.stream));
    return y;
}

// ---- Linear layer on the way out ------------------------------------------------------------
struct LinearNode : public torch::autograd::Function<LinearNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x, const Tensor& w, const OptTensor& b) {
        ctx->saved_data["bias"] = b.has_value();
        ctx->saved_data["need_x"] = x.requires_grad();
        ctx->save_for_backward({x, w});
        if (own_linear(x, w, b)) return projection(x, w, b);
        return at::linear(x, w, b);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &x = saved[0], &w = saved[1];
        check_saved("x", x, g[0]);
        check_saved("weight", w, g[0]);
        const Tensor dy2 = g[0].reshape({-1, g[0].size(-1)}), x2 = x.reshape({-1, x.size(-1)});
        check_saved_layers(x, &w, 1, dy2.size(0), dy2.size(1));
        Tensor dx;
        const std::vector<bool> bias{ctx->saved_data["bias"].toBool()};
        if (ctx->saved_data["need_x"].toBool()) {
            const Tensor dyc = dy2.contiguous();
            const bool own = own_input_grad(dyc.size(0), &w, 1) && aligned16(dyc);
            std::vector<Tensor> dw;
            std::vector<OptTensor> db;
            if (own && linear_grads({ptr(dyc)}, w.size(0), &w, x, x2, bias, dx, dw, db)) return {dx, dw[0], opt(db[0])};
            dx = own ? input_grad({ptr(dyc)}, w.size(0), &w, x) : at::mm(dyc, w).view(x.sizes());
        }
        auto [dws, dbs] = param_grads(x2, {dy2}, bias);
        return {dx, dws[0], opt(dbs[0])};
    }
};

// Without autograd the row kernel takes up to 512 rows while its workgroups (64 rows x 32 columns) are at most one to
// a CU and the contraction is short (four waves share E_in), or a few rows of anything up to 192 M products.
// Device us there, row kernel / library: 512 -> 512 64 rows 2.8 / 5.6, 512 rows 3.9 / 5.2; 1024 -> 3072 64 rows 6.3 / 8.3,
// 128 rows 8.4 / 9.2; 768 -> 2304 96 rows 5.4 / 6.3; at worst 1024 -> 1024 320 rows 7.7 / 6.5; 2048 -> 2048 32 rows 7.7 /
// 8.4.  Past it two rounds of workgroups: 1024 -> 1024 768 rows 14.0 / 8.7; rows of x that every column tile reads again,
// from other XCDs' caches where they were just written (a layer's forward over 1024 rows of 512: 26.9 with the output
// projection by it, 25.0 by the projection kernel); a long contraction: 2048 -> 2048 64 rows 11.2 / 8.9.
// Widths that the projection kernel does not take stay with the library past 256 rows.
bool few_rows(int64_t R, int64_t e_in, int64_t e_out, int64_t cus) {
    if (R <= 32 && R * e_in * e_out <= (int64_t)192 << 20) return true;
    return e_in <= 1024 && R <= (e_in % 64 == 0 && e_out % 64 == 0 ? 512 : 256) &&
           (R + 63) / 64 * ((e_out + 31) / 32) <= cus;
}

// More rows go to the projection kernel, up to E_in = 1024 and 2^31 products, beyond that to the library: its tiles walk
// the contraction alone, 0.27 us per 32 columns of E_in however few they are.  Device us, projection kernel /
// library: 512 -> 512 2048 rows 7.3 / 7.2, 8192 10.3 / 11.3; 768 -> 768 768 rows 9.0 / 6.7, 2048 9.4 / 9.1; 1024 -> 1024 768
// rows 10.8 / 8.7, 2048 11.5 / 10.7; not taken: 1536 -> 1536 512 rows 15.2 / 9.4; 2048 -> 2048 64 rows 17.5 / 8.9, 512
// rows 19.0 / 11.3.  Both kernels may lose up to 2.4 us on the device to the library, for the 15 us of host time that
// each saves: a layer taking in one prompt of 512 tokens, E 1024, takes 63 us eagerly (130 through the library)
// and 53 from a replayed graph (51), 1024 tokens 66 (133) and 66 (58); a token for each of 64 sequences at E 2048, on
// the projection kernel 81 and 83, on the library 68 and 65.
constexpr int64_t kWidestOwnProjection = 1024;

// for the callers' condition (fp16, grad mode on, widths that are multiples of 128) see linear_out
OptTensor node_linear(const Tensor& x, const Tensor& w, const OptTensor& b) {
    if (!plain_mode() || at::autocast::is_autocast_enabled(at::kCUDA) || x.dim() < 1 || !plain_half(x, x.dim()) ||
        !plain_half(w, 2) || !plain_half(b, 1))
        return c10::nullopt;
    return LinearNode::apply(x, w, b);
}

// x W^T + b of n layers [e_out, e_in] side by side by the row kernel (for few_rows), where the tensors are as it takes them
OptTensor row_products(const Tensor& x, const Tensor* w, const OptTensor* b, int64_t n) {
    const int64_t e_out = w[0].size(0), e_in = w[0].size(1), R = e_in ? x.numel() / e_in : 0;
    if (R < 1 || e_out == 0 || e_in % 32 != 0 || e_out % 16 != 0 || x.size(-1) != e_in || !x.is_contiguous() || !aligned16(x))
        return c10::nullopt;
    std::array<const void*, 3> wp{}, bp{};
    for (int64_t p = 0; p < n; ++p) {
        if (w[p].size(0) != e_out || w[p].size(1) != e_in || !w[p].is_contiguous() || !aligned16(w[p]) || w[p].device() != x.device())
            return c10::nullopt;
        if (b[p].has_value() && (b[p]->size(0) != e_out || !b[p]->is_contiguous() || b[p]->device() != x.device())) return c10::nullopt;
        wp[p] = ptr(w[p]);
        bp[p] = ptr(b[p]);
    }
    auto shape = x.sizes().vec();
    shape.back() = n * e_out;
    Tensor y = torch::empty(shape, x.options());
    Launch l(x);
    check_rc(rfa_linear_rows_layers(ptr(x), wp.data(), bp.data(), (int)n, ptr(y), R, (int)e_in, (int)e_out, l.stream));
    return y;
}

// y = x W^T + b without autograd: few rows by the row kernel, more by the projection kernel, the largest products
// by the library (and all whenever autocast would choose the type).
OptTensor node_linear_rows(const Tensor& x, const Tensor& w, const OptTensor& b) {
    if (!plain_mode() || at::GradMode::is_enabled() || at::autocast::is_autocast_enabled(at::kCUDA) || x.dim() < 1 ||
        !plain_half(x, x.dim()) || !plain_half(w, 2) || !plain_half(b, 1))
        return c10::nullopt;
    const int64_t e_in = w.size(1), e_out = w.size(0), R = e_in ? x.numel() / e_in : 0;
    if (R < 1 || x.size(-1) != e_in) return c10::nullopt;
    if (!few_rows(R, e_in, e_out, at::cuda::getDeviceProperties(x.get_device())->multiProcessorCount))
        return e_in <= kWidestOwnProjection && R * e_in * e_out <= (int64_t)1 << 31 && own_linear(x, w, b)
                   ? OptTensor(projection(x, w, b)) : c10::nullopt;
    return row_products(x, &w, &b, 1);
}

// ---- what decoding keeps between calls --------------------------------------------------------
// Tensors that a value was made from, as rfa_amd/_derived.py remembers them: the very same objects (a weak reference
// keeps another from taking a dead one's place) in the very same state.
class Sources {
    struct Source {
        c10::weak_intrusive_ptr<at::TensorImpl> impl;
        uint32_t version;
        const void* data;
        std::vector<int64_t> sizes, strides;      // p.data = p.data.t() changes nothing but the strides
        at::ScalarType type;
        at::Device device;
    };
    std::vector<c10::optional<Source>> sources_;
    double extra_ = 0;

public:
    using List = std::vector<const OptTensor*>;
    static bool can_remember(const List& tensors) {      // inference tensors count no versions
        for (const OptTensor* t : tensors)
            if (t->has_value() && ((*t)->is_inference() || !(*t)->has_storage())) return false;
        return true;
    }
    bool same(const List& tensors, double extra) const {
        if (sources_.size() != tensors.size() || extra != extra_) return false;
        for (size_t i = 0; i < tensors.size(); ++i) {
            const auto& k = sources_[i];
            const OptTensor& t = *tensors[i];
            if (k.has_value() != t.has_value()) return false;
            if (k.has_value() && !(k->impl._unsafe_get_target() == t->unsafeGetTensorImpl() && k->version == t->_version() &&
                                   k->data == t->data_ptr() && k->sizes == t->sizes() && k->strides == t->strides() &&
                                   k->type == t->scalar_type() && k->device == t->device()))
                return false;
        }
        return true;
    }
    void remember(const List& tensors, double extra) {
        sources_.clear();
        for (const OptTensor* t : tensors) {
            if (!t->has_value()) sources_.emplace_back(c10::nullopt);
            else
                sources_.emplace_back(Source{c10::weak_intrusive_ptr<at::TensorImpl>((*t)->getIntrusivePtr()), (uint32_t)(*t)->_version(),
                                             (*t)->data_ptr(), (*t)->sizes().vec(), (*t)->strides().vec(),
                                             (*t)->scalar_type(), (*t)->device()});
        }
        extra_ = extra;
    }
};

// The scaled matrices W' and the stacked q, k, v layer of one CausalAttention, and with them the first half of a decoding
// step: rows [T, B, 3, H, d] of all three projections, W' and the tensors that the step writes its state to (none where it
// stays in place).  In Python this half costs 16 us of a step whose kernels take 11 (four sequences of 8 heads).
// What a stream made is for its own kernels alone: another one has nothing to wait on, and memory given back is used
// again by the stream that it came from.  A captured step forms what it needs anew: kept tensors would die under the graph
// with the next change of a parameter, and the graph's own hold nothing before its first replay.  Few rows then take the
// layers where they are: 4 sequences of 8 heads of 64 11.7 us a replay, 64 of 16 25.9 (with stacks of weights and biases 16.6
// and 33.4; with kept ones 9.7 and 23.2).  The kept stack stays where it can: one launch over it is 0.1 to 0.5 shorter.
class DecodeCache {
    struct Kept {
        hipStream_t stream = nullptr;
        Sources matrix_sources, layer_sources;
        Tensor w, weight;
        OptTensor bias;
    };
    static constexpr size_t kStreams = 4;
    std::vector<Kept> kept_;       // the stream used last comes first

    Kept& kept(hipStream_t stream) {
        size_t i = 0;
        while (i < kept_.size() && kept_[i].stream != stream) ++i;
        if (i == kept_.size()) {
            if (i == kStreams) kept_.pop_back();
            kept_.emplace_back();
            kept_.back().stream = stream;
            i = kept_.size() - 1;
        }
        std::rotate(kept_.begin(), kept_.begin() + i, kept_.begin() + i + 1);
        return kept_.front();
    }

public:
    using Rows = std::tuple<Tensor, Tensor, OptTensor, OptTensor>;
    c10::optional<Rows> rows(const Tensor& x, const Tensor& matrices, const OptTensor& sigma, double tau, const OptTensor& wq,
                             const OptTensor& bq, const OptTensor& wk, const OptTensor& bk, const OptTensor& wv,
                             const OptTensor& bv, int64_t heads, const Tensor& s, const Tensor& z, bool in_place) {
        if (!plain_mode() || at::GradMode::is_enabled() || at::autocast::is_autocast_enabled(at::kCUDA) || !plain_half(x, 3) ||
            !plain_matrices(matrices, sigma, tau) || !plain(s, torch::kFloat32, 4) || !plain(z, torch::kFloat32, 3) ||
            !s.is_contiguous() || !z.is_contiguous())
            return c10::nullopt;
        const int64_t E = x.size(2);
        for (const OptTensor* w : {&wq, &wk, &wv})
            if (!w->has_value() || !plain_half(**w, 2) || (*w)->size(0) != E || (*w)->size(1) != E) return c10::nullopt;
        for (const OptTensor* b : {&bq, &bk, &bv})
            if (b->has_value() != bq.has_value() || !plain_half(*b, 1)) return c10::nullopt;
        const OptTensor m(matrices);
        const Sources::List ms{&m, &sigma}, ls{&wq, &bq, &wk, &bk, &wv, &bv};
        if (heads < 1 || E % heads != 0 || !Sources::can_remember(ms) || !Sources::can_remember(ls)) return c10::nullopt;
        const hipStream_t stream = c10::hip::getCurrentHIPStream(x.get_device()).stream();
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        if (stream) C10_HIP_CHECK(hipStreamIsCapturing(stream, &status));      // the default stream cannot be
        const bool capturing = status != hipStreamCaptureStatusNone;
        Kept captured;
        Kept& c = capturing ? captured : kept(stream);
        if (!c.matrix_sources.same(ms, tau)) {
            c.w = build_random_matrices(matrices.contiguous(), sigma.has_value() ? OptTensor(sigma->contiguous()) : c10::nullopt, tau);
            c.matrix_sources.remember(ms, tau);
        }
        OptTensor y;
        if (capturing) {      // few rows: the layers where they are, the bits of their stack
            const std::array<Tensor, 3> w{*wq, *wk, *wv};
            const std::array<OptTensor, 3> b{bq, bk, bv};
            if (few_rows(x.size(0) * x.size(1), E, 3 * E, at::cuda::getDeviceProperties(x.get_device())->multiProcessorCount))
                y = row_products(x, w.data(), b.data(), 3);
        }
        if (!y.has_value()) {
            if (!c.layer_sources.same(ls, 0)) {
                c.weight = at::cat({*wq, *wk, *wv}, 0);
                c.bias = bq.has_value() ? OptTensor(at::cat({*bq, *bk, *bv}, 0)) : c10::nullopt;
                c.layer_sources.remember(ls, 0);
            }
            y = node_linear_rows(x, c.weight, c.bias);
            if (!y.has_value()) y = at::linear(x, c.weight, c.bias);
        }
        auto fresh = [&](const Tensor& t) { return in_place ? c10::nullopt : OptTensor(torch::empty_like(t)); };
        return Rows{y->view({x.size(0), x.size(1), 3, heads, E / heads}), c.w, fresh(s), fresh(z)};
    }
};

// ---- causal attention -------------------------------------------------------------------------
// phi_q, phi_k [T, B, H, K], v [T, B, H, d] -> attn [T, B, H * d], through the saving pair
struct ScanDims {
    int64_t T, N;
    int K, d;
    explicit ScanDims(const Tensor& q, const Tensor& v)
        : T(q.size(0)), N(q.size(1) * q.size(2)), K((int)q.size(3)), d((int)v.size(3)) {}
};

Tensor scan_output(const Tensor& v) { return torch::empty({v.size(0), v.size(1), v.size(2) * v.size(3)}, v.options()); }

// rows of t [T, B, H, K] whose key is padded set to zero: of a copy, or where they are
void mask_rows(const Tensor& src, const Tensor& dst, const Tensor& pad) {
    Launch l(src);
    check_rc(rfa_mask_rows(ptr(src), ptr(dst), static_cast<const uint8_t*>(pad.data_ptr()), pad.stride(0), pad.stride(1),
                           src.size(0), src.size(1), src.size(2) * src.size(3), l.stream));
}

Tensor masked_keys(const Tensor& phi_k, const OptTensor& pad) {
    const Tensor k = phi_k.contiguous();
    if (!pad.has_value()) return k;
    Tensor out = torch::empty_like(k);
    mask_rows(k, out, *pad);
    return out;
}

// [B, T] of any type and strides on the tensors' device (bools are read where they are)
bool plain_pad(const OptTensor& pad, const Tensor& k) {
    return !pad.has_value() ||
           (plain(*pad, pad->scalar_type(), 2) && !pad->is_complex() && pad->size(0) == k.size(1) &&
            pad->size(1) == k.size(0) && pad->device() == k.device() && aligned16(k) && k.size(2) * k.size(3) % 8 == 0);
}

struct CausalNode : public torch::autograd::Function<CausalNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& phi_q, const Tensor& phi_k, const Tensor& values,
                          const OptTensor& pad) {
        const Tensor q = phi_q.contiguous(), k = masked_keys(phi_k, pad), v = values.contiguous();
        const ScanDims n(q, v);
        Tensor attn = scan_output(v);
        Launch l(q);
        const size_t nbytes = rfa_causal_forward_workspace_bytes(n.T, n.N, n.K, n.d);
        const size_t sbytes = rfa_causal_saved_state_bytes(n.T, n.N, n.K, n.d);
        Tensor ws = workspace(nbytes, q), state = workspace(sbytes, q);
        check_rc(rfa_causal_forward_save(ptr(q), ptr(k), ptr(v), ptr(attn), ptr(state), sbytes, n.T, n.N, n.K, n.d, ptr(ws),
                                         nbytes, l.stream));
        ctx->save_for_backward({q, k, v, attn, state, opt(pad)});
        return attn;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &q = saved[0], &k = saved[1], &v = saved[2], &state = saved[4], &pad = saved[5];
        const Tensor attn = saved[3].contiguous(), grad = g[0].contiguous();
        check_half("q", q, 4);
        check_half("k", k, 4);
        check_half("v", v, 4);
        check_half("out", attn, 3);
        for (const Tensor* t : {&k, &v, &attn, &grad}) check_saved("a saved tensor", *t, q);
        const ScanDims n(q, v);
        TORCH_CHECK_VALUE(k.sizes() == q.sizes() && v.size(0) == n.T && v.size(1) == q.size(1) && v.size(2) == q.size(2) &&
                              attn.numel() == v.numel() && grad.numel() == v.numel(),
                          "saved q ", q.sizes(), ", k ", k.sizes(), ", v ", v.sizes(), ", out ", attn.sizes(), " do not fit");
        TORCH_CHECK_TYPE(state.is_cuda() && state.device() == q.device() && state.scalar_type() == torch::kUInt8 &&
                             state.is_contiguous(), "saved must be the byte buffer of the forward");
        if (pad.defined())
            TORCH_CHECK_VALUE(pad.device() == q.device() && pad.scalar_type() == torch::kBool && pad.dim() == 2 &&
                                  pad.size(0) == q.size(1) && pad.size(1) == n.T, "saved key_padding_mask does not fit");
        Tensor dq = torch::empty_like(q), dk = torch::empty_like(k), dv = torch::empty_like(v);
        Launch l(q);
        const size_t nbytes = rfa_causal_backward_saved_workspace_bytes(ptr(state), n.T, n.N, n.K, n.d);
        Tensor ws = workspace(nbytes, q);
        check_rc(rfa_causal_backward_saved(ptr(q), ptr(k), ptr(v), ptr(grad), ptr(attn), ptr(state), (size_t)state.numel(),
                                           ptr(dq), ptr(dk), ptr(dv), n.T, n.N, n.K, n.d, ptr(ws), nbytes, l.stream));
        if (pad.defined()) mask_rows(dk, dk, pad);
        return {dq, dk, dv, Tensor()};
    }
};

bool plain_scan(const Tensor& q, const Tensor& k, const Tensor& v) {
    return plain_half(q, 4) && plain_half(k, 4) && plain_half(v, 4) && q.sizes() == k.sizes() && v.size(0) == q.size(0) &&
           v.size(1) == q.size(1) && v.size(2) == q.size(2) && q.device() == k.device() && q.device() == v.device();
}

Tensor causal(const Tensor& phi_q, const Tensor& phi_k, const Tensor& values, const OptTensor& pad) {
    if (wants_grad(phi_q, phi_k, values)) return CausalNode::apply(phi_q, phi_k, values, pad);
    const Tensor q = phi_q.contiguous(), k = masked_keys(phi_k, pad), v = values.contiguous();
    const ScanDims n(q, v);
    Tensor attn = scan_output(v);
    Launch l(q);
    const size_t nbytes = rfa_causal_forward_workspace_bytes(n.T, n.N, n.K, n.d);
    Tensor ws = workspace(nbytes, q);
    check_rc(rfa_causal_forward(ptr(q), ptr(k), ptr(v), ptr(attn), n.T, n.N, n.K, n.d, ptr(ws), nbytes, l.stream));
    return attn;
}

OptTensor node_causal(const Tensor& phi_q, const Tensor& phi_k, const Tensor& v, const OptTensor& pad) {
    if (!plain_mode() || !plain_scan(phi_q, phi_k, v) || !plain_pad(pad, phi_k)) return c10::nullopt;
    return causal(phi_q, phi_k, v, pad.has_value() ? OptTensor(pad->to(torch::kBool)) : c10::nullopt);
}

// A prompt without autograd: q, k, v [T, B, H, d] -> (attn [T, B, H * d], s [B, H, 2D, d], z [B, H, 2D]), the
// feature maps inside the scan; nothing where the sequences do not fill the chip or a tensor is not plain.
c10::optional<std::tuple<Tensor, Tensor, Tensor>> node_prefill(const Tensor& q, const Tensor& k, const Tensor& v,
                                                               const Tensor& w, double scale) {
    if (!plain_mode() || !plain_scan(q, k, v) || !plain_half(w, 3) || q.size(3) != v.size(3) || w.size(0) != q.size(2) ||
        w.size(2) != q.size(3) || w.device() != q.device() || !q.is_contiguous() || !k.is_contiguous() || !v.is_contiguous() ||
        !w.is_contiguous() || !aligned16(q) || !aligned16(k) || !aligned16(v) || !aligned16(w))
        return c10::nullopt;
    const int64_t T = q.size(0), B = q.size(1), H = q.size(2), d = q.size(3), D = w.size(1);
    if (!rfa_causal_prefill_rows_supported(T, B * H, (int)D, (int)d)) return c10::nullopt;
    const auto f32 = q.options().dtype(torch::kFloat32);
    Tensor attn = scan_output(v), s = torch::empty({B, H, 2 * D, d}, f32), z = torch::empty({B, H, 2 * D}, f32);
    Launch l(q);
    check_rc(rfa_causal_prefill_rows(ptr(q), ptr(k), ptr(v), ptr(w), (float)scale, ptr(attn), s.data_ptr<float>(),
                                     z.data_ptr<float>(), T, B, (int)H, (int)D, (int)d, l.stream));
    return std::tuple(attn, s, z);
}

// q, k, v projections, phi(q) and phi(k), the scan: x [T, B, E] -> attn [T, B, H * d].  `matrices` is
// W' itself where `build` is false.
OptTensor node_causal_layer(const Tensor& x, const Tensor& matrices, const OptTensor& sigma, double tau, bool build,
                            const std::vector<Tensor>& weights, const std::vector<OptTensor>& biases, int64_t heads,
                            double scale) {
    Layers l{weights, biases, {true, true, false}};
    if (!plain_mode() || weights.size() != 3 || biases.size() != 3 || !plain_layers(x, matrices, l, heads) ||
        (build && !plain_matrices(matrices, sigma, tau)))
        return c10::nullopt;
    const Tensor w = build ? build_matrices(matrices, sigma, tau) : matrices;
    const auto out = project(x, w, scale, heads, l);
    return causal(out[0], out[1], out[2], c10::nullopt);
}

// ---- quadratic form with explicit masks ---------------------------------------------------------
struct MaskedNode : public torch::autograd::Function<MaskedNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& phi_q, const Tensor& phi_k, const Tensor& values,
                          const OptTensor& pad, const OptTensor& mask, const OptTensor& mask_t) {
        const Tensor q = phi_q.contiguous(), k = phi_k.contiguous(), v = values.contiguous();
        auto [out, rsum] = masked_forward(q.flatten(1, 2), k.flatten(1, 2), v.flatten(1, 2), q.size(2), pad, mask);
        Tensor attn = at::_unsafe_view(out, {v.size(0), v.size(1), v.size(2) * v.size(3)});
        ctx->saved_data["pad"] = pad;
        ctx->saved_data["mask"] = mask;
        ctx->saved_data["mask_t"] = mask_t;
        ctx->save_for_backward({q, k, v, attn, rsum});
        return attn;
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &q = saved[0], &k = saved[1], &v = saved[2];
        const Tensor v3 = v.flatten(1, 2);
        auto mask = [&](const char* name) { return ctx->saved_data[name].toOptional<Tensor>(); };
        auto grads = masked_backward(q.flatten(1, 2), k.flatten(1, 2), v3, g[0].contiguous().view(v3.sizes()),
                                     saved[3].contiguous().view(v3.sizes()), saved[4], q.size(2), mask("pad"), mask("mask"),
                                     mask("mask_t"));
        return {grads[0].view(q.sizes()), grads[1].view(k.sizes()), grads[2].view(v.sizes()), Tensor(), Tensor(), Tensor()};
    }
};

OptTensor node_masked(const Tensor& phi_q, const Tensor& phi_k, const Tensor& v, const OptTensor& pad, const OptTensor& mask,
                      const OptTensor& mask_t) {
    if (!plain_mode() || !plain_scan(phi_q, phi_k, v) || phi_q.numel() == 0 || !wants_grad(phi_q, phi_k, v))
        return c10::nullopt;
    return MaskedNode::apply(phi_q, phi_k, v, pad, mask, mask_t);
}

// ---- cross attention ------------------------------------------------------------------------------
struct CrossStateNode : public torch::autograd::Function<CrossStateNode> {
    static variable_list forward(AutogradContext* ctx, const Tensor& phi_k, const Tensor& values, const OptTensor& pad) {
        const Tensor k = phi_k.contiguous(), v = values.contiguous();
        auto [s, z] = cross_state(k, v, pad);
        ctx->saved_data["pad"] = pad;
        ctx->save_for_backward({k, v});
        return {s, z};
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto saved = ctx->get_saved_variables();
        auto [dk, dv] = cross_state_backward(saved[0], saved[1], g[0].contiguous(), g[1].contiguous(),
                                             ctx->saved_data["pad"].toOptional<Tensor>());
        return {dk, dv, Tensor()};
    }
};

// phi_q [T, B, H, K], s, z -> attn [T, B, H * d]
struct CrossReadoutNode : public torch::autograd::Function<CrossReadoutNode> {
    static Tensor forward(AutogradContext* ctx, const Tensor& phi_q, const Tensor& s, const Tensor& z) {
        const Tensor q = phi_q.contiguous(), sc = s.contiguous(), zc = z.contiguous();
        ctx->save_for_backward({q, sc, zc});
        const Tensor out = cross_readout(q, sc, zc);
        return at::_unsafe_view(out, {out.size(0), out.size(1), out.size(2) * out.size(3)});
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &q = saved[0], &s = saved[1];
        auto [dq, ds, dz] = cross_readout_backward(q, s, saved[2],
                                                   g[0].contiguous().view({q.size(0), q.size(1), q.size(2), s.size(3)}));
        return {dq, ds, dz};
    }
};

// the source side of a layer: enc [S, B, E], pad [B, S] -> (s, z, W')
c10::optional<std::tuple<Tensor, Tensor, Tensor>> node_cross_source(
    const Tensor& enc, const Tensor& matrices, const OptTensor& sigma, double tau, const std::vector<Tensor>& weights,
    const std::vector<OptTensor>& biases, int64_t heads, double scale, const OptTensor& pad) {
    Layers l{weights, biases, {true, false, false}};
    if (!plain_mode() || weights.size() != 2 || biases.size() != 2 || !plain_layers(enc, matrices, l, heads) ||
        !plain_matrices(matrices, sigma, tau))
        return c10::nullopt;
    const Tensor w = build_matrices(matrices, sigma, tau);
    const auto out = project(enc, w, scale, heads, l);
    if (wants_grad(out[0], out[1])) {
        const auto state = CrossStateNode::apply(out[0], out[1], pad);
        return std::tuple(state[0], state[1], w);
    }
    auto [s, z] = cross_state(out[0], out[1], pad);
    return std::tuple(s, z, w);
}

// the target side up to the output projection: query [T, B, E] -> attn [T, B, H * d]
OptTensor node_cross_query(const Tensor& query, const Tensor& w, const Tensor& weight, const OptTensor& bias, int64_t heads,
                           double scale, const Tensor& s, const Tensor& z) {
    Layers l{{weight}, {bias}, {true, false, false}};
    if (!plain_mode() || !plain_layers(query, w, l, heads) || !plain(s, torch::kFloat32, 4) || !plain(z, torch::kFloat32, 3))
        return c10::nullopt;
    if (query.size(0) == 1 && !at::GradMode::is_enabled() && s.is_contiguous() && z.is_contiguous() && w.is_contiguous()) {
        // one step: the row kernel for q, then feature map and readout in one launch
        const int64_t B = query.size(1), d = weight.size(0) / heads, D = w.size(1);
        const bool fits = s.size(0) == B && s.size(1) == heads && s.size(2) == 2 * D && s.size(3) == d && z.size(0) == B &&
                          z.size(1) == heads && z.size(2) == 2 * D && w.size(0) == heads && w.size(2) == d &&
                          aligned16(s) && aligned16(z) && aligned16(w) && s.device() == query.device() &&
                          z.device() == query.device() && w.device() == query.device();
        const OptTensor q = fits ? node_linear_rows(query, weight, bias) : c10::nullopt;
        if (q.has_value()) {
            Tensor out = torch::empty_like(*q);
            Launch g(query);
            check_rc(rfa_cross_step(ptr(*q), ptr(w), (float)scale, s.data_ptr<float>(), z.data_ptr<float>(), ptr(out), B,
                                    (int)heads, (int)D, (int)d, g.stream));
            return out;
        }
    }
    const auto phi_q = project(query, w, scale, heads, l)[0];
    if (wants_grad(phi_q, s, z)) return CrossReadoutNode::apply(phi_q, s, z);
    const Tensor out = cross_readout(phi_q, s.contiguous(), z.contiguous());
    return out.view({out.size(0), out.size(1), out.size(2) * out.size(3)});
}

void bind_nodes(pybind11::module_& m) {
    namespace py = pybind11;
    m.def("node_plain", &node_plain, py::arg("t"));
    py::class_<DecodeCache>(m, "DecodeCache").def(py::init<>()).def("rows", &DecodeCache::rows);
    // each of the others returns None where the call is not plain: the caller's general path takes it
    m.def("node_random_project", &node_random_project, py::arg("x"), py::arg("w"), py::arg("scale"));
    m.def("node_linear", &node_linear, py::arg("x"), py::arg("weight"), py::arg("bias"));
    m.def("node_linear_rows", &node_linear_rows, py::arg("x"), py::arg("weight"), py::arg("bias"));
    m.def("node_causal", &node_causal, py::arg("phi_q"), py::arg("phi_k"), py::arg("v"),
          py::arg("key_padding_mask") = py::none());
    m.def("node_prefill", &node_prefill, py::arg("q"), py::arg("k"), py::arg("v"), py::arg("w"), py::arg("scale"));
    m.def("node_causal_layer", &node_causal_layer, py::arg("x"), py::arg("matrices"), py::arg("sigma"), py::arg("tau"),
          py::arg("build"), py::arg("weights"), py::arg("biases"), py::arg("heads"), py::arg("scale"));
    m.def("node_masked", &node_masked, py::arg("phi_q"), py::arg("phi_k"), py::arg("v"), py::arg("key_padding_mask"),
          py::arg("mask"), py::arg("mask_t"));
    m.def("node_cross_source", &node_cross_source, py::arg("enc"), py::arg("matrices"), py::arg("sigma"), py::arg("tau"),
          py::arg("weights"), py::arg("biases"), py::arg("heads"), py::arg("scale"), py::arg("key_padding_mask"));
    m.def("node_cross_query", &node_cross_query, py::arg("query"), py::arg("w"), py::arg("weight"), py::arg("bias"),
          py::arg("heads"), py::arg("scale"), py::arg("s"), py::arg("z"));
}

}  // namespace
