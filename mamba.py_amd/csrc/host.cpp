// Host side of the operators: argument checks, allocation, autograd nodes and the calls into
// libmambapy_amd.so, as a Python extension module over PyTorch's C++ API.
//
// The kernels of a small call take microseconds, so the work around them decides what the call
// costs.  Written in Python (an autograd.Function, a ctypes call with twenty arguments, a dozen
// torch.empty), forward + backward of a tiny scan spent 200 us on the host for 28 us of kernels;
// here every operator is one call from Python, one graph node and the launches.
#include "host.h"

namespace mpa_host {
namespace {

// ---- fused selective scan -----------------------------------------------------------------------

mpa_sscan_shape sscan_shape(const Tensor& x, const Tensor& delta, const Tensor& B, const Tensor& y, const Tensor& g,
                            const Tensor& dbc, int64_t N, int flags, const Tensor& z, const Plan& plan, bool backward) {
    mpa_sscan_shape s{};
    s.batch = x.size(0); s.seqlen = x.size(1); s.dim = x.size(2); s.dstate = N;
    s.io_dtype = io_dtype(x.scalar_type());
    s.flags = flags;
    s.u_sb = x.stride(0); s.u_sl = x.stride(1); s.u_sd = x.stride(2);
    if (z.defined()) { s.z_sb = z.stride(0); s.z_sl = z.stride(1); s.z_sd = z.stride(2); }
    s.d_sb = delta.stride(0); s.d_sl = delta.stride(1); s.d_sd = delta.stride(2);
    // delta may be float32 next to bfloat16 tensors (the reference's call under autocast,
    // mambapy/mamba.py:264-265): it is read, and its gradient written, as float32
    s.delta_dtype = delta.scalar_type() == at::kFloat && x.scalar_type() != at::kFloat ? MPA_DELTA_F32 : 0;
    s.y_sb = y.stride(0); s.y_sl = y.stride(1); s.y_sd = y.stride(2);
    s.g_sb = g.stride(0); s.g_sl = g.stride(1); s.g_sd = g.stride(2);
    s.bc_sb = B.stride(0); s.bc_sl = B.stride(1);
    s.dbc_sb = dbc.stride(0); s.dbc_sl = dbc.stride(1);
    s.plan_states_per_lane = backward ? plan.bwd_ns : plan.fwd_ns;
    s.plan_segments = backward ? plan.bwd_segments : plan.fwd_segments;
    s.plan_flags = plan.flags;
    return s;
}

struct ScanBackward : public Node {
    SavedVariable x, delta, A, B, C, D, z, bias, h0, ckpt, y_pre;
    int flags = 0;
    Plan plan;
    std::array<at::ScalarType, 8> dtypes;  // of the caller's x, delta, A, B, C, D, z, bias
    std::string name() const override { return "SelectiveScanBackward"; }
    void release_variables() override {
        for (SavedVariable* v : {&x, &delta, &A, &B, &C, &D, &z, &bias, &h0, &ckpt, &y_pre}) v->reset_data();
    }
    variable_list apply(variable_list&& grads) override;
};

variable_list ScanBackward::apply(variable_list&& grads) {
    variable_list out(8);
    Tensor dy = grads[0];
    if (!dy.defined()) return out;
    // (unpacked outside of the guard, here and in the other nodes: a hook may run a whole forward pass)
    const Tensor x_ = x.unpack(), delta_ = delta.unpack(), A_ = dense(A.unpack()), D_ = dense(D.unpack()), z_ = z.unpack(),
                 bias_ = dense(bias.unpack()), h0_ = dense(h0.unpack()), ckpt_ = dense(ckpt.unpack()), y_pre_ = y_pre.unpack();
    Tensor B_ = unit_rows(B.unpack()), C_ = unit_rows(C.unpack());
    if (B_.strides() != C_.strides()) { B_ = B_.contiguous(); C_ = C_.contiguous(); }
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x_.device());
    const auto dt = x_.scalar_type();
    const int64_t Bs = x_.size(0), L = x_.size(1), ED = x_.size(2), N = A_.size(1);
    dy = cast(dy, dt);
    // the saved pre-gate output is addressed with dy's strides
    if (y_pre_.defined() && dy.strides() != y_pre_.strides()) dy = dy.contiguous();
    const Tensor dx = empty({Bs, L, ED}, dt, x_), ddelta = empty({Bs, L, ED}, delta_.scalar_type(), x_);
    const Tensor dz = z_.defined() ? empty({Bs, L, ED}, dt, x_) : Tensor();
    const Tensor dB = empty({Bs, L, N}, dt, x_), dC = empty({Bs, L, N}, dt, x_);
    const Tensor dA = empty({ED, N}, at::kFloat, x_), dD = empty({ED}, at::kFloat, x_);
    const Tensor dbias = bias_.defined() ? empty({ED}, at::kFloat, x_) : Tensor();
    const mpa_sscan_shape s = sscan_shape(x_, delta_, B_, dy, dx, dB, N, flags, z_, plan, true);
    const size_t nbytes = mpa_sscan_bwd_workspace_bytes(&s);
    const Tensor ws = scratch(nbytes, x_);
    check(mpa_sscan_bwd(&s, ptr(x_), ptr(delta_), fptr(A_), ptr(B_), ptr(C_), fptr(D_), ptr(z_), fptr(bias_), fptr(h0_), ptr(dy),
                        ptr(y_pre_), fptr(ckpt_), ptr(dx), ptr(ddelta), fptr(dA), ptr(dB), ptr(dC), fptr(dD), ptr(dz), fptr(dbias),
                        ptr(ws), nbytes, stream_of(x_)),
          "mpa_sscan_bwd");
    const std::array<Tensor, 8> g = {dx, ddelta, dA, dB, dC, dD, dz, dbias};
    for (size_t i = 0; i < 8; ++i) out[i] = grad_as(g[i], dtypes[i]);
    return out;
}

std::tuple<Tensor, Opt> scan_fwd(const Tensor& x, const Tensor& delta_in, const Tensor& A_in, const Tensor& B_in, const Tensor& C_in,
                                 const Tensor& D_in, const Opt& z_in, const Opt& bias_in, bool softplus, const Opt& h0_in,
                                 bool return_last, bool reverse, const PackedPlan& packed) {
    const Tensor zc = val(z_in), bc = val(bias_in), hc = val(h0_in);
    require_gpu({&x, &delta_in, &A_in, &B_in, &C_in, &D_in, &zc, &bc, &hc});
    require_plain({&x, &delta_in, &A_in, &B_in, &C_in, &D_in, &zc, &bc, &hc});
    const Plan plan = unpack(packed);
    const auto dt = x.scalar_type();
    io_dtype(dt);
    TORCH_CHECK(x.dim() == 3 && A_in.dim() == 2, "x must be (B, L, ED) and A (ED, N), got x", x.sizes(), " A", A_in.sizes());
    const int64_t Bs = x.size(0), L = x.size(1), ED = x.size(2), N = A_in.size(1);
    TORCH_CHECK(delta_in.sizes() == x.sizes() && A_in.size(0) == ED && B_in.sizes() == at::IntArrayRef({Bs, L, N}) &&
                    C_in.sizes() == B_in.sizes() && D_in.sizes() == at::IntArrayRef({ED}),
                "shape mismatch: x", x.sizes(), " delta", delta_in.sizes(), " A", A_in.sizes(), " B", B_in.sizes(), " C", C_in.sizes(),
                " D", D_in.sizes());
    TORCH_CHECK(!zc.defined() || zc.sizes() == x.sizes(), "z must have the shape of x");
    TORCH_CHECK(!bc.defined() || softplus, "delta_bias needs delta_softplus=True");
    TORCH_CHECK(!bc.defined() || bc.numel() == ED, "delta_bias must have ", ED, " elements, got ", bc.sizes());
    TORCH_CHECK(!hc.defined() || hc.numel() == Bs * ED * N, "h0 must be (B, ED, N), got ", hc.sizes());
    // whether a backward can follow decides what is kept: checkpoints (and the pre-gate output)
    // are written only then; without them the library may also cut a sequence more finely
    const bool need_grad = tracked({&x, &delta_in, &A_in, &B_in, &C_in, &D_in, &zc, &bc});
    TORCH_CHECK(!(need_grad && hc.defined() && hc.requires_grad()),
                "selective_scan_fn: no gradient is computed for h0; pass h0.detach()");
    std::shared_ptr<ScanBackward> node;
    if (need_grad) node = make_node<ScanBackward>({&x, &delta_in, &A_in, &B_in, &C_in, &D_in, &zc, &bc});
    Tensor y, h_last;
    Tensor delta, A, B, C, D, z, bias, h0, ckpt, y_pre;
    const int flags = (softplus ? MPA_SSCAN_DELTA_SOFTPLUS : 0) | (reverse ? MPA_SSCAN_REVERSE : 0);
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x.device());
        // the general backward kernel, which only a pinned plan selects, has no float32 delta
        const bool wide = delta_in.scalar_type() == at::kFloat && dt == at::kBFloat16 && !(plan.flags & MPA_PLAN_BWD_GENERAL);
        delta = wide ? delta_in : cast(delta_in, dt);
        B = unit_rows(cast(B_in, dt));
        C = unit_rows(cast(C_in, dt));
        if (B.strides() != C.strides()) { B = B.contiguous(); C = C.contiguous(); }
        z = cast(zc, dt);
        A = f32c(A_in);
        D = f32c(D_in);
        bias = f32c(bc);
        h0 = f32c(hc);
        y = empty({Bs, L, ED}, dt, x);
        const mpa_sscan_shape s = sscan_shape(x, delta, B, y, y, B, N, flags, z, plan, false);
        if (need_grad) {
            ckpt = empty({mpa_sscan_ckpt_elems(&s)}, at::kFloat, x);
            if (z.defined()) y_pre = empty({Bs, L, ED}, dt, x);  // output before the gate, read again by the backward
        }
        if (return_last) h_last = empty({Bs, ED, N}, at::kFloat, x);
        const size_t nbytes = mpa_sscan_fwd_workspace_bytes(&s, need_grad ? 1 : 0);
        const Tensor ws = scratch(nbytes, x);
        check(mpa_sscan_fwd(&s, ptr(x), ptr(delta), fptr(A), ptr(B), ptr(C), fptr(D), ptr(z), fptr(bias), fptr(h0), ptr(y), ptr(y_pre),
                            fptr(ckpt), fptr(h_last), ptr(ws), nbytes, stream_of(x)),
              "mpa_sscan_fwd");
    }
    if (node) {
        node->flags = flags;
        node->plan = plan;
        node->x = keep(x); node->delta = keep(delta); node->A = keep(A); node->B = keep(B); node->C = keep(C); node->D = keep(D);
        node->z = keep(z); node->bias = keep(bias); node->h0 = keep(h0); node->ckpt = keep(ckpt); node->y_pre = keep(y_pre);
        const std::array<const Tensor*, 8> in = {&x, &delta_in, &A_in, &B_in, &C_in, &D_in, &zc, &bc};
        for (size_t i = 0; i < 8; ++i) node->dtypes[i] = in[i]->defined() ? in[i]->scalar_type() : at::kFloat;
        torch::autograd::set_history(y, node);
    }
    return {y, return_last ? Opt(h_last) : Opt()};
}

// ---- generic scan -------------------------------------------------------------------------------

mpa_pscan_shape pscan_shape(const Tensor& A, const Tensor& X, const Tensor& H, const Tensor& gA, const Tensor& gX, bool reverse,
                            int chunks) {
    mpa_pscan_shape s{};
    s.batch = X.size(0); s.seqlen = X.size(1); s.dim = X.size(2); s.dstate = X.size(3);
    s.io_dtype = io_dtype(X.scalar_type());
    s.reverse = reverse ? 1 : 0;
    s.plan_chunks = chunks;
    auto put = [](int64_t (&dst)[4], const Tensor& t) {
        if (t.defined())
            for (int i = 0; i < 4; ++i) dst[i] = t.stride(i);
    };
    put(s.a_st, A); put(s.x_st, X); put(s.h_st, H); put(s.ga_st, gA); put(s.gx_st, gX);
    return s;
}

struct PScanBackward : public Node {
    SavedVariable A, H;
    bool reverse = false;
    int chunks = 0;
    at::ScalarType ta, tx;
    std::string name() const override { return "PScanBackward"; }
    void release_variables() override { A.reset_data(); H.reset_data(); }
    variable_list apply(variable_list&& grads) override {
        variable_list out(2);
        if (!grads[0].defined()) return out;
        const Tensor A_ = A.unpack(), H_ = H.unpack(shared_from_this());
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(H_.device());
        const Tensor G = cast(grads[0], H_.scalar_type());
        const Tensor gA = at::empty_like(H_), gX = at::empty_like(H_);
        const mpa_pscan_shape s = pscan_shape(A_, G, H_, gA, gX, reverse, chunks);
        const size_t nbytes = mpa_pscan_workspace_bytes(&s);
        const Tensor ws = scratch(nbytes, H_);
        check(mpa_pscan_bwd(&s, ptr(A_), ptr(H_), ptr(G), ptr(gA), ptr(gX), ptr(ws), nbytes, stream_of(H_)), "mpa_pscan_bwd");
        out[0] = grad_as(gA, ta);
        out[1] = grad_as(gX, tx);
        return out;
    }
};

Tensor pscan(const Tensor& A_in, const Tensor& X_in, bool reverse, const PackedPlan& packed) {
    require_gpu({&A_in, &X_in});
    require_plain({&A_in, &X_in});
    TORCH_CHECK(A_in.sizes() == X_in.sizes() && X_in.dim() == 4, "pscan expects two (B, L, D, N) tensors, got ", A_in.sizes(), " and ",
                X_in.sizes());
    const auto dt = at::promote_types(A_in.scalar_type(), X_in.scalar_type());
    io_dtype(dt);
    const Plan plan = unpack(packed);
    std::shared_ptr<PScanBackward> node;
    if (tracked({&A_in, &X_in})) node = make_node<PScanBackward>({&A_in, &X_in});
    Tensor H, A;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(X_in.device());
        A = cast(A_in, dt);
        const Tensor X = cast(X_in, dt);
        H = empty(X.sizes(), dt, X);
        const mpa_pscan_shape s = pscan_shape(A, X, H, Tensor(), Tensor(), reverse, plan.pscan_chunks);
        const size_t nbytes = mpa_pscan_workspace_bytes(&s);
        const Tensor ws = scratch(nbytes, X);
        check(mpa_pscan_fwd(&s, ptr(A), ptr(X), ptr(H), ptr(ws), nbytes, stream_of(X)), "mpa_pscan_fwd");
    }
    if (node) {
        node->reverse = reverse;
        node->chunks = plan.pscan_chunks;
        node->ta = A_in.scalar_type();
        node->tx = X_in.scalar_type();
        node->A = keep(A);
        torch::autograd::set_history(H, node);
        node->H = SavedVariable(H, true);
    }
    return H;
}

// ---- causal convolution -------------------------------------------------------------------------

mpa_conv_shape conv_shape(const Tensor& x, const Tensor& y, const Tensor& g, int64_t K, bool silu) {
    mpa_conv_shape s{};
    s.batch = x.size(0); s.seqlen = x.size(1); s.dim = x.size(2);
    s.kernel = (int)K;
    s.io_dtype = io_dtype(x.scalar_type());
    s.flags = silu ? MPA_CONV_SILU : 0;
    s.x_sb = x.stride(0); s.x_sl = x.stride(1); s.x_sd = x.stride(2);
    s.y_sb = y.stride(0); s.y_sl = y.stride(1); s.y_sd = y.stride(2);
    s.g_sb = g.stride(0); s.g_sl = g.stride(1); s.g_sd = g.stride(2);
    return s;
}

struct ConvBackward : public Node {
    SavedVariable x, w, b, win;
    bool silu = true;
    std::vector<int64_t> wshape;
    at::ScalarType tw, tb;
    std::string name() const override { return "CausalConv1dBackward"; }
    void release_variables() override {
        for (SavedVariable* v : {&x, &w, &b, &win}) v->reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        variable_list out(3);
        if (!grads[0].defined()) return out;
        const Tensor x_ = x.unpack(), w_ = dense(w.unpack()), b_ = dense(b.unpack()), win_ = dense(win.unpack());
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x_.device());
        const int64_t ED = x_.size(2), K = w_.size(1);
        const Tensor dy = cast(grads[0], x_.scalar_type());
        const Tensor dx = empty(x_.sizes(), x_.scalar_type(), x_), dw = empty({ED, K}, at::kFloat, x_);
        const Tensor db = b_.defined() ? empty({ED}, at::kFloat, x_) : Tensor();
        const mpa_conv_shape s = conv_shape(x_, dy, dx, K, silu);
        const size_t nbytes = mpa_conv1d_bwd_workspace_bytes(&s);
        const Tensor ws = scratch(nbytes, x_);
        check(mpa_conv1d_bwd(&s, ptr(x_), fptr(w_), fptr(b_), ptr(win_), ptr(dy), ptr(dx), fptr(dw), fptr(db), ptr(ws), nbytes,
                             stream_of(x_)),
              "mpa_conv1d_bwd");
        out[0] = dx;
        out[1] = grad_as(dw.view(wshape), tw);
        out[2] = grad_as(db, tb);
        return out;
    }
};

std::tuple<Tensor, Opt> conv(const Tensor& x, const Tensor& w_in, const Opt& b_in, const Opt& win_in, bool silu, bool return_window) {
    const Tensor bc = val(b_in), wc = val(win_in);
    require_gpu({&x, &w_in, &bc, &wc});
    require_plain({&x, &w_in, &bc, &wc});
    TORCH_CHECK(x.dim() == 3, "x must be (B, L, ED)");
    const int64_t Bs = x.size(0), L = x.size(1), ED = x.size(2), K = w_in.size(-1);
    TORCH_CHECK(w_in.numel() == ED * K, "weight must be (ED, 1, K) or (ED, K), got ", w_in.sizes());
    TORCH_CHECK(!wc.defined() || wc.sizes() == at::IntArrayRef({Bs, ED, K - 1}), "window must be (B, ED, K-1)");
    TORCH_CHECK(!bc.defined() || bc.numel() == ED, "bias must have ", ED, " elements, got ", bc.sizes());
    const auto dt = x.scalar_type();
    io_dtype(dt);
    std::shared_ptr<ConvBackward> node;
    if (tracked({&x, &w_in, &bc})) node = make_node<ConvBackward>({&x, &w_in, &bc});
    Tensor y, wout, w, b, win;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x.device());
        w = f32c(w_in).view({ED, K});
        b = f32c(bc);
        win = wc.defined() ? cast(wc, dt).contiguous() : wc;
        y = empty({Bs, L, ED}, dt, x);
        if (return_window) wout = empty({Bs, ED, K - 1}, dt, x);
        const mpa_conv_shape s = conv_shape(x, y, y, K, silu);
        check(mpa_conv1d_fwd(&s, ptr(x), fptr(w), fptr(b), ptr(win), ptr(y), ptr(wout), stream_of(x)), "mpa_conv1d_fwd");
    }
    if (node) {
        node->silu = silu;
        node->wshape = w_in.sizes().vec();
        node->tw = w_in.scalar_type();
        node->tb = bc.defined() ? bc.scalar_type() : at::kFloat;
        node->x = keep(x); node->w = keep(w); node->b = keep(b); node->win = keep(win);
        torch::autograd::set_history(y, node);
    }
    return {y, return_window ? Opt(wout) : Opt()};
}

// One decode step of the convolution; `window` is updated in place.
Tensor conv_update(const Tensor& x, const Tensor& window, const Tensor& w_in, const Opt& b_in, bool silu) {
    const Tensor bc = val(b_in);
    require_gpu({&x, &window, &w_in, &bc});
    TORCH_CHECK(x.dim() == 2, "x must be (B, ED)");
    const int64_t Bs = x.size(0), ED = x.size(1), K = w_in.size(-1);
    TORCH_CHECK(w_in.numel() == ED * K && (!bc.defined() || bc.numel() == ED), "weight must be (ED, 1, K) or (ED, K) and bias (ED), got ",
                w_in.sizes(), bc.defined() ? bc.sizes() : at::IntArrayRef());
    TORCH_CHECK(window.sizes() == at::IntArrayRef({Bs, ED, K - 1}) && window.scalar_type() == x.scalar_type() && window.is_contiguous(),
                "window must be a contiguous (B, ED, K-1) tensor of x's dtype");
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x.device());
    const Tensor x3 = x.unsqueeze(1), w = f32c(w_in).view({ED, K}), b = f32c(bc), y = empty({Bs, 1, ED}, x.scalar_type(), x);
    const mpa_conv_shape s = conv_shape(x3, y, y, K, silu);
    check(mpa_conv1d_fwd(&s, ptr(x3), fptr(w), fptr(b), ptr(window), ptr(y), ptr(window), stream_of(x)), "mpa_conv1d_fwd");
    return y.select(1, 0);
}

// ---- RMSNorm ------------------------------------------------------------------------------------

// (x [, residual]) -> rmsnorm(x [+ residual]) [, x + residual]; inputs of the node: x, residual, weight
int weight_flag(const Tensor& w) { return w.defined() && w.scalar_type() == at::kBFloat16 ? MPA_NORM_WEIGHT_BF16 : 0; }

struct NormBackward : public Node {
    SavedVariable x, w;
    double eps = 0;
    bool with_sum = false;
    at::ScalarType tw;
    std::string name() const override { return "RMSNormBackward"; }
    void release_variables() override { x.reset_data(); w.reset_data(); }
    variable_list apply(variable_list&& grads) override {
        variable_list out(3);
        const bool has_dy = grads[0].defined(), has_ds = with_sum && grads[1].defined();
        if (!has_dy && !has_ds) return out;
        const Tensor x_ = dense(with_sum ? x.unpack(shared_from_this()) : x.unpack()), w_ = dense(w.unpack());
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x_.device());
        const auto dt = x_.scalar_type();
        const int64_t d = x_.size(-1), rows = x_.numel() / d;
        const Tensor dy = has_dy ? cast(grads[0], dt).contiguous() : at::zeros_like(x_);
        const Tensor ds = has_ds ? cast(grads[1], dt).contiguous() : Tensor();
        const Tensor dx = at::empty_like(x_);
        Tensor dw, ws;
        size_t nbytes = 0;
        if (w_.defined()) {
            dw = empty({d}, w_.scalar_type(), x_);
            nbytes = mpa_rmsnorm_bwd_workspace_bytes(rows, d);
            ws = scratch(nbytes, x_);
        }
        check(mpa_rmsnorm_bwd(ptr(x_), ptr(w_), ptr(dy), ptr(ds), ptr(dx), ptr(dw), rows, d, (float)eps, io_dtype(dt) | weight_flag(w_),
                              ptr(ws), nbytes, stream_of(x_)),
              "mpa_rmsnorm_bwd");
        out[0] = dx;
        if (with_sum) out[1] = dx;
        out[2] = grad_as(dw, tw);
        return out;
    }
};

std::tuple<Tensor, Opt> rmsnorm(const Tensor& x_in, const Opt& res_in, const Opt& w_in, double eps) {
    const Tensor rc = val(res_in), wc = val(w_in);
    require_gpu({&x_in, &rc, &wc});
    require_plain({&x_in, &rc, &wc});
    TORCH_CHECK(!rc.defined() || (rc.sizes() == x_in.sizes() && rc.scalar_type() == x_in.scalar_type()),
                "residual must have the shape and dtype of x");
    const int io = io_dtype(x_in.scalar_type());
    const int64_t d = x_in.size(-1);
    TORCH_CHECK(d > 0 && (!wc.defined() || wc.numel() == d), "the last dimension of x must not be empty, and weight as long, got x", x_in.sizes(),
                " weight", wc.defined() ? wc.sizes() : at::IntArrayRef());
    const int64_t rows = x_in.numel() / d;
    std::shared_ptr<NormBackward> node;
    if (tracked({&x_in, &rc, &wc})) node = make_node<NormBackward>({&x_in, &rc, &wc});
    Tensor y, sum, x, w;
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x_in.device());
        x = x_in.contiguous();
        w = wc.defined() && wc.scalar_type() == at::kBFloat16 ? wc.contiguous() : f32c(wc);
        const Tensor r = rc.defined() ? rc.contiguous() : rc;
        y = at::empty_like(x);
        if (r.defined()) sum = at::empty_like(x);
        check(mpa_rmsnorm_fwd(ptr(x), ptr(r), ptr(w), ptr(y), ptr(sum), nullptr, rows, d, (float)eps, io | weight_flag(w), stream_of(x)),
              "mpa_rmsnorm_fwd");
    }
    if (node) {
        node->eps = eps;
        node->with_sum = sum.defined();
        node->tw = wc.defined() ? wc.scalar_type() : at::kFloat;
        node->w = keep(w);
        torch::autograd::set_history(y, node);
        if (sum.defined()) {
            torch::autograd::set_history(sum, node);
            node->x = SavedVariable(sum, true);
        } else {
            node->x = keep(x);
        }
    }
    return {y, sum.defined() ? Opt(sum) : Opt()};
}

// ---- decode step of the scan --------------------------------------------------------------------

std::tuple<Tensor, Tensor> step(const Tensor& x_in, const Tensor& delta_in, const Tensor& A_in, const Tensor& B_in, const Tensor& C_in,
                                const Tensor& D_in, const Opt& h_in, const Opt& z_in, const Opt& bias_in, bool softplus, bool inplace) {
    const Tensor hc = val(h_in), zc = val(z_in), bc = val(bias_in);
    require_gpu({&x_in, &delta_in, &A_in, &B_in, &C_in, &D_in, &hc, &zc, &bc});
    const auto dt = x_in.scalar_type();
    const int io = io_dtype(dt);
    TORCH_CHECK(x_in.dim() == 2 && A_in.dim() == 2, "x must be (B, ED) and A (ED, N)");
    const int64_t Bs = x_in.size(0), ED = x_in.size(1), N = A_in.size(1);
    auto rows_of = [&](const Tensor& t) { return t.dim() >= 2 && t.size(0) == Bs && t.numel() == Bs * N; };
    TORCH_CHECK(delta_in.numel() == Bs * ED && A_in.size(0) == ED && rows_of(B_in) && rows_of(C_in) && D_in.numel() == ED &&
                    (!zc.defined() || (zc.size(0) == Bs && zc.numel() == Bs * ED)) && (!bc.defined() || bc.numel() == ED) &&
                    (!hc.defined() || hc.numel() == Bs * ED * N),
                "shape mismatch: x", x_in.sizes(), " delta", delta_in.sizes(), " A", A_in.sizes(), " B", B_in.sizes(), " C", C_in.sizes(),
                " D", D_in.sizes());
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x_in.device());
    const Tensor x = x_in.contiguous(), delta = cast(delta_in, dt).contiguous();
    auto rows = [&](const Tensor& t, int64_t n) { return unit_rows(cast(t.dim() == 2 ? t : t.reshape({Bs, n}), dt)); };
    const Tensor z = zc.defined() ? rows(zc, ED) : zc;
    Tensor B = rows(B_in, N), C = rows(C_in, N);
    if (B.stride(0) != C.stride(0)) { B = B.contiguous(); C = C.contiguous(); }
    const Tensor A = f32c(A_in), D = f32c(D_in), bias = f32c(bc);
    Tensor h = hc;
    if (h.defined() && (h.scalar_type() != at::kFloat || !h.is_contiguous() || h.sizes() != at::IntArrayRef({Bs, ED, N}))) {
        TORCH_CHECK(!inplace, "in-place step needs a contiguous float32 (B, ED, N) state");
        h = f32c(h);
    }
    TORCH_CHECK(!inplace || h.defined(), "in-place step needs an existing state tensor");
    const Tensor h_out = inplace ? h : empty({Bs, ED, N}, at::kFloat, x), y = empty({Bs, ED}, dt, x);
    check(mpa_ssm_step(ptr(x), ptr(delta), fptr(A), ptr(B), ptr(C), fptr(D), ptr(z), fptr(bias), fptr(h), fptr(h_out), ptr(y), Bs, ED, N,
                       B.stride(0), z.defined() ? z.stride(0) : 0, io, softplus ? 1 : 0, stream_of(x)),
          "mpa_ssm_step");
    return {y, h_out};
}

}  // namespace
}  // namespace mpa_host

using namespace mpa_host;

PYBIND11_MODULE(_mpa_host, m) {
    typedef py::call_guard<py::gil_scoped_release> nogil;
    m.def("scan", &scan_fwd, nogil());
    m.def("pscan", &pscan, nogil());
    m.def("conv", &conv, nogil());
    m.def("conv_update", &conv_update, nogil());
    m.def("rmsnorm", &rmsnorm, nogil());
    m.def("step", &step, nogil());
    bind_model(m);
    bind_train(m);
}
