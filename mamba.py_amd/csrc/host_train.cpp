// One mixer (MambaBlock) with gradients as one graph node.
//
// Recorded operation by operation, the backward of a block spends a third of its time around the
// kernels that do the work: concatenating the gradients of the two halves of in_proj's output, adding those
// of x_proj's to the scan's, filling and copying slices for the padded projections, converting the
// gradients of small parameters, and weight gradients as library GEMMs whose grids are too small.  Here the
// kernels write where the next one reads: the scan leaves dz and the convolution dx as the two halves of
// one matrix, dB and dC go into the columns of x_proj's output gradient, x_proj's input gradient is
// added to the scan's by the GEMM itself, and the four weight gradients are one launch (mpa_wgrad).
#include "host_layer.h"

namespace mpa_host {
namespace {

enum { kIX, kIInW, kIInB, kIConvW, kIConvB, kIXW, kIDtW, kIDtB, kIALog, kID, kIOutW, kIOutB, kInputs };

// What the node keeps: inputs, activations and derived weights, all of them as saved variables, so that hooks on saved
// tensors (checkpointing, offloading) have them; and the parameters the derived ones are made from, whose version
// counters are checked when they are unpacked.
enum { kSWin, kSH0, kSXz, kSXs, kSDbc, kSDelta, kSY, kSYPre, kSCkpt, kSA, kSD, kSDtB, kSConvW, kSConvB, kSXp, kSDtp, kSaved };

struct MixerBackward : public Node {
    SavedVariable inputs[kInputs], saved[kSaved];
    int64_t Bs = 0, L = 0, d = 0, ED = 0, N = 0, R = 0, Rp = 0, K = 0, P = 0;
    Plan plan;
    std::string name() const override { return "MambaBlockBackward"; }
    void release_variables() override {
        for (SavedVariable& v : inputs) v.reset_data();
        for (SavedVariable& v : saved) v.reset_data();
    }
    variable_list apply(variable_list&& grads) override;
};

mpa_sscan_shape mixer_scan_shape(const MixerBackward& m, int io, bool backward) {
    mpa_sscan_shape s{};
    const int64_t L = m.L, ED = m.ED, P = m.P;
    s.batch = m.Bs; s.seqlen = L; s.dim = ED; s.dstate = m.N;
    s.io_dtype = io;
    s.flags = MPA_SSCAN_DELTA_SOFTPLUS;
    s.u_sb = s.d_sb = s.y_sb = L * ED; s.u_sl = s.d_sl = s.y_sl = ED;
    s.u_sd = s.d_sd = s.y_sd = s.z_sd = s.g_sd = 1;
    s.z_sb = L * 2 * ED; s.z_sl = 2 * ED;
    // the gradients of x and delta are the halves of one (T, 2 ED) matrix, that of z the second half of another
    s.g_sb = L * 2 * ED; s.g_sl = 2 * ED;
    s.bc_sb = s.dbc_sb = L * P; s.bc_sl = s.dbc_sl = P;
    s.plan_states_per_lane = backward ? m.plan.bwd_ns : m.plan.fwd_ns;
    s.plan_segments = backward ? m.plan.bwd_segments : m.plan.fwd_segments;
    s.plan_flags = m.plan.flags;
    return s;
}

mpa_conv_shape mixer_conv_shape(const MixerBackward& m, int io, bool backward) {
    mpa_conv_shape s{};
    const int64_t L = m.L, ED = m.ED, out = backward ? 2 * ED : ED;
    s.batch = m.Bs; s.seqlen = L; s.dim = ED;
    s.kernel = (int)m.K;
    s.io_dtype = io;
    s.flags = MPA_CONV_SILU;
    s.x_sb = s.g_sb = L * 2 * ED; s.x_sl = s.g_sl = 2 * ED;
    s.y_sb = L * out; s.y_sl = out;
    s.x_sd = s.y_sd = s.g_sd = 1;
    return s;
}

// The forward pass and its node; (y, h_last, window), the latter two if asked for.  Runs without the interpreter's lock.
std::tuple<Tensor, Tensor, Tensor> mixer_forward(Weights& l, const std::array<const Tensor*, kInputs>& in, const Tensor& hc, const Tensor& wc,
                                                 bool return_cache, const Plan& plan) {
    const Tensor& x_in = *in[kIX];
    auto node = make_node<MixerBackward>({in[0], in[1], in[2], in[3], in[4], in[5], in[6], in[7], in[8], in[9], in[10], in[11]});
    Tensor x, out, h_last, window, t[kSaved];
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x_in.device());
        MixerBackward& m = *node;
        x = dense16(x_in);
        const auto dt = x.scalar_type();
        const int io = io_dtype(dt);
        const size_t es = x.element_size();
        m.Bs = x.size(0); m.L = x.size(1); m.d = l.d; m.ED = l.ED; m.N = l.N; m.R = l.R; m.Rp = l.Rp; m.K = l.K;
        m.P = l.padded_rows();
        m.plan = plan;
        l.form_for_training();
        const int64_t T = m.Bs * m.L, ED = m.ED, N = m.N, P = m.P;
        const Tensor x2 = x.view({T, m.d});
        void* stream = stream_of(x);
        const bool own = use_linear(dt, true, T, m.d, ED, P, {&x, &l.p[kInW], &l.p[kOutW], &l.xp, &l.dtp, &l.p[kInB], &l.p[kOutB]});
        auto product = [&](const Tensor& in, int64_t K, const Tensor& weight, const Tensor& bias) {
            const int64_t M = weight.size(0);
            const Tensor y = empty({T, M}, dt, x);
            mpa_linear q = linear_of(io, T, ptr(in), in.size(1), K, ptr(weight), M, ptr(y), M);
            q.bias = ptr(bias);
            run_linear(q, stream);
            return y;
        };
        // in_proj and out_proj
        auto wide = [&](const Tensor& in, const Tensor& weight, const Tensor& bias) {
            if (own) return product(in, weight.size(1), weight, bias);
            const Tensor y = empty({T, weight.size(0)}, dt, x);
            if (split_product(in, weight, bias, y, stream)) return y;
            Tensor out = y;
            if (bias.defined()) at::addmm_out(out, bias, in, weight.t());
            else mm_into(y, in, weight, false, stream);
            return y;
        };
        const Tensor xz = wide(x2, l.p[kInW], l.p[kInB]);
        const Tensor xs = empty({T, ED}, dt, x);
        if (return_cache) {
            window = empty({m.Bs, ED, m.K - 1}, dt, x);
            h_last = empty({m.Bs, ED, N}, at::kFloat, x);
        }
        const mpa_conv_shape cv = mixer_conv_shape(m, io, false);
        Tensor dbc = empty({T, P}, dt, x);
        if (!conv_proj(cv, l, ptr(xz), ptr(wc), ptr(xs), ptr(window), ptr(dbc), P, stream)) {
            check(mpa_conv1d_fwd(&cv, ptr(xz), fptr(l.conv_w), fptr(l.conv_b), ptr(wc), ptr(xs), ptr(window), stream), "mpa_conv1d_fwd");
            dbc = own ? product(xs, ED, l.xp, Tensor()) : at::mm_out(dbc, xs, l.xp.t());
        }
        const Tensor delta = own ? product(dbc, m.Rp, l.dtp, Tensor()) : at::mm(dbc.narrow(1, 0, m.Rp), l.dtp.t());
        const Tensor y = empty({T, ED}, dt, x), y_pre = empty({T, ED}, dt, x);
        const mpa_sscan_shape sc = mixer_scan_shape(m, io, false);
        const Tensor ckpt = empty({mpa_sscan_ckpt_elems(&sc)}, at::kFloat, x);
        const size_t nbytes = mpa_sscan_fwd_workspace_bytes(&sc, 1);
        const Tensor ws = scratch(nbytes, x);
        const char* bc = static_cast<const char*>(ptr(dbc)) + m.Rp * es;
        check(mpa_sscan_fwd(&sc, ptr(xs), ptr(delta), fptr(l.A), bc, bc + N * es, fptr(l.D), static_cast<const char*>(ptr(xz)) + ED * es,
                            fptr(l.dt_b), fptr(hc), ptr(y), ptr(y_pre), fptr(ckpt), fptr(h_last), ptr(ws), nbytes, stream),
              "mpa_sscan_fwd");
        out = wide(y, l.p[kOutW], l.p[kOutB]).view({m.Bs, m.L, m.d});
        const std::array<const Tensor*, kSaved> made = {&wc, &hc, &xz, &xs, &dbc, &delta, &y, &y_pre, &ckpt, &l.A, &l.D, &l.dt_b, &l.conv_w,
                                                        &l.conv_b, &l.xp, &l.dtp};
        for (int i = 0; i < kSaved; ++i) t[i] = *made[i];
    }
    // (outside of the guard: hooks on saved tensors are called here)
    node->inputs[kIX] = keep(x);
    for (int i = 1; i < kInputs; ++i) node->inputs[i] = keep(*in[i]);
    for (int i = 0; i < kSaved; ++i) node->saved[i] = keep(t[i]);
    torch::autograd::set_history(out, node);
    return {out, h_last, window};
}

// (y, h_last or None, window or None), or None: not a block that can run here
py::object block_train(const py::object& block, const Tensor& x_in, const Opt& h_in, const Opt& win_in, bool return_cache,
                       const PackedPlan& packed) {
    if (!at::GradMode::is_enabled() || !native_call(x_in) || x_in.dim() != 3 || x_in.numel() == 0) return py::none();
    Weights l;
    const Tensor hc = val(h_in), wc = val(win_in);
    {
        at::AutoDispatchBelowADInplaceOrView below;
        const c10::DeviceGuard guard(x_in.device());
        MixerHandle* handle = ready_mixer(block.ptr(), x_in, l);
        // (mpa_wgrad takes whole 16-byte parts of a row)
        if (!handle || !handle->forward_ok || handle->N % 4 || handle->ED % (16 / (int64_t)x_in.element_size())) return py::none();
        if (unpack(packed).flags & MPA_PLAN_BWD_GENERAL) return py::none();
        const int64_t Bs = x_in.size(0);
        if (hc.defined() && !fits(hc, {Bs, l.ED, l.N}, at::kFloat, l.device)) return py::none();
        if (wc.defined() && !fits(wc, {Bs, l.ED, l.K - 1}, l.dt, l.device)) return py::none();
    }
    const std::array<int, kInputs> from = {-1, kInW, kInB, kConvW, kConvB, kXW, kDtW, kDtB, kALog, kD, kOutW, kOutB};
    std::array<const Tensor*, kInputs> in;
    in[kIX] = &x_in;
    bool any = x_in.requires_grad();
    for (int i = 1; i < kInputs; ++i) {
        in[i] = &l.p[from[i]];
        any |= in[i]->defined() && in[i]->requires_grad();
    }
    if (!any) return py::none();
    Tensor out, h_last, window;
    {
        const py::gil_scoped_release nogil;
        std::tie(out, h_last, window) = mixer_forward(l, in, hc, wc, return_cache, unpack(packed));
    }
    return py::make_tuple(out, return_cache ? py::cast(h_last) : py::object(py::none()),
                          return_cache ? py::cast(window) : py::object(py::none()));
}

variable_list MixerBackward::apply(variable_list&& grads) {
    variable_list g(kInputs);
    if (!grads[0].defined()) return g;
    // (unpacked outside of the guard: a hook may run a whole forward pass)
    Tensor w[kInputs], t[kSaved];
    for (int i = 0; i < kInputs; ++i) w[i] = inputs[i].unpack();
    for (int i = 0; i < kSaved; ++i) t[i] = saved[i].unpack();
    const int64_t T = Bs * L, used = Rp + 2 * N;
    const auto dt = w[kIX].scalar_type();
    const auto f32 = at::kFloat;
    // (a hook may also give back another tensor than it was given: the kernels rely on these)
    const auto given = [&](Tensor& v, at::IntArrayRef shape, at::ScalarType type) {
        if (!v.defined()) return;
        TORCH_CHECK(v.sizes() == shape && v.scalar_type() == type && v.device() == w[kIX].device(), "a saved tensor of a MambaBlock came back as ",
                    v.scalar_type(), v.sizes(), " on ", v.device(), ", was ", type, shape);
        v = dense16(v);
    };
    given(w[kIX], {Bs, L, d}, dt); given(w[kIInW], {2 * ED, d}, dt); given(w[kIOutW], {d, ED}, dt);
    given(t[kSWin], {Bs, ED, K - 1}, dt); given(t[kSH0], {Bs, ED, N}, f32);
    given(t[kSXz], {T, 2 * ED}, dt); given(t[kSDbc], {T, P}, dt);
    for (int i : {kSXs, kSDelta, kSY, kSYPre}) given(t[i], {T, ED}, dt);
    given(t[kSCkpt], {Bs * ((L + MPA_CKPT_STEPS - 1) / MPA_CKPT_STEPS) * N * ED}, f32);
    given(t[kSA], {ED, N}, f32);
    for (int i : {kSD, kSDtB, kSConvB}) given(t[i], {ED}, f32);
    given(t[kSConvW], {ED, 1, K}, f32);
    given(t[kSXp], {P, ED}, dt); given(t[kSDtp], {ED, Rp}, dt);
    const Tensor &x_ = w[kIX], &win_ = t[kSWin], &h0_ = t[kSH0], &xz = t[kSXz], &xs = t[kSXs], &dbc = t[kSDbc], &delta = t[kSDelta], &y = t[kSY],
                 &y_pre = t[kSYPre], &ckpt = t[kSCkpt], &A = t[kSA], &D = t[kSD], &dt_b = t[kSDtB], &conv_w = t[kSConvW], &conv_b = t[kSConvB],
                 &xp = t[kSXp], &dtp = t[kSDtp];
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x_.device());
    const int io = io_dtype(dt);
    const size_t es = x_.element_size();
    void* stream = stream_of(x_);
    auto at_col = [&](const Tensor& t, int64_t col) { return static_cast<char*>(ptr(t)) + col * es; };
    const Tensor x2 = x_.view({T, d}), dout = dense16(cast(grads[0], dt)).view({T, d});

    const bool own = use_linear(dt, true, T, d, ED, P, {&dout, &w[kIOutW], &w[kIInW], &xp, &dtp});
    // out (T x M) = in (T x K) . weight (K x M), or added to out
    auto product = [&](const void* in, int64_t in_pitch, int64_t K, const Tensor& weight, void* out, int64_t out_pitch, bool add) {
        mpa_linear q = linear_of(io, T, in, in_pitch, K, ptr(weight), weight.size(1), out, out_pitch);
        q.weight_kxm = 1;
        if (add) { q.residual = out; q.accumulate = 1; }
        run_linear(q, stream);
    };
    Tensor dy;
    if (own) {
        dy = empty({T, ED}, dt, x_);
        product(ptr(dout), d, d, w[kIOutW], ptr(dy), ED, false);
    } else if (use_split(dt, T, ED, d, {&dout, &w[kIOutW]})) {
        dy = empty({T, ED}, dt, x_);
        Split s(x_, stream);
        const int weight = s.cols(ptr(w[kIOutW]), ED, d, ED), in = s.rows(ptr(dout), T, d, d);
        s.run();
        s.product(weight, in, Tensor(), ptr(dy), ED);
        s.run_products();
    } else {
        dy = empty({T, ED}, dt, x_);
        mm_into(dy, dout, w[kIOutW], true, stream);
    }
    const Tensor dxz = empty({T, 2 * ED}, dt, x_), dxs_ddelta = empty({T, 2 * ED}, dt, x_), ddbc = empty({T, P}, dt, x_);
    const Tensor dA = empty({ED, N}, at::kFloat, x_), dD = empty({ED}, at::kFloat, x_), ddt_b = empty({ED}, at::kFloat, x_);
    {
        const mpa_sscan_shape s = mixer_scan_shape(*this, io, true);
        const size_t nbytes = mpa_sscan_bwd_workspace_bytes(&s);
        const Tensor ws = scratch(nbytes, x_);
        check(mpa_sscan_bwd(&s, ptr(xs), ptr(delta), fptr(A), at_col(dbc, Rp), at_col(dbc, Rp + N), fptr(D), at_col(xz, ED), fptr(dt_b),
                            fptr(h0_), ptr(dy), ptr(y_pre), fptr(ckpt), ptr(dxs_ddelta), at_col(dxs_ddelta, ED), fptr(dA), at_col(ddbc, Rp),
                            at_col(ddbc, Rp + N), fptr(dD), at_col(dxz, ED), fptr(ddt_b), ptr(ws), nbytes, stream),
              "mpa_sscan_bwd");
    }
    // (the columns of ddbc past `used` were never written)
    if (own) {
        product(at_col(dxs_ddelta, ED), 2 * ED, ED, dtp, ptr(ddbc), P, false);
        product(ptr(ddbc), P, used, xp, ptr(dxs_ddelta), 2 * ED, true);
    } else {
        Tensor dxs = dxs_ddelta.narrow(1, 0, ED), ddlow = ddbc.narrow(1, 0, Rp);
        at::mm_out(ddlow, dxs_ddelta.narrow(1, ED, ED), dtp);
        at::addmm_out(dxs, dxs, ddbc.narrow(1, 0, used), xp.narrow(0, 0, used));
    }
    const Tensor dconv_w = empty({ED, K}, at::kFloat, x_), dconv_b = conv_b.defined() ? empty({ED}, at::kFloat, x_) : Tensor();
    {
        const mpa_conv_shape s = mixer_conv_shape(*this, io, true);
        const size_t nbytes = mpa_conv1d_bwd_workspace_bytes(&s);
        const Tensor ws = scratch(nbytes, x_);
        check(mpa_conv1d_bwd(&s, ptr(xz), fptr(conv_w), fptr(conv_b), ptr(win_), ptr(dxs_ddelta), ptr(dxz), fptr(dconv_w), fptr(dconv_b),
                             ptr(ws), nbytes, stream),
              "mpa_conv1d_bwd");
    }
    const bool want_x = task_should_compute_output(kIX), want_in = task_should_compute_output(kIInW), want_out = task_should_compute_output(kIOutW);
    const bool cut = !own && use_split_three(dt, T, d, 2 * ED, {&dout, &x_, &y, &w[kIInW]});
    if (cut && (want_x || want_in || want_out)) {
        // the input's gradient and those of the wide weights, in one launch
        Split s(x_, stream);
        int weight = 0, rows = 0, by_in = 0, in = 0, by_out = 0, gated = 0;
        if (want_x) {
            weight = s.cols(ptr(w[kIInW]), d, 2 * ED, d);
            rows = s.rows(ptr(dxz), T, 2 * ED, 2 * ED);
        }
        if (want_in) {
            by_in = s.cols(ptr(dxz), 2 * ED, T, 2 * ED);
            in = s.cols(ptr(x2), d, T, d);
        }
        if (want_out) {
            by_out = s.cols(ptr(dout), d, T, d);
            gated = s.cols(ptr(y), ED, T, ED);
        }
        s.run();
        if (want_x) {
            g[kIX] = empty({Bs, L, d}, dt, x_);
            s.product(weight, rows, Tensor(), ptr(g[kIX]), d);
        }
        if (want_in) {
            g[kIInW] = empty({2 * ED, d}, dt, x_);
            s.product(in, by_in, Tensor(), ptr(g[kIInW]), d);
        }
        if (want_out) {
            g[kIOutW] = empty({d, ED}, dt, x_);
            s.product(gated, by_out, Tensor(), ptr(g[kIOutW]), ED);
        }
        s.run_products();
    } else if (want_x) {
        if (own) {
            g[kIX] = empty({Bs, L, d}, dt, x_);
            product(ptr(dxz), 2 * ED, 2 * ED, w[kIInW], ptr(g[kIX]), d, false);
        } else {
            g[kIX] = empty({Bs, L, d}, dt, x_);
            mm_into(g[kIX].view({T, d}), dxz, w[kIInW], true, stream);
        }
    }

    // weight gradients.  float32: the wide ones are compute bound and run on cut operands or stay with the GEMM library
    std::vector<mpa_wgrad_job> jobs;
    auto want = [&](int i, const void* p, int64_t ldp, int64_t rows, const void* q, int64_t ldq, int64_t cols, int64_t keep_cols,
                    int64_t gap_at, int64_t gap) {
        if (!task_should_compute_output(i)) return;
        g[i] = empty(w[i].sizes(), dt, x_);
        jobs.push_back(mpa_wgrad_job{p, q, ldp, ldq, rows, cols, keep_cols, gap_at, gap, ptr(g[i])});
    };
    if (io == MPA_BF16) {
        want(kIInW, ptr(dxz), 2 * ED, 2 * ED, ptr(x2), d, d, d, 0, 0);
        want(kIOutW, ptr(dout), d, d, ptr(y), ED, ED, ED, 0, 0);
    } else if (!cut) {
        if (want_in) g[kIInW] = at::mm(dxz.t(), x2);
        if (want_out) g[kIOutW] = at::mm(dout.t(), y);
    }
    want(kIXW, ptr(ddbc), P, used, ptr(xs), ED, ED, ED, R, Rp - R);
    want(kIDtW, at_col(dxs_ddelta, ED), 2 * ED, ED, ptr(dbc), P, Rp, R, 0, 0);
    if (!jobs.empty()) {
        const size_t nbytes = mpa_wgrad_workspace_bytes(jobs.data(), (int)jobs.size(), T, io);
        const Tensor ws = scratch(nbytes, x_);
        check(mpa_wgrad(jobs.data(), (int)jobs.size(), T, io, ptr(ws), nbytes, stream), "mpa_wgrad");
    }
    if (w[kIInB].defined() && task_should_compute_output(kIInB)) g[kIInB] = dxz.sum(0);
    if (w[kIOutB].defined() && task_should_compute_output(kIOutB)) g[kIOutB] = dout.sum(0);

    // small parameters: their own types; dA_log = dA * A, because A = -exp(A_log)
    std::vector<mpa_cast_job> casts;
    auto small = [&](int i, const Tensor& f32, int op, const float* factor) {
        if (!w[i].defined() || !f32.defined() || !task_should_compute_output(i)) return;
        if (op == MPA_CAST_COPY && w[i].scalar_type() == at::kFloat) { g[i] = f32.view(w[i].sizes()); return; }
        g[i] = empty(w[i].sizes(), w[i].scalar_type(), x_);
        casts.push_back(cast_job(f32, g[i], 1, f32.numel(), 0, 0, op, factor));
        casts.back().src_pitch = casts.back().dst_pitch = f32.numel();
    };
    small(kIConvW, dconv_w, MPA_CAST_COPY, nullptr);
    small(kIConvB, dconv_b, MPA_CAST_COPY, nullptr);
    small(kIDtB, ddt_b, MPA_CAST_COPY, nullptr);
    small(kIALog, dA, MPA_CAST_TIMES, fptr(A));
    small(kID, dD, MPA_CAST_COPY, nullptr);
    if (!casts.empty()) check(mpa_cast(casts.data(), (int)casts.size(), stream), "mpa_cast");
    return g;
}

}  // namespace

void bind_train(py::module_& m) { m.def("block_train", &block_train); }

}  // namespace mpa_host
