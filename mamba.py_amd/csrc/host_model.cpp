// The layer stack without gradients, from C++: decode steps and forward passes of a list of
// residual blocks in one call from Python.
#include "host_layer.h"

#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/jit/frontend/tracer.h>

namespace mpa_host {
namespace {

// (h or None, window) pairs; false if one of them is not what the kernels take
struct Cache {
    Tensor h, window;
};
bool read_cache(PyObject* pair, Cache& c) {
    if (!(PyTuple_Check(pair) || PyList_Check(pair)) || PySequence_Fast_GET_SIZE(pair) != 2) return false;
    PyObject* h = PySequence_Fast_GET_ITEM(pair, 0);
    PyObject* w = PySequence_Fast_GET_ITEM(pair, 1);
    if (h != Py_None) {
        if (!THPVariable_Check(h)) return false;
        c.h = THPVariable_Unpack(h);
    }
    if (!THPVariable_Check(w)) return false;
    c.window = THPVariable_Unpack(w);
    return true;
}
bool cache_fits(const Cache& c, const LayerSizes& l, int64_t batch, bool need_h) {
    if (!c.h.defined() ? need_h : !fits(c.h, {batch, l.ED, l.N}, at::kFloat, l.device)) return false;
    return c.window.scalar_type() == l.dt && c.window.device() == l.device && c.window.is_contiguous() &&
           c.window.sizes() == at::IntArrayRef({batch, l.ED, l.K - 1});
}

void form_layers(std::vector<Layer>& layers, bool sequence) {
    Forming f(layers[0].m->device);
    for (Layer& l : layers) l.m->form(f, sequence, l.w, l.n, &l.norm_w);
    f.done();
}

py::object pair(const Tensor& h, const Tensor& w) { return py::make_tuple(h, w); }

// ---- decode -------------------------------------------------------------------------------------

// The launches of a step, without the interpreter's lock; `cs` becomes the caches after it.
Tensor run_steps(const std::vector<Layer>& layers, const Tensor& x, std::vector<Cache>& cs, bool inplace) {
    const size_t n = layers.size();
    const int64_t batch = x.size(0);
    std::vector<mpa_decode_layer> desc(n);
    for (size_t i = 0; i < n; ++i) {
        desc[i] = layers[i].w.desc(batch);
        desc[i].norm = 1;
        desc[i].eps = (float)layers[i].eps;
        desc[i].norm_weight = fptr(layers[i].norm_w);
    }
    const auto dt = x.scalar_type();
    const int64_t d = x.size(1);
    // two rows per sequence and two scaled rows, used in turn (a kernel never writes what it reads), with
    // the partial sums of squares of the latter
    const int64_t tiles = (d + 15) / 16;
    const size_t scaled_bytes = mpa_decode_scaled_bytes(&desc[0]);
    const Tensor spare = empty({batch, d}, dt, x), y = empty({batch, d}, dt, x), scaled_rows = scratch(2 * scaled_bytes, x),
                 ssq = empty({2, tiles * batch}, at::kFloat, x);
    size_t ws_bytes = 0;
    for (const mpa_decode_layer& s : desc) ws_bytes = std::max(ws_bytes, mpa_decode_layer_workspace_bytes(&s));
    const Tensor ws = scratch(ws_bytes, x);
    void* stream = stream_of(x);
    // the last layer writes y, the others y and a spare row in turn
    const void* in = ptr(x);
    const void* scaled = nullptr;
    const float* sums = nullptr;
    for (size_t i = 0; i < n; ++i) {
        const Weights& l = layers[i].w;
        Cache out = cs[i];
        if (!inplace) {
            out.h = empty({batch, l.ED, l.N}, at::kFloat, x);
            out.window = empty({batch, l.ED, l.K - 1}, dt, x);
        }
        void* to = (n - 1 - i) % 2 == 0 ? ptr(y) : ptr(spare);
        // (a norm without a weight has nothing to scale by: the next layer forms its own sums)
        const float* next_w = i + 1 < n ? desc[i + 1].norm_weight : nullptr;
        void* to_scaled = static_cast<char*>(ptr(scaled_rows)) + (i % 2) * scaled_bytes;
        float* to_sums = fptr(ssq) + (i % 2) * tiles * batch;
        check(mpa_decode_layer_step(&desc[i], in, scaled, sums, to, next_w, to_scaled, to_sums, fptr(cs[i].h), fptr(out.h), ptr(cs[i].window),
                                    ptr(out.window), ptr(ws), ws_bytes, stream),
              "mpa_decode_layer_step");
        in = to;
        scaled = next_w ? to_scaled : nullptr;
        sums = next_w ? to_sums : nullptr;
        cs[i] = out;
    }
    return y;
}

// One token through the residual blocks `layers`; the caches are updated in place or replaced in the
// list.  None: not a stack that can run here (the caller goes on in Python).
py::object stack_step(const py::list& layers, const Tensor& x_in, const py::list& caches, bool inplace) {
    const size_t n = layers.size();
    if (at::GradMode::is_enabled() || !native_call(x_in) || x_in.dim() != 2 || n == 0 || caches.size() < n ||
        x_in.size(0) > MPA_DECODE_MAX_BATCH || x_in.size(0) == 0)
        return py::none();
    const int64_t batch = x_in.size(0);
    std::vector<Layer> hs(n);
    std::vector<Cache> cs(n);
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x_in.device());
    for (size_t i = 0; i < n; ++i) {
        if (!find_layer(layers[i].ptr(), x_in, hs[i]) || !hs[i].m->decode_ok || hs[i].m->d != hs[0].m->d) return py::none();
        if (!read_cache(caches[i].ptr(), cs[i]) || !cache_fits(cs[i], *hs[i].m, batch, inplace)) return py::none();
    }
    const Tensor x = x_in.contiguous();
    if (reinterpret_cast<uintptr_t>(x.const_data_ptr()) % 16) return py::none();
    form_layers(hs, false);
    Tensor y;
    {
        const py::gil_scoped_release nogil;
        y = run_steps(hs, x, cs, inplace);
    }
    if (!inplace)
        for (size_t i = 0; i < n; ++i) caches[i] = pair(cs[i].h, cs[i].window);
    return py::cast(y);
}

// One token through one MambaBlock (no norm, no residual): (y, h, window) or None.
py::object block_step(const py::object& block, const Tensor& x_in, const Opt& h_in, const Tensor& window, bool inplace) {
    if (at::GradMode::is_enabled() || !native_call(x_in) || x_in.dim() != 2 || x_in.size(0) > MPA_DECODE_MAX_BATCH || x_in.size(0) == 0)
        return py::none();
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x_in.device());
    Weights w;
    MixerHandle* l = ready_mixer(block.ptr(), x_in, w);
    const int64_t batch = x_in.size(0);
    const Cache in{val(h_in), window};
    if (!l || !l->decode_ok || !cache_fits(in, *l, batch, inplace)) return py::none();
    const Tensor x = x_in.contiguous();
    if (reinterpret_cast<uintptr_t>(x.const_data_ptr()) % 16) return py::none();
    {
        Forming f(l->device);
        l->form(f, false, w, nullptr, nullptr);
        f.done();
    }
    py::gil_scoped_release nogil;
    Cache out = in;
    if (!inplace) {
        out.h = empty({batch, w.ED, w.N}, at::kFloat, x);
        out.window = empty({batch, w.ED, w.K - 1}, x.scalar_type(), x);
    }
    const Tensor y = empty({batch, w.d}, x.scalar_type(), x);
    const mpa_decode_layer s = w.desc(batch);
    const size_t nbytes = mpa_decode_layer_workspace_bytes(&s);
    const Tensor ws = scratch(nbytes, x);
    check(mpa_decode_layer_step(&s, ptr(x), nullptr, nullptr, ptr(y), nullptr, nullptr, nullptr, fptr(in.h), fptr(out.h), ptr(in.window),
                                ptr(out.window), ptr(ws), nbytes, stream_of(x)),
          "mpa_decode_layer_step");
    const py::gil_scoped_acquire gil;
    return py::make_tuple(y, out.h, out.window);
}

// ---- forward without gradients ------------------------------------------------------------------

// The launches of a sequence, without the interpreter's lock; with `keep`, `cs` becomes the caches after it.
// The activations of a layer live in buffers that every layer uses again.
Tensor run_sequence(const std::vector<Layer>& hs, const Tensor& x, std::vector<Cache>& cs, bool keep, const Plan& plan) {
    const size_t n = hs.size();
    const int64_t Bs = x.size(0), L = x.size(1), T = Bs * L;
    const Weights& a = hs[0].w;
    const auto dt = x.scalar_type();
    const int io = io_dtype(dt);
    const int64_t d = a.d, ED = a.ED, N = a.N, P = a.xp.size(0);
    const size_t es = x.element_size();
    void* stream = stream_of(x);
    const Tensor normed = empty({T, d}, dt, x), xz = empty({T, 2 * ED}, dt, x), xs = empty({Bs, L, ED}, dt, x),
                 dbc = empty({T, P}, dt, x), y = empty({T, ED}, dt, x), hidden = empty({T, d}, dt, x);
    bool own = use_linear(dt, false, T, d, ED, P, {&x});
    for (const Layer& h : hs)
        own &= h.norm_w.defined() &&
               use_linear(dt, false, T, d, ED, P, {&h.w.p[kInW], &h.w.p[kOutW], &h.w.xp, &h.w.dtp, &h.norm_w, &h.w.p[kInB], &h.w.p[kOutB]});
    // The scan forms delta from dt_proj's rows itself where it has the form for it.  (On dt_proj's padded weight, or one of that rank.)
    bool proj = dt == at::kBFloat16 && a.Rp == MPA_PROJ_RANK && N <= 16 && plan.fwd_ns == 0;
    for (const Layer& h : hs) proj &= aligned(h.w.dtp.const_data_ptr(), 16);
    const Tensor delta = proj ? Tensor() : empty({T, ED}, dt, x);
    // The residual stream between the layers.  The own products keep it in float32: at bfloat16, its roundings were
    // the larger part of a deep stack's error (24 layers of width 768: see tests/test_deep_stack_gpu.py).
    Tensor sum[2];
    const auto sum_dt = own ? at::kFloat : dt;
    if (n > 1) { sum[0] = empty({T, d}, sum_dt, x); sum[1] = empty({T, d}, sum_dt, x); }
    const int64_t parts = (d + 31) / 32;
    const Tensor ssq = own ? empty({parts, T}, at::kFloat, x) : Tensor();
    auto linear = [&](const void* in, int64_t pitch, int64_t K, const Tensor& weight, const Tensor& bias, const Tensor& out) {
        const int64_t M = weight.size(0);
        mpa_linear q = linear_of(io, T, in, pitch, K, ptr(weight), M, ptr(out), M);
        q.bias = ptr(bias);
        return q;
    };
    auto run = [&](const mpa_linear& q, const float* y_weight = nullptr, void* y_scaled = nullptr) {
        check(mpa_linear_run_scaled(&q, y_weight, y_scaled, stream), "mpa_linear_run_scaled");
    };
    const Tensor xs2 = xs.view({T, ED}), dlow = dbc.narrow(1, 0, a.Rp);

    mpa_conv_shape cv{};
    cv.batch = Bs; cv.seqlen = L; cv.dim = ED;
    cv.io_dtype = io;
    cv.flags = MPA_CONV_SILU;
    cv.x_sb = L * 2 * ED; cv.x_sl = 2 * ED; cv.x_sd = 1;
    cv.y_sb = cv.g_sb = L * ED; cv.y_sl = cv.g_sl = ED; cv.y_sd = cv.g_sd = 1;
    mpa_sscan_shape sc{};
    sc.batch = Bs; sc.seqlen = L; sc.dim = ED; sc.dstate = N;
    sc.io_dtype = io;
    sc.flags = MPA_SSCAN_DELTA_SOFTPLUS;
    sc.u_sb = sc.d_sb = sc.y_sb = sc.g_sb = L * ED; sc.u_sl = sc.d_sl = sc.y_sl = sc.g_sl = ED; sc.u_sd = sc.d_sd = sc.y_sd = sc.g_sd = 1;
    sc.z_sb = L * 2 * ED; sc.z_sl = 2 * ED; sc.z_sd = 1;
    sc.bc_sb = sc.dbc_sb = L * P; sc.bc_sl = sc.dbc_sl = P;
    if (proj) { sc.d_sb = L * P; sc.d_sl = P; }
    sc.plan_states_per_lane = plan.fwd_ns; sc.plan_segments = plan.fwd_segments; sc.plan_flags = plan.flags;
    const size_t ws_bytes = mpa_sscan_fwd_workspace_bytes(&sc, 0);
    const Tensor ws = scratch(ws_bytes, x);

    const Tensor result = own ? empty({Bs, L, d}, dt, x) : Tensor();
    const void* in = ptr(x);
    const void* residual = nullptr;
    for (size_t i = 0; i < n; ++i) {
        const Weights& l = hs[i].w;
        const float* norm_w = fptr(hs[i].norm_w);
        const float eps = (float)hs[i].eps;
        const Tensor& s = sum[i % 2];
        if (!own || i == 0)
            check(mpa_rmsnorm_fwd(in, residual, norm_w, ptr(normed), residual ? ptr(s) : nullptr, nullptr, T, d, eps, io, stream),
                  "mpa_rmsnorm_fwd");
        if (!own) residual = residual ? ptr(s) : in;
        Tensor out = xz;
        if (own) {
            mpa_linear q = linear(ptr(normed), d, d, l.p[kInW], l.p[kInB], xz);
            if (i > 0) { q.x_ssq = fptr(ssq); q.ssq_parts = parts; q.eps = eps; }
            run(q);
        } else if (split_product(normed, l.p[kInW], l.p[kInB], xz, stream)) {
        } else if (l.p[kInB].defined()) {
            at::addmm_out(out, l.p[kInB], normed, l.p[kInW].t());
        } else {
            mm_into(xz, normed, l.p[kInW], false, stream);
        }
        Tensor window, h_last;
        if (keep) {
            window = empty({Bs, ED, l.K - 1}, dt, x);
            h_last = empty({Bs, ED, N}, at::kFloat, x);
        }
        cv.kernel = (int)l.K;
        if (!conv_proj(cv, l, ptr(xz), ptr(cs[i].window), ptr(xs), ptr(window), ptr(dbc), P, stream)) {
            check(mpa_conv1d_fwd(&cv, ptr(xz), fptr(l.conv_w), fptr(l.conv_b), ptr(cs[i].window), ptr(xs), ptr(window), stream),
                  "mpa_conv1d_fwd");
            out = dbc;
            if (own) run(linear(ptr(xs), ED, ED, l.xp, Tensor(), dbc));
            else at::mm_out(out, xs2, l.xp.t());
        }
        out = delta;
        if (!proj && own) run(linear(ptr(dbc), P, l.Rp, l.dtp, Tensor(), delta));
        else if (!proj) at::mm_out(out, dlow, l.dtp.t());
        const char* bc = static_cast<const char*>(ptr(dbc)) + l.Rp * es;
        const char* z = static_cast<const char*>(ptr(xz)) + ED * es;
        if (proj)
            check(mpa_sscan_fwd_proj(&sc, ptr(xs), ptr(dbc), ptr(l.dtp), a.Rp, fptr(l.A), bc, bc + N * es, fptr(l.D), z, fptr(l.dt_b),
                                     fptr(cs[i].h), ptr(y), fptr(h_last), ptr(ws), ws_bytes, stream),
                  "mpa_sscan_fwd_proj");
        else
            check(mpa_sscan_fwd(&sc, ptr(xs), ptr(delta), fptr(l.A), bc, bc + N * es, fptr(l.D), z, fptr(l.dt_b), fptr(cs[i].h), ptr(y),
                                nullptr, nullptr, fptr(h_last), ptr(ws), ws_bytes, stream),
                  "mpa_sscan_fwd");
        out = hidden;
        if (own) {
            const bool last = i + 1 == n;
            mpa_linear q = linear(ptr(y), ED, ED, l.p[kOutW], l.p[kOutB], last ? result : s);
            q.residual = i == 0 ? ptr(x) : ptr(sum[(i - 1) % 2]);
            q.accumulate = 1;
            if (i > 0) q.io_dtype |= MPA_LINEAR_RESIDUAL_F32;
            if (!last) {
                q.io_dtype |= MPA_LINEAR_Y_F32;
                q.y_ssq = fptr(ssq);
            }
            // the rows of the next layer's in_proj: those of the stream times its norm's weight (1 / rms is a factor of the product)
            run(q, last ? nullptr : fptr(hs[i + 1].norm_w), last ? nullptr : ptr(normed));
        } else if (split_product(y, l.p[kOutW], l.p[kOutB], hidden, stream)) {
        } else if (l.p[kOutB].defined()) {
            at::addmm_out(out, l.p[kOutB], y, l.p[kOutW].t());
        } else {
            mm_into(hidden, y, l.p[kOutW], false, stream);
        }
        in = ptr(hidden);
        if (keep) cs[i] = {h_last, window};
    }
    if (own) return result;
    const Tensor last = n > 1 ? sum[(n - 1) % 2] : x.view({T, d});
    return at::add(hidden, last).view({Bs, L, d});
}

// A sequence through the residual blocks: (y, list of caches or None), or None.
py::object stack_forward(const py::list& layers, const Tensor& x_in, const py::object& caches, bool return_caches,
                         const PackedPlan& packed) {
    const size_t n = layers.size();
    if (at::GradMode::is_enabled() || !native_call(x_in) || x_in.dim() != 3 || n == 0 || x_in.numel() == 0) return py::none();
    const int64_t Bs = x_in.size(0);
    std::vector<Layer> hs(n);
    std::vector<Cache> cs(n);
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x_in.device());
    for (size_t i = 0; i < n; ++i) {
        if (!find_layer(layers[i].ptr(), x_in, hs[i]) || !hs[i].m->forward_ok) return py::none();
        const MixerHandle &l = *hs[i].m, &a = *hs[0].m;
        if (l.d != a.d || l.ED != a.ED || l.N != a.N || l.Rp != a.Rp || l.padded_rows() != a.padded_rows()) return py::none();
        if (!caches.is_none()) {
            const py::object c = caches[py::int_(i)];
            if (!read_cache(c.ptr(), cs[i]) || !cache_fits(cs[i], l, Bs, false)) return py::none();
        }
    }
    const Tensor x = x_in.contiguous();
    if (reinterpret_cast<uintptr_t>(x.const_data_ptr()) % 16) return py::none();
    form_layers(hs, true);
    Tensor y;
    {
        const py::gil_scoped_release nogil;
        y = run_sequence(hs, x, cs, return_caches, unpack(packed));
    }
    if (!return_caches) return py::make_tuple(y, py::none());
    py::list after;
    for (const Cache& c : cs) after.append(pair(c.h, c.window));
    return py::make_tuple(y, after);
}

// A plain bfloat16 nn.Linear without bias over many rows (the head of a model, by which its scores of a sequence are formed), where a kernel of
// this package is the faster one; else None.  (Not float32, though a product on cut operands takes half the library's time: it keeps 2^-23 of a
// value, so that a weight that selects a column does not give that column.)
constexpr int64_t kHeadRows = 64;
py::object linear_rows(const py::object& module, const Tensor& x_in) {
    if (at::GradMode::is_enabled() || !native_call(x_in) || (PyObject*)Py_TYPE(module.ptr()) != types->linear.ptr() || x_in.dim() < 2 ||
        x_in.scalar_type() != at::kBFloat16 || x_in.numel() == 0)
        return py::none();
    // (a trace or a mode sees the calls of torch that this one would stand in for)
    if (torch::jit::tracer::isTracing() || c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::PythonTorchFunctionTLS::stack_len() > 0 ||
        x_in.key_set().has(c10::DispatchKey::Python))
        return py::none();
    Instance self;
    if (!self.plain(dict_of(module.ptr()), types->linear_names)) return py::none();
    const Keys& k = keys();
    self.find(k.weight, k.bias);
    Param weight;
    Tensor w;
    bool changed = false;
    if (self.pair[1] != Py_None || !weight.take(self.pair[0], w, changed) || !w.defined() || w.scalar_type() != at::kBFloat16 || w.dim() != 2 ||
        w.device() != x_in.device() || w.size(1) != x_in.size(-1) || !w.is_contiguous())
        return py::none();
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x_in.device());
    const int64_t K = w.size(1), M = w.size(0), T = x_in.numel() / K;
    if (T < kHeadRows || !x_in.is_contiguous()) return py::none();
    mpa_gemm g{ptr(x_in), ptr(w), ptr(w), T, M, K, K, K, M, 0};  // (y: for the rule)
    if (!mpa_gemm_faster(&g)) return py::none();
    std::vector<int64_t> sizes = x_in.sizes().vec();
    sizes.back() = M;
    const py::gil_scoped_release nogil;
    const Tensor y = empty(sizes, at::kBFloat16, x_in);
    g.y = ptr(y);
    check(mpa_gemm_run(&g, stream_of(x_in)), "mpa_gemm_run");
    const py::gil_scoped_acquire gil;
    return py::cast(y);
}

}  // namespace

void bind_model(py::module_& m) {
    // copies of a module (copy.deepcopy, pickle) take None in a handle's place and make their own
    const auto copies = [](auto& cls) {
        typedef typename std::remove_reference_t<decltype(cls)>::type H;
        cls.def("__reduce__", [](const H&) { return py::make_tuple(py::type::of(py::none()), py::tuple()); })
            .def("__deepcopy__", [](const H&, const py::object&) { return py::none(); });
    };
    py::class_<MixerHandle> mixer(m, "MixerHandle");
    copies(mixer);
    mixer.def("expire", &MixerHandle::expire);
    py::class_<NormHandle> norm(m, "NormHandle");
    copies(norm);
    // {method: what it was when the package was imported} of each class that native calls stand in for
    m.def("register_types", [](const py::object& block, const py::dict& block_methods, const py::object& norm, const py::dict& norm_methods,
                               const py::object& linear, const py::dict& linear_methods, const py::object& module, const py::dict& module_methods,
                               const py::object& conv, const py::list& global_hooks) {
        Types* t = new Types();
        t->block = block;
        t->norm = norm;
        t->linear = linear;
        t->conv = conv;
        auto watch = [&](const py::object& cls, const py::dict& methods, std::vector<Ref>* names) {
            PyObject* dict = reinterpret_cast<PyTypeObject*>(cls.ptr())->tp_dict;
            for (const auto& [name, was] : methods) {
                t->methods.push_back({Ref(dict), Ref(name.ptr()), Ref(was.ptr())});
                if (names) names->push_back(Ref(name.ptr()));
            }
        };
        watch(block, block_methods, &t->block_names);
        watch(norm, norm_methods, &t->norm_names);
        watch(linear, linear_methods, &t->linear_names);
        watch(module, module_methods, nullptr);
        for (const auto& h : global_hooks) t->global_hooks.push_back(Ref(h.ptr()));
        types = t;
    });
    m.def("stack_step", &stack_step);
    m.def("block_step", &block_step);
    m.def("stack_forward", &stack_forward);
    m.def("linear_rows", &linear_rows);
}

}  // namespace mpa_host
