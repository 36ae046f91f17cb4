// The layer stack without gradients, from C++: decode steps and forward passes of a list of
// residual blocks in one call from Python.
//
// What a layer needs from its modules is looked up once and kept in a LayerHandle in the
// block's __dict__: raw pointers for the kernels, float32 forms of the small parameters, the weights
// of the two narrow projections padded for the GEMM library.  Every call checks, by comparing pointers
// and version counters, that the parameters are the ones the handle was made from and that nothing
// (a hook, a wrapped or replaced submodule) wants to see the calls that are skipped; a stack that
// fails the check is run module by module in Python.
#include "host.h"

namespace mpa_host {
namespace {

// ---- views of Python modules --------------------------------------------------------------------

struct Ref {  // an owned PyObject*
    PyObject* o = nullptr;
    Ref() = default;
    explicit Ref(PyObject* borrowed) : o(borrowed) { Py_XINCREF(o); }
    Ref(const Ref& r) : o(r.o) { Py_XINCREF(o); }
    Ref(Ref&& r) noexcept : o(r.o) { r.o = nullptr; }
    Ref& operator=(Ref r) { std::swap(o, r.o); return *this; }
    ~Ref() { Py_XDECREF(o); }
};

PyObject* key(const char* s) { return PyUnicode_InternFromString(s); }
struct Keys {
    PyObject *modules = key("_modules"), *params = key("_parameters"), *fwd = key("_forward_hooks"), *pre = key("_forward_pre_hooks"),
             *handle = key("_mpa_handle"), *mixer = key("mixer"), *norm = key("norm"), *weight = key("weight"), *bias = key("bias"),
             *A_log = key("A_log"), *D = key("D"), *forward = key("forward");
};
const Keys& keys() {
    static const Keys k;
    return k;
}

PyObject* dict_of(PyObject* module) {
    PyObject** d = _PyObject_GetDictPtr(module);
    return d ? *d : nullptr;
}
PyObject* get(PyObject* dict, PyObject* k) { return dict ? PyDict_GetItem(dict, k) : nullptr; }

// A submodule: found under its name, of exactly the expected type, without hooks.
struct Sub {
    PyObject* name = nullptr;
    bool called = false;  // through __call__, so that hooks would run
    Ref mod, params, fwd, pre;
    bool open(PyObject* modules, const char* n, PyObject* type, bool is_called) {
        name = key(n);
        called = is_called;
        PyObject* m = get(modules, name);
        if (!m || (PyObject*)Py_TYPE(m) != type) return false;
        PyObject* d = dict_of(m);
        mod = Ref(m);
        params = Ref(get(d, keys().params));
        fwd = Ref(get(d, keys().fwd));
        pre = Ref(get(d, keys().pre));
        return params.o && fwd.o && pre.o && !get(d, keys().forward);
    }
    bool same(PyObject* modules) const {
        return get(modules, name) == mod.o && (!called || (PyDict_Size(fwd.o) == 0 && PyDict_Size(pre.o) == 0));
    }
};

// A parameter and the state it was last seen in.
struct Param {
    PyObject *params = nullptr, *name = nullptr;
    Tensor t;
    const void* impl = nullptr;
    const void* data = nullptr;
    uint32_t version = 0;
    static uint32_t version_of(const Tensor& t) { return t.is_inference() ? 0 : t._version(); }
    bool changed() {  // also takes the new state over
        PyObject* o = get(params, name);
        const bool there = o && THPVariable_Check(o);
        if (!there) {
            const bool was = impl != nullptr;
            *this = Param{params, name};
            return was;
        }
        const Tensor& now = THPVariable_Unpack(o);
        const void* im = now.unsafeGetTensorImpl();
        if (im == impl && now.const_data_ptr() == data && version_of(now) == version) return false;
        t = now;
        impl = im;
        data = now.const_data_ptr();
        version = version_of(now);
        return true;
    }
};

enum { kNormW, kInW, kInB, kConvW, kConvB, kXW, kDtW, kDtB, kALog, kD, kOutW, kOutB, kParams };

// Refreshed in place, so that a captured graph goes on reading current values from the same memory.
void refresh(Tensor& kept, const Tensor& fresh) {
    if (kept.defined() && kept.sizes() == fresh.sizes() && kept.device() == fresh.device() && kept.scalar_type() == fresh.scalar_type())
        kept.copy_(fresh);
    else
        kept = fresh;
}
// float32 form of a small parameter: the parameter itself when it is that already, else a buffer
struct F32 {
    Tensor t, own;
    void take(const Tensor& p) {
        if (!p.defined()) t = Tensor();
        else if (p.scalar_type() == at::kFloat && p.is_contiguous()) t = p.detach();
        else { refresh(own, f32c(p.detach())); t = own; }
    }
};

struct LayerHandle {
    bool usable = false;      // the block has the plain structure
    bool decode_ok = false;   // ... and shapes that mpa_decode_layer_step takes
    bool forward_ok = false;  // ... and that stack_forward takes
    bool with_norm = false;
    Ref block_modules, mixer_modules, mixer, mixer_params, mixer_fwd, mixer_pre;
    Sub norm, in_proj, conv1d, x_proj, dt_proj, out_proj;
    Param p[kParams];
    int64_t d = 0, ED = 0, N = 0, R = 0, K = 0;
    double eps = 0;
    bool fused_softplus = true, stale = true;
    F32 norm_w, conv_w, conv_b, dt_b, D;
    Tensor A;                                    // -exp(A_log), float32
    Tensor in_wt, out_wt, xp, dtp, xp_t, dtp_t;  // (transposed views of) the GEMM weights
    int64_t Rp = 0;
    bool padded = false;  // xp .. dtp_t are up to date
    at::ScalarType dt = at::kFloat;
    c10::Device device{at::kCPU};

    // `block`: a ResidualBlock (norm + mixer) or a bare MambaBlock; types: the exact classes expected
    LayerHandle(const py::object& block, const py::object& block_type, const py::object& norm_type, bool residual) {
        with_norm = residual;
        PyObject* bm = get(dict_of(block.ptr()), keys().modules);
        if (!bm) return;
        PyObject* mx = block.ptr();
        if (residual) {
            block_modules = Ref(bm);
            mx = get(bm, keys().mixer);
            if (!norm.open(bm, "norm", norm_type.ptr(), false)) return;
        }
        if (!mx || (PyObject*)Py_TYPE(mx) != block_type.ptr()) return;
        if (residual) mixer = Ref(mx);  // (a bare block's handle sits in its own __dict__: no reference to itself)
        PyObject* md = dict_of(mx);
        PyObject* mm = get(md, keys().modules);
        mixer_modules = Ref(mm);
        mixer_params = Ref(get(md, keys().params));
        mixer_fwd = Ref(get(md, keys().fwd));
        mixer_pre = Ref(get(md, keys().pre));
        const py::module_ nn = py::module_::import("torch.nn");
        PyObject* linear = nn.attr("Linear").ptr();
        if (!mm || !mixer_params.o || !mixer_fwd.o || !mixer_pre.o || get(md, keys().forward)) return;
        if (!in_proj.open(mm, "in_proj", linear, true) || !conv1d.open(mm, "conv1d", nn.attr("Conv1d").ptr(), false) ||
            !x_proj.open(mm, "x_proj", linear, true) || !dt_proj.open(mm, "dt_proj", linear, false) ||
            !out_proj.open(mm, "out_proj", linear, true))
            return;
        const py::object cfg = py::reinterpret_borrow<py::object>(mx).attr("config");
        if (cfg.attr("inner_layernorms").cast<bool>()) return;
        d = cfg.attr("d_model").cast<int64_t>();
        ED = cfg.attr("d_inner").cast<int64_t>();
        N = cfg.attr("d_state").cast<int64_t>();
        R = cfg.attr("dt_rank").cast<int64_t>();
        K = cfg.attr("d_conv").cast<int64_t>();
        Rp = (R + 63) / 64 * 64;
        fused_softplus = cfg.attr("fused_softplus").cast<bool>();
        if (residual) eps = py::reinterpret_borrow<py::object>(norm.mod.o).attr("eps").cast<double>();
        const Keys& k = keys();
        if (residual) p[kNormW] = Param{norm.params.o, k.weight};
        else p[kNormW] = Param{mixer_params.o, k.weight};  // no such parameter: stays undefined
        p[kInW] = Param{in_proj.params.o, k.weight};
        p[kInB] = Param{in_proj.params.o, k.bias};
        p[kConvW] = Param{conv1d.params.o, k.weight};
        p[kConvB] = Param{conv1d.params.o, k.bias};
        p[kXW] = Param{x_proj.params.o, k.weight};
        p[kDtW] = Param{dt_proj.params.o, k.weight};
        p[kDtB] = Param{dt_proj.params.o, k.bias};
        p[kALog] = Param{mixer_params.o, k.A_log};
        p[kD] = Param{mixer_params.o, k.D};
        p[kOutW] = Param{out_proj.params.o, k.weight};
        p[kOutB] = Param{out_proj.params.o, k.bias};
        usable = true;
    }

    // the dictionaries are those of this block (a shallow copy brings the handle of its original along)
    bool belongs_to(PyObject* dict) const {
        return !usable || get(dict, keys().modules) == (with_norm ? block_modules.o : mixer_modules.o);
    }

    bool same_modules() const {
        if (with_norm && (!norm.same(block_modules.o) || get(block_modules.o, keys().mixer) != mixer.o)) return false;
        PyObject* mm = mixer_modules.o;
        return in_proj.same(mm) && conv1d.same(mm) && x_proj.same(mm) && dt_proj.same(mm) && out_proj.same(mm) &&
               PyDict_Size(mixer_fwd.o) == 0 && PyDict_Size(mixer_pre.o) == 0;
    }

    // Whether the block can run here with activations like x; brings the derived weights up to date.
    bool ready(const Tensor& x) {
        if (!usable || !same_modules()) return false;
        bool changed = stale;
        for (Param& q : p) changed |= q.changed();
        if (changed) {
            stale = true;
            decode_ok = forward_ok = false;
            if (!prepare()) return false;
            stale = false;
        }
        return (decode_ok || forward_ok) && x.scalar_type() == dt && x.device() == device && x.size(-1) == d;
    }

    bool prepare() {
        const Tensor& w = p[kInW].t;
        if (!w.defined() || !w.is_cuda() || (w.scalar_type() != at::kFloat && w.scalar_type() != at::kBFloat16)) return false;
        dt = w.scalar_type();
        device = w.device();
        for (int i : {kInW, kXW, kDtW, kOutW, kInB, kOutB}) {
            const Tensor& t = p[i].t;
            const bool optional = i == kInB || i == kOutB;
            if (!t.defined() && optional) continue;
            if (!t.defined() || t.scalar_type() != dt || t.device() != device || !t.is_contiguous()) return false;
        }
        for (int i : {kNormW, kConvW, kConvB, kDtB, kALog, kD})
            if (p[i].t.defined() && p[i].t.device() != device) return false;
        if (!p[kConvW].t.defined() || !p[kALog].t.defined() || !p[kD].t.defined()) return false;
        if (p[kInW].t.sizes() != at::IntArrayRef({2 * ED, d}) || p[kXW].t.sizes() != at::IntArrayRef({R + 2 * N, ED}) ||
            p[kDtW].t.sizes() != at::IntArrayRef({ED, R}) || p[kOutW].t.sizes() != at::IntArrayRef({d, ED}) ||
            p[kConvW].t.numel() != ED * K || p[kALog].t.sizes() != at::IntArrayRef({ED, N}) || p[kD].t.numel() != ED)
            return false;
        norm_w.take(p[kNormW].t);
        conv_w.take(p[kConvW].t);
        conv_b.take(p[kConvB].t);
        dt_b.take(p[kDtB].t);
        D.take(p[kD].t);
        refresh(A, p[kALog].t.detach().to(at::kFloat).exp().neg_());
        in_wt = p[kInW].t.detach().t();
        out_wt = p[kOutW].t.detach().t();
        padded = false;
        const int64_t vec = dt == at::kFloat ? 4 : 8;
        decode_ok = K >= 2 && K <= 4 && d % vec == 0 && ED % vec == 0 && N % 4 == 0 && N <= MPA_MAX_DSTATE && R <= 2048;
        for (int i : {kInW, kXW, kOutW}) decode_ok &= reinterpret_cast<uintptr_t>(p[i].data) % 16 == 0;
        for (const Tensor* t : {&norm_w.t, &A})
            decode_ok &= !t->defined() || reinterpret_cast<uintptr_t>(t->const_data_ptr()) % 16 == 0;
        forward_ok = K >= 2 && K <= 4 && N <= MPA_MAX_DSTATE && fused_softplus && d % vec == 0 && d <= 512 * vec && dt_b.t.defined();
        return true;
    }

    // x_proj and dt_proj in the shape the GEMM library serves best: the low-rank width R is the K of
    // dt_proj and R + 2N the rows of x_proj, both odd for its tiles (48 and 80 at width 768).  With R
    // rounded up to a multiple of 64 by zeros and the rows regrouped as [delta | 0 | B | C | 0], the two
    // products take 21 + 26 us instead of 25 + 38 us at 32768 rows in bfloat16.
    void pad() {
        if (padded) return;
        padded = true;
        const Tensor &xw = p[kXW].t, &dw = p[kDtW].t;
        if (Rp == R) {
            xp = xw.detach();
            dtp = dw.detach();
        } else {
            const int64_t rows = (Rp + 2 * N + 63) / 64 * 64;
            Tensor fx = at::zeros({rows, ED}, xw.options()), fd = at::zeros({ED, Rp}, dw.options());
            fx.narrow(0, 0, R).copy_(xw.detach().narrow(0, 0, R));
            fx.narrow(0, Rp, 2 * N).copy_(xw.detach().narrow(0, R, 2 * N));
            fd.narrow(1, 0, R).copy_(dw.detach());
            refresh(xp, fx);
            refresh(dtp, fd);
        }
        xp_t = xp.t();
        dtp_t = dtp.t();
    }

    mpa_decode_layer desc(int64_t batch) const {
        mpa_decode_layer s{};
        s.batch = batch; s.d_model = d; s.dim = ED; s.dstate = N; s.dt_rank = R;
        s.d_conv = (int)K;
        s.io_dtype = dt == at::kFloat ? MPA_F32 : MPA_BF16;
        s.norm = with_norm;
        s.eps = (float)eps;
        s.norm_weight = fptr(norm_w.t);
        s.in_weight = p[kInW].data; s.in_bias = p[kInB].data;
        s.conv_weight = fptr(conv_w.t); s.conv_bias = fptr(conv_b.t);
        s.x_weight = p[kXW].data; s.dt_weight = p[kDtW].data;
        s.dt_bias = fptr(dt_b.t); s.A = fptr(A); s.D = fptr(D.t);
        s.out_weight = p[kOutW].data; s.out_bias = p[kOutB].data;
        return s;
    }
};

struct Types {  // the exact Python classes that a handle is made for
    py::object block, norm;
};
Types* types = nullptr;  // set by register_types, kept for the interpreter's lifetime

LayerHandle* handle_of(PyObject* block, bool residual) {
    PyObject* dict = dict_of(block);
    if (!dict || !types) return nullptr;
    PyObject* o = get(dict, keys().handle);
    if (!o || o == Py_None || !py::cast<LayerHandle*>(py::handle(o))->belongs_to(dict)) {
        const py::object h = py::cast(new LayerHandle(py::reinterpret_borrow<py::object>(block), types->block, types->norm, residual),
                                      py::return_value_policy::take_ownership);
        PyDict_SetItem(dict, keys().handle, h.ptr());
        o = h.ptr();
    }
    return py::cast<LayerHandle*>(py::handle(o));
}

bool fits(const Tensor& t, at::IntArrayRef shape, at::ScalarType dt, const c10::Device& dev) {
    return t.scalar_type() == dt && t.device() == dev && t.sizes() == shape && t.is_contiguous() &&
           reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
}

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
bool cache_fits(const Cache& c, const LayerHandle& l, int64_t batch, bool need_h) {
    if (!c.h.defined() ? need_h : !fits(c.h, {batch, l.ED, l.N}, at::kFloat, l.device)) return false;
    return c.window.scalar_type() == l.dt && c.window.device() == l.device && c.window.is_contiguous() &&
           c.window.sizes() == at::IntArrayRef({batch, l.ED, l.K - 1});
}

py::object pair(const Tensor& h, const Tensor& w) { return py::make_tuple(h, w); }

// ---- decode -------------------------------------------------------------------------------------

// One token through the residual blocks `layers`; the caches are updated in place or replaced in the
// list.  None: not a stack that can run here (the caller goes on in Python).
py::object stack_step(const py::list& layers, const Tensor& x_in, const py::list& caches, bool inplace) {
    const size_t n = layers.size();
    if (at::GradMode::is_enabled() || !x_in.is_cuda() || x_in.dim() != 2 || n == 0 || caches.size() < n ||
        x_in.size(0) > MPA_DECODE_MAX_BATCH || x_in.size(0) == 0)
        return py::none();
    const int64_t batch = x_in.size(0);
    std::vector<LayerHandle*> hs(n);
    std::vector<Cache> cs(n);
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x_in.device());
    for (size_t i = 0; i < n; ++i) {
        hs[i] = handle_of(layers[i].ptr(), true);
        if (!hs[i] || !hs[i]->ready(x_in) || !hs[i]->decode_ok || hs[i]->d != hs[0]->d) return py::none();
        if (!read_cache(caches[i].ptr(), cs[i]) || !cache_fits(cs[i], *hs[i], batch, inplace)) return py::none();
    }
    const Tensor x = x_in.contiguous();
    if (reinterpret_cast<uintptr_t>(x.const_data_ptr()) % 16) return py::none();
    const auto dt = x.scalar_type();
    const int64_t d = x.size(1);
    // two rows per sequence and two scaled rows, used in turn (a kernel never writes what it reads), with
    // the partial sums of squares of the latter
    const int64_t tiles = (d + 15) / 16;
    const mpa_decode_layer any = hs[0]->desc(batch);
    const size_t scaled_bytes = mpa_decode_scaled_bytes(&any);
    const Tensor spare = empty({batch, d}, dt, x), y = empty({batch, d}, dt, x), scaled_rows = scratch(2 * scaled_bytes, x),
                 ssq = empty({2, tiles * batch}, at::kFloat, x);
    size_t ws_bytes = 0;
    for (LayerHandle* h : hs) {
        const mpa_decode_layer s = h->desc(batch);
        ws_bytes = std::max(ws_bytes, mpa_decode_layer_workspace_bytes(&s));
    }
    const Tensor ws = scratch(ws_bytes, x);
    void* stream = stream_of(x);
    // the last layer writes y, the others y and a spare row in turn
    const void* in = ptr(x);
    const void* scaled = nullptr;
    const float* sums = nullptr;
    for (size_t i = 0; i < n; ++i) {
        LayerHandle& l = *hs[i];
        Cache out = cs[i];
        if (!inplace) {
            out.h = empty({batch, l.ED, l.N}, at::kFloat, x);
            out.window = empty({batch, l.ED, l.K - 1}, dt, x);
        }
        const mpa_decode_layer s = l.desc(batch);
        void* to = (n - 1 - i) % 2 == 0 ? ptr(y) : ptr(spare);
        // (a norm without a weight has nothing to scale by: the next layer forms its own sums)
        const float* next_w = i + 1 < n ? fptr(hs[i + 1]->norm_w.t) : nullptr;
        void* to_scaled = static_cast<char*>(ptr(scaled_rows)) + (i % 2) * scaled_bytes;
        float* to_sums = fptr(ssq) + (i % 2) * tiles * batch;
        check(mpa_decode_layer_step(&s, in, scaled, sums, to, next_w, to_scaled, to_sums, fptr(cs[i].h), fptr(out.h), ptr(cs[i].window),
                                    ptr(out.window), ptr(ws), ws_bytes, stream),
              "mpa_decode_layer_step");
        in = to;
        scaled = next_w ? to_scaled : nullptr;
        sums = next_w ? to_sums : nullptr;
        if (!inplace) caches[i] = pair(out.h, out.window);
    }
    return py::cast(y);
}

// One token through one MambaBlock (no norm, no residual): (y, h, window) or None.
py::object block_step(const py::object& block, const Tensor& x_in, const Opt& h_in, const Tensor& window, bool inplace) {
    if (at::GradMode::is_enabled() || !x_in.is_cuda() || x_in.dim() != 2 || x_in.size(0) > MPA_DECODE_MAX_BATCH || x_in.size(0) == 0)
        return py::none();
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x_in.device());
    LayerHandle* l = handle_of(block.ptr(), false);
    const int64_t batch = x_in.size(0);
    const Cache in{val(h_in), window};
    if (!l || !l->ready(x_in) || !l->decode_ok || !cache_fits(in, *l, batch, inplace)) return py::none();
    const Tensor x = x_in.contiguous();
    if (reinterpret_cast<uintptr_t>(x.const_data_ptr()) % 16) return py::none();
    Cache out = in;
    if (!inplace) {
        out.h = empty({batch, l->ED, l->N}, at::kFloat, x);
        out.window = empty({batch, l->ED, l->K - 1}, x.scalar_type(), x);
    }
    const Tensor y = empty({batch, l->d}, x.scalar_type(), x);
    const mpa_decode_layer s = l->desc(batch);
    const size_t nbytes = mpa_decode_layer_workspace_bytes(&s);
    const Tensor ws = scratch(nbytes, x);
    check(mpa_decode_layer_step(&s, ptr(x), nullptr, nullptr, ptr(y), nullptr, nullptr, nullptr, fptr(in.h), fptr(out.h), ptr(in.window),
                                ptr(out.window), ptr(ws), nbytes, stream_of(x)),
          "mpa_decode_layer_step");
    return py::make_tuple(y, out.h, out.window);
}

// ---- forward without gradients ------------------------------------------------------------------

// A sequence through the residual blocks: (y, list of caches or None), or None.  The activations of a
// layer live in buffers that every layer uses again.
py::object stack_forward(const py::list& layers, const Tensor& x_in, const py::object& caches, bool return_caches,
                         const PackedPlan& packed) {
    const size_t n = layers.size();
    if (at::GradMode::is_enabled() || !x_in.is_cuda() || x_in.dim() != 3 || n == 0 || x_in.numel() == 0) return py::none();
    const int64_t Bs = x_in.size(0), L = x_in.size(1), T = Bs * L;
    std::vector<LayerHandle*> hs(n);
    std::vector<Cache> cs(n);
    at::AutoDispatchBelowADInplaceOrView below;
    const c10::DeviceGuard guard(x_in.device());
    for (size_t i = 0; i < n; ++i) {
        hs[i] = handle_of(layers[i].ptr(), true);
        const LayerHandle& a = *hs[0];
        if (!hs[i] || !hs[i]->ready(x_in) || !hs[i]->forward_ok) return py::none();
        hs[i]->pad();
        if (hs[i]->d != a.d || hs[i]->ED != a.ED || hs[i]->N != a.N || hs[i]->Rp != a.Rp) return py::none();
        if (!caches.is_none()) {
            const py::object c = caches[py::int_(i)];
            if (!read_cache(c.ptr(), cs[i]) || !cache_fits(cs[i], *hs[i], Bs, false)) return py::none();
        }
    }
    const Plan plan = unpack(packed);
    const LayerHandle& a = *hs[0];
    const Tensor x = x_in.contiguous();
    if (reinterpret_cast<uintptr_t>(x.const_data_ptr()) % 16) return py::none();
    const auto dt = x.scalar_type();
    const int io = io_dtype(dt);
    const int64_t d = a.d, ED = a.ED, N = a.N, P = a.xp.size(0);
    const size_t es = x.element_size();
    void* stream = stream_of(x);
    const Tensor normed = empty({T, d}, dt, x), xz = empty({T, 2 * ED}, dt, x), xs = empty({Bs, L, ED}, dt, x),
                 dbc = empty({T, P}, dt, x), delta = empty({T, ED}, dt, x), y = empty({T, ED}, dt, x), hidden = empty({T, d}, dt, x);
    Tensor sum[2];
    if (n > 1) { sum[0] = empty({T, d}, dt, x); sum[1] = empty({T, d}, dt, x); }
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
    sc.plan_states_per_lane = plan.fwd_ns; sc.plan_segments = plan.fwd_segments; sc.plan_flags = plan.flags;
    const size_t ws_bytes = mpa_sscan_fwd_workspace_bytes(&sc, 0);
    const Tensor ws = scratch(ws_bytes, x);

    py::list new_caches;
    const void* in = ptr(x);
    const void* residual = nullptr;
    for (size_t i = 0; i < n; ++i) {
        LayerHandle& l = *hs[i];
        const Tensor& s = sum[i % 2];
        check(mpa_rmsnorm_fwd(in, residual, fptr(l.norm_w.t), ptr(normed), residual ? ptr(s) : nullptr, nullptr, T, d, (float)l.eps, io, stream),
              "mpa_rmsnorm_fwd");
        residual = residual ? ptr(s) : in;
        Tensor out = xz;
        if (l.p[kInB].t.defined()) at::addmm_out(out, l.p[kInB].t.detach(), normed, l.in_wt);
        else at::mm_out(out, normed, l.in_wt);
        Tensor window, h_last;
        if (return_caches) {
            window = empty({Bs, ED, l.K - 1}, dt, x);
            h_last = empty({Bs, ED, N}, at::kFloat, x);
        }
        cv.kernel = (int)l.K;
        check(mpa_conv1d_fwd(&cv, ptr(xz), fptr(l.conv_w.t), fptr(l.conv_b.t), ptr(cs[i].window), ptr(xs), ptr(window), stream),
              "mpa_conv1d_fwd");
        out = dbc;
        at::mm_out(out, xs2, l.xp_t);
        out = delta;
        at::mm_out(out, dlow, l.dtp_t);
        const char* bc = static_cast<const char*>(ptr(dbc)) + l.Rp * es;
        check(mpa_sscan_fwd(&sc, ptr(xs), ptr(delta), fptr(l.A), bc, bc + N * es, fptr(l.D.t), static_cast<const char*>(ptr(xz)) + ED * es,
                            fptr(l.dt_b.t), fptr(cs[i].h), ptr(y), nullptr, nullptr, fptr(h_last), ptr(ws), ws_bytes, stream),
              "mpa_sscan_fwd");
        out = hidden;
        if (l.p[kOutB].t.defined()) at::addmm_out(out, l.p[kOutB].t.detach(), y, l.out_wt);
        else at::mm_out(out, y, l.out_wt);
        in = ptr(hidden);
        if (return_caches) new_caches.append(pair(h_last, window));
    }
    const Tensor last = n > 1 ? sum[(n - 1) % 2] : x.view({T, d});
    const Tensor result = at::add(hidden, last).view({Bs, L, d});
    return py::make_tuple(result, return_caches ? py::object(new_caches) : py::object(py::none()));
}

}  // namespace

void bind_model(py::module_& m) {
    // copies of a module (copy.deepcopy, pickle) take None in its place and make their own
    const auto gone = [](const LayerHandle&) { return py::make_tuple(py::type::of(py::none()), py::tuple()); };
    py::class_<LayerHandle>(m, "LayerHandle")
        .def("__reduce__", gone)
        .def("__deepcopy__", [](const LayerHandle&, const py::object&) { return py::none(); });
    m.def("register_types", [](const py::object& block, const py::object& norm) {
        if (!types) types = new Types();
        types->block = block;
        types->norm = norm;
    });
    m.def("stack_step", &stack_step);
    m.def("block_step", &block_step);
    m.def("stack_forward", &stack_forward);
}

}  // namespace mpa_host
