// A residual block or mixer of the package as C++ sees it: which parameters it has, whether it is of the
// plain kind, and the forms of its weights that the kernels take.
//
// What a layer needs from its modules is looked up once and kept in handles, a MixerHandle in the mixer's
// __dict__ and a NormHandle in the residual block's.  Every call checks, by comparing pointers and version counters, that the parameters are
// the ones the handle was made from and that nothing (a hook, a wrapped or replaced submodule, autocast) wants
// to see the calls that are skipped; a block that fails the check is run module by module in Python.
#pragma once

#include <ATen/autocast_mode.h>
#include <c10/core/Event.h>
#include <c10/hip/HIPGraphsC10Utils.h>

#include "host.h"

namespace mpa_host {

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

inline PyObject* key(const char* s) { return PyUnicode_InternFromString(s); }
struct Keys {
    PyObject *modules = key("_modules"), *params = key("_parameters"), *fwd = key("_forward_hooks"), *pre = key("_forward_pre_hooks"),
             *bwd = key("_backward_hooks"), *bpre = key("_backward_pre_hooks"),
             *handle = key("_mpa_handle"), *mixer = key("mixer"), *norm = key("norm"), *weight = key("weight"), *bias = key("bias"),
             *A_log = key("A_log"), *D = key("D"), *forward = key("forward");
};
inline const Keys& keys() {
    static const Keys k;
    return k;
}

inline PyObject* dict_of(PyObject* module) {
    PyObject** d = _PyObject_GetDictPtr(module);
    return d ? *d : nullptr;
}
inline PyObject* get(PyObject* dict, PyObject* k) { return dict ? PyDict_GetItem(dict, k) : nullptr; }

struct Hooks {
    Ref dicts[4];
    bool open(PyObject* module_dict) {
        const Keys& k = keys();
        PyObject* const names[4] = {k.fwd, k.pre, k.bwd, k.bpre};
        for (int i = 0; i < 4; ++i) {
            dicts[i] = Ref(get(module_dict, names[i]));
            if (!dicts[i].o) return false;
        }
        return true;
    }
    bool none() const {
        for (const Ref& d : dicts)
            if (PyDict_Size(d.o) != 0) return false;
        return true;
    }
};

// A submodule: found under its name, of exactly the expected type, without hooks.
struct Sub {
    PyObject* name = nullptr;
    bool called = false;  // through __call__, so that hooks would run
    Ref mod, params;
    Hooks hooks;
    bool open(PyObject* modules, const char* n, PyObject* type, bool is_called) {
        name = key(n);
        called = is_called;
        PyObject* m = get(modules, name);
        if (!m || (PyObject*)Py_TYPE(m) != type) return false;
        PyObject* d = dict_of(m);
        mod = Ref(m);
        params = Ref(get(d, keys().params));
        return hooks.open(d) && params.o && !get(d, keys().forward);
    }
    bool same(PyObject* modules) const {
        return get(modules, name) == mod.o && (!called || hooks.none());
    }
};

// A parameter and the state it was last seen in.
struct Param {
    PyObject *params = nullptr, *name = nullptr;
    Tensor t;
    const void* impl = nullptr;
    const void* data = nullptr;
    uint32_t version = 0;
    bool changed() {  // also takes the new state over; an inference tensor has no version counter and may always have changed
        PyObject* o = get(params, name);
        const bool there = o && THPVariable_Check(o);
        if (!there) {
            const bool was = impl != nullptr;
            *this = Param{params, name};
            return was;
        }
        const Tensor& now = THPVariable_Unpack(o);
        const void* im = now.unsafeGetTensorImpl();
        const bool counted = !now.is_inference();
        if (counted && im == impl && now.const_data_ptr() == data && now._version() == version) return false;
        t = now;
        impl = im;
        data = now.const_data_ptr();
        version = counted ? now._version() : 0;
        return true;
    }
};

enum { kInW, kInB, kConvW, kConvB, kXW, kDtW, kDtB, kALog, kD, kOutW, kOutB, kParams };

// A tensor derived from a parameter for the calls without gradients.  It is refreshed in place, so that a captured
// graph goes on reading current values from the same memory.
inline const Tensor& derived(Tensor& kept, at::IntArrayRef shape, at::ScalarType dt, const Tensor& like) {
    if (!kept.defined() || kept.sizes() != shape || kept.device() != like.device() || kept.scalar_type() != dt)
        kept = at::zeros(shape, at::TensorOptions().dtype(dt).device(like.device()));
    return kept;
}
inline mpa_cast_job cast_job(const Tensor& src, const Tensor& dst, int64_t rows, int64_t cols, int64_t src_at = 0, int64_t dst_at = 0,
                             int op = MPA_CAST_COPY, const float* factor = nullptr) {
    mpa_cast_job j{};
    j.src = static_cast<const char*>(ptr(src)) + src_at * src.element_size();
    j.dst = static_cast<char*>(ptr(dst)) + dst_at * dst.element_size();
    j.factor = factor;
    j.rows = rows; j.cols = cols;
    j.src_pitch = src.dim() > 1 ? src.size(-1) : cols;
    j.dst_pitch = dst.dim() > 1 ? dst.size(-1) : cols;
    j.src_dtype = io_dtype(src.scalar_type()); j.dst_dtype = io_dtype(dst.scalar_type());
    j.op = op;
    return j;
}
inline void run_casts(const std::vector<mpa_cast_job>& jobs, const Tensor& like) {
    if (!jobs.empty()) check(mpa_cast(jobs.data(), (int)jobs.size(), stream_of(like)), "mpa_cast");
}
// the elements of a small parameter as one row
inline mpa_cast_job row_job(const Tensor& src, const Tensor& dst) {
    mpa_cast_job j = cast_job(src, dst, 1, src.numel());
    j.src_pitch = j.dst_pitch = src.numel();
    return j;
}
inline mpa_cast_job zero_job(const Tensor& dst, int64_t rows, int64_t cols, int64_t dst_at) {
    return cast_job(dst, dst, rows, cols, 0, dst_at, MPA_CAST_ZERO);
}
// float32 form of a small parameter: the parameter itself when it is that already, else a buffer
struct F32 {
    Tensor t, own;
    void take(const Tensor& p, std::vector<mpa_cast_job>& jobs) {
        t = Tensor();
        if (!p.defined()) return;
        if (p.scalar_type() == at::kFloat) { t = p.detach(); return; }
        t = derived(own, p.sizes(), at::kFloat, p);
        jobs.push_back(row_job(p, own));
    }
};

inline c10::Stream current_stream(const c10::Device& device) { return c10::impl::VirtualGuardImpl(device.type()).getStream(device); }
inline bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }

// Orders the streams that read kept forms after the one that last wrote them, and tells the allocator of them.
// (A capture cannot wait for an event from outside; torch synchronises the device before it begins one.)
struct Written {
    std::optional<c10::Event> event;
    std::optional<c10::Stream> last;  // the stream that wrote, or one that has waited since
    void before(const c10::Stream& s) const {
        if (event && last != s && !capturing()) event->block(s);
    }
    void after(const c10::Stream& s, bool wrote, std::initializer_list<const Tensor*> forms) {
        if (last && last != s)
            for (const Tensor* t : forms)
                if (t->defined()) t->record_stream(s);
        if (capturing()) return;
        if (wrote) {
            if (!event || event->device_index() != s.device_index()) event.emplace(s.device_type());
            event->record(s);
        }
        last = s;
    }
};

struct MixerHandle {
    bool usable = false;      // the block has the plain structure
    bool decode_ok = false;   // ... and shapes that mpa_decode_layer_step takes
    bool forward_ok = false;  // ... and that stack_forward and block_train take
    Ref modules, params;
    Hooks hooks;
    Sub in_proj, conv1d, x_proj, dt_proj, out_proj;
    Param p[kParams];
    int64_t d = 0, ED = 0, N = 0, R = 0, K = 0, Rp = 0;
    bool fused_softplus = true;
    at::ScalarType dt = at::kFloat;
    c10::Device device{at::kCPU};
    // Forms kept for calls without gradients, and the epoch they are of.  Version counters do not show every change
    // of a parameter (writes through .data), and a training loop makes one after each of its calls: a call with
    // gradients forms its own (TrainForms) and begins an epoch.
    uint64_t epoch = 1, formed = 0, padded = 0;  // padded: that of xp .. dtp_t
    Written written;
    F32 conv_w, conv_b, dt_b, D;
    Tensor A;                                    // -exp(A_log), float32
    Tensor in_wt, out_wt, xp, dtp, xp_t, dtp_t;  // (transposed views of) the GEMM weights

    MixerHandle(const py::object& block, const py::object& block_type) {
        PyObject* mx = block.ptr();
        if ((PyObject*)Py_TYPE(mx) != block_type.ptr()) return;
        PyObject* md = dict_of(mx);
        PyObject* mm = get(md, keys().modules);
        modules = Ref(mm);
        params = Ref(get(md, keys().params));
        const py::module_ nn = py::module_::import("torch.nn");
        PyObject* linear = nn.attr("Linear").ptr();
        if (!mm || !params.o || !hooks.open(md) || get(md, keys().forward)) return;
        if (!in_proj.open(mm, "in_proj", linear, true) || !conv1d.open(mm, "conv1d", nn.attr("Conv1d").ptr(), false) ||
            !x_proj.open(mm, "x_proj", linear, true) || !dt_proj.open(mm, "dt_proj", linear, false) ||
            !out_proj.open(mm, "out_proj", linear, true))
            return;
        const py::object cfg = block.attr("config");
        if (cfg.attr("inner_layernorms").cast<bool>()) return;
        d = cfg.attr("d_model").cast<int64_t>();
        ED = cfg.attr("d_inner").cast<int64_t>();
        N = cfg.attr("d_state").cast<int64_t>();
        R = cfg.attr("dt_rank").cast<int64_t>();
        K = cfg.attr("d_conv").cast<int64_t>();
        Rp = (R + 63) / 64 * 64;
        fused_softplus = cfg.attr("fused_softplus").cast<bool>();
        const Keys& k = keys();
        p[kInW] = Param{in_proj.params.o, k.weight};
        p[kInB] = Param{in_proj.params.o, k.bias};
        p[kConvW] = Param{conv1d.params.o, k.weight};
        p[kConvB] = Param{conv1d.params.o, k.bias};
        p[kXW] = Param{x_proj.params.o, k.weight};
        p[kDtW] = Param{dt_proj.params.o, k.weight};
        p[kDtB] = Param{dt_proj.params.o, k.bias};
        p[kALog] = Param{params.o, k.A_log};
        p[kD] = Param{params.o, k.D};
        p[kOutW] = Param{out_proj.params.o, k.weight};
        p[kOutB] = Param{out_proj.params.o, k.bias};
        usable = true;
    }

    // the dictionaries are those of this block (a shallow copy brings the handle of its original along)
    bool belongs_to(PyObject* dict) const { return !usable || get(dict, keys().modules) == modules.o; }

    bool same_modules() const {
        PyObject* mm = modules.o;
        return in_proj.same(mm) && conv1d.same(mm) && x_proj.same(mm) && dt_proj.same(mm) && out_proj.same(mm) && hooks.none();
    }

    // Whether the block can run here with activations like x.
    bool ready(const Tensor& x) {
        if (!usable || !same_modules()) return false;
        bool changed = false;
        for (Param& q : p) changed |= q.changed();
        if (changed) {
            ++epoch;
            decode_ok = forward_ok = false;
            look_over();
        }
        return (decode_ok || forward_ok) && x.scalar_type() == dt && x.device() == device && x.size(-1) == d;
    }

    void expire() { ++epoch; }

    void look_over() {
        const Tensor& w = p[kInW].t;
        if (!w.defined() || !w.is_cuda() || (w.scalar_type() != at::kFloat && w.scalar_type() != at::kBFloat16)) return;
        dt = w.scalar_type();
        device = w.device();
        for (int i : {kInW, kXW, kDtW, kOutW, kInB, kOutB}) {
            const Tensor& t = p[i].t;
            const bool optional = i == kInB || i == kOutB;
            if (!t.defined() && optional) continue;
            if (!t.defined() || t.scalar_type() != dt || t.device() != device || !t.is_contiguous()) return;
        }
        for (int i : {kConvW, kConvB, kDtB, kALog, kD})
            if (p[i].t.defined() && !small_ok(p[i].t, device)) return;
        if (!p[kConvW].t.defined() || !p[kALog].t.defined() || !p[kD].t.defined()) return;
        if (p[kInW].t.sizes() != at::IntArrayRef({2 * ED, d}) || p[kXW].t.sizes() != at::IntArrayRef({R + 2 * N, ED}) ||
            p[kDtW].t.sizes() != at::IntArrayRef({ED, R}) || p[kOutW].t.sizes() != at::IntArrayRef({d, ED}) ||
            p[kConvW].t.numel() != ED * K || p[kALog].t.sizes() != at::IntArrayRef({ED, N}) || p[kD].t.numel() != ED)
            return;
        for (const auto& [i, n] : {std::pair<int, int64_t>{kInB, 2 * ED}, {kConvB, ED}, {kDtB, ED}, {kOutB, d}})
            if (p[i].t.defined() && p[i].t.numel() != n) return;
        const int64_t vec = dt == at::kFloat ? 4 : 8;
        decode_ok = K >= 2 && K <= 4 && d % vec == 0 && ED % vec == 0 && N % 4 == 0 && N <= MPA_MAX_DSTATE && R <= 2048;
        for (int i : {kInW, kXW, kOutW}) decode_ok &= reinterpret_cast<uintptr_t>(p[i].data) % 16 == 0;
        forward_ok = K >= 2 && K <= 4 && N <= MPA_MAX_DSTATE && fused_softplus && d % vec == 0 && d <= 512 * vec && p[kDtB].t.defined();
    }
    static bool small_ok(const Tensor& t, const c10::Device& device) {
        return t.device() == device && t.is_contiguous() && (t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16);
    }

    // Brings the kept forms up to date, xp .. dtp_t among them for a sequence; after ready().  Within a capture nothing
    // runs yet: the next call still finds them old.
    void form(bool sequence) {
        const c10::Stream s = current_stream(device);
        written.before(s);
        const bool small = formed != epoch, wide = sequence && padded != epoch;
        if (small) form_small();
        if (wide) form_padded();
        if (small || wide) {
            const uint64_t of = capturing() ? 0 : epoch;
            if (small) formed = of;
            if (wide) padded = of;
        }
        written.after(s, small || wide, {&conv_w.own, &conv_b.own, &dt_b.own, &D.own, &A, &xp, &dtp});
    }
    void form_small() {
        const Tensor& w = p[kInW].t;
        std::vector<mpa_cast_job> jobs;
        conv_w.take(p[kConvW].t, jobs);
        conv_b.take(p[kConvB].t, jobs);
        dt_b.take(p[kDtB].t, jobs);
        D.take(p[kD].t, jobs);
        derived(A, {ED, N}, at::kFloat, w);
        jobs.push_back(cast_job(p[kALog].t, A, ED, N, 0, 0, MPA_CAST_NEG_EXP));
        run_casts(jobs, w);
        in_wt = p[kInW].t.detach().t();
        out_wt = p[kOutW].t.detach().t();
    }

    // x_proj and dt_proj in the shape the GEMM library serves best: the low-rank width R is the K of
    // dt_proj and R + 2N the rows of x_proj, both odd for its tiles (48 and 80 at width 768).  With R
    // rounded up to a multiple of 64 by zeros and the rows regrouped as [delta | 0 | B | C | 0], the two
    // products take 21 + 26 us instead of 25 + 38 us at 32768 rows in bfloat16.
    int64_t padded_rows() const { return Rp == R ? R + 2 * N : (Rp + 2 * N + 63) / 64 * 64; }
    void pad_jobs(const Tensor& xp, const Tensor& dtp, std::vector<mpa_cast_job>& jobs) const {
        const Tensor &xw = p[kXW].t, &dw = p[kDtW].t;
        jobs.push_back(cast_job(xw, xp, R, ED));
        jobs.push_back(cast_job(xw, xp, 2 * N, ED, R * ED, Rp * ED));
        jobs.push_back(cast_job(dw, dtp, ED, R));
    }
    void form_padded() {
        const Tensor &xw = p[kXW].t, &dw = p[kDtW].t;
        if (Rp == R) {
            xp = xw.detach();
            dtp = dw.detach();
        } else {
            derived(xp, {padded_rows(), ED}, dt, xw);
            derived(dtp, {ED, Rp}, dt, dw);
            std::vector<mpa_cast_job> jobs;
            pad_jobs(xp, dtp, jobs);
            run_casts(jobs, xw);
        }
        xp_t = xp.t();
        dtp_t = dtp.t();
    }

    // What a call with gradients takes in place of the kept forms: made in the call, on its stream, from the parameters
    // as they are, and held by its graph node; one launch.
    struct TrainForms {
        Tensor A, D, dt_b, conv_w, conv_b, xp, dtp;
    };
    TrainForms train_forms() const {
        const Tensor& w = p[kInW].t;
        TrainForms f;
        std::vector<mpa_cast_job> jobs;
        auto f32 = [&](const Tensor& q) {
            if (!q.defined() || q.scalar_type() == at::kFloat) return q.defined() ? q.detach() : q;
            const Tensor t = empty(q.sizes(), at::kFloat, q);
            jobs.push_back(row_job(q, t));
            return t;
        };
        f.conv_w = f32(p[kConvW].t);
        f.conv_b = f32(p[kConvB].t);
        f.dt_b = f32(p[kDtB].t);
        f.D = f32(p[kD].t);
        f.A = empty({ED, N}, at::kFloat, w);
        jobs.push_back(cast_job(p[kALog].t, f.A, ED, N, 0, 0, MPA_CAST_NEG_EXP));
        if (Rp == R) {
            f.xp = p[kXW].t.detach();
            f.dtp = p[kDtW].t.detach();
        } else {
            const int64_t rows = padded_rows(), used = Rp + 2 * N;
            f.xp = empty({rows, ED}, dt, w);
            f.dtp = empty({ED, Rp}, dt, w);
            pad_jobs(f.xp, f.dtp, jobs);
            jobs.push_back(zero_job(f.xp, Rp - R, ED, R * ED));
            if (rows > used) jobs.push_back(zero_job(f.xp, rows - used, ED, used * ED));
            jobs.push_back(zero_job(f.dtp, ED, Rp - R, R));
        }
        run_casts(jobs, w);
        return f;
    }

    mpa_decode_layer desc(int64_t batch) const {
        mpa_decode_layer s{};
        s.batch = batch; s.d_model = d; s.dim = ED; s.dstate = N; s.dt_rank = R;
        s.d_conv = (int)K;
        s.io_dtype = dt == at::kFloat ? MPA_F32 : MPA_BF16;
        s.in_weight = p[kInW].data; s.in_bias = p[kInB].data;
        s.conv_weight = fptr(conv_w.t); s.conv_bias = fptr(conv_b.t);
        s.x_weight = p[kXW].data; s.dt_weight = p[kDtW].data;
        s.dt_bias = fptr(dt_b.t); s.A = fptr(A); s.D = fptr(D.t);
        s.out_weight = p[kOutW].data; s.out_bias = p[kOutB].data;
        return s;
    }
};

// The norm in front of a mixer.
struct NormHandle {
    bool usable = false, ok = false, changed = false;
    Ref modules;
    Sub norm;
    Param p;
    double eps = 0;
    F32 w;
    uint64_t formed = 0;  // epoch of the mixer's handle that w is of
    Written written;

    NormHandle(const py::object& block, const py::object& norm_type) {
        PyObject* bm = get(dict_of(block.ptr()), keys().modules);
        modules = Ref(bm);
        if (!bm || !norm.open(bm, "norm", norm_type.ptr(), false)) return;
        eps = py::reinterpret_borrow<py::object>(norm.mod.o).attr("eps").cast<double>();
        p = Param{norm.params.o, keys().weight};
        usable = true;
    }
    bool belongs_to(PyObject* dict) const { return !usable || get(dict, keys().modules) == modules.o; }
    bool ready(const MixerHandle& m) {
        if (!usable || !norm.same(modules.o)) return false;
        changed |= p.changed();
        const Tensor& t = p.t;
        return !t.defined() || (t.numel() == m.d && MixerHandle::small_ok(t, m.device) && reinterpret_cast<uintptr_t>(p.data) % 16 == 0);
    }
    void form(const MixerHandle& m) {
        const c10::Stream s = current_stream(m.device);
        written.before(s);
        const bool old = changed || formed != m.epoch;
        if (old) {
            std::vector<mpa_cast_job> jobs;
            w.take(p.t, jobs);
            run_casts(jobs, m.p[kInW].t);
            changed = false;
            formed = capturing() ? 0 : m.epoch;
        }
        written.after(s, old, {&w.own});
    }
};

// The products of a layer run on mpa_linear_run while they are small: it costs the host a quarter of a library call
// (18 us) and takes norms and residual adds along: a bfloat16 stack of width 768 without gradients, 512 steps, 1.4 ms
// for 24 layers, 2.1 with library calls.  The line is steps x width^2, which the products' arithmetic goes with.  Over
// 50 shapes of widths 64 to 968 bfloat16 stacks below it are 1.0 to 1.6 times faster than with library calls, float32
// ones too; at twice the float32 line (1342 steps of width 896, a quarter of the bfloat16 rate) the library's
// large tiles win 1.1 times.  kLinearSteps bounds what was measured.
constexpr int64_t kLinearWorkBf16 = 2048LL * 768 * 768, kLinearWorkF32 = 1024LL * 704 * 704, kLinearSteps = 3072 * 768;
inline bool aligned(const void* p, size_t a) { return reinterpret_cast<uintptr_t>(p) % a == 0; }
inline bool use_linear(at::ScalarType dt, int64_t T, int64_t d, int64_t ED, int64_t P, std::initializer_list<const Tensor*> operands) {
    const bool bf16 = dt == at::kBFloat16;
    if (!bf16 && dt != at::kFloat) return false;
    const int64_t vec = bf16 ? 8 : 4, span = (int64_t)1 << 28;  // (32-bit byte offsets in the kernel)
    bool ok = T * d <= kLinearSteps && T * d * d <= (bf16 ? kLinearWorkBf16 : kLinearWorkF32) && d % vec == 0 && ED % vec == 0 && P % vec == 0 &&
              ED * d < span && ED * P < span && T * std::max(ED, P) < span;
    for (const Tensor* t : operands) ok &= !t->defined() || aligned(t->const_data_ptr(), 16);
    return ok;
}
// out (T x M, rows y_pitch apart) = in (T x K, rows x_pitch apart) . weight^T
inline mpa_linear linear_of(int io, int64_t T, const void* in, int64_t x_pitch, int64_t K, const void* weight, int64_t M, void* out, int64_t y_pitch) {
    mpa_linear q{};
    q.T = T; q.M = M; q.K = K;
    q.x_pitch = x_pitch; q.y_pitch = y_pitch;
    q.x = in; q.weight = weight; q.y = out;
    q.io_dtype = io;
    return q;
}
inline void run_linear(const mpa_linear& q, void* stream) { check(mpa_linear_run(&q, stream), "mpa_linear_run"); }

struct Types {  // the exact Python classes that a handle is made for
    py::object block, norm;
};
inline Types* types = nullptr;  // set by register_types, kept for the interpreter's lifetime

template <typename H>
inline H* handle_in(PyObject* module, const py::object& type) {
    PyObject* dict = dict_of(module);
    if (!dict) return nullptr;
    PyObject* o = get(dict, keys().handle);
    if (!o || o == Py_None || !py::cast<H*>(py::handle(o))->belongs_to(dict)) {
        const py::object h = py::cast(new H(py::reinterpret_borrow<py::object>(module), type), py::return_value_policy::take_ownership);
        PyDict_SetItem(dict, keys().handle, h.ptr());
        o = h.ptr();
    }
    return py::cast<H*>(py::handle(o));
}
inline MixerHandle* mixer_handle(PyObject* mixer) {
    return mixer && types && (PyObject*)Py_TYPE(mixer) == types->block.ptr() ? handle_in<MixerHandle>(mixer, types->block) : nullptr;
}

// A residual block: its norm and its mixer.
struct Layer {
    NormHandle* n = nullptr;
    MixerHandle* m = nullptr;
};
inline bool find_layer(PyObject* block, const Tensor& x, Layer& l) {
    PyObject* mods = get(dict_of(block), keys().modules);
    l.m = mixer_handle(get(mods, keys().mixer));
    if (!l.m || !l.m->ready(x)) return false;
    l.n = handle_in<NormHandle>(block, types->norm);
    return l.n && l.n->ready(*l.m);
}

// Whether the calls a native path replaces would be rewritten by autocast.
inline bool autocast_on() { return at::autocast::is_autocast_enabled(at::kCUDA); }

inline bool fits(const Tensor& t, at::IntArrayRef shape, at::ScalarType dt, const c10::Device& dev) {
    return t.scalar_type() == dt && t.device() == dev && t.sizes() == shape && t.is_contiguous() &&
           reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
}

}  // namespace mpa_host
