// A residual block or mixer of the package as C++ sees it: which parameters it has, whether it is of the
// plain kind, and the forms of its weights that the kernels take.
//
// What is made from a layer's parameters is kept in handles, a MixerHandle in the mixer's __dict__ and a NormHandle
// in the residual block's.  Nothing about the modules is: every call looks whether the submodules are of the plain
// types and nothing (a hook, a method put on an instance or a class, autocast) wants to see the calls that are skipped,
// and takes the parameters from where they are.  A block that fails is run module by module in Python.
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
    PyObject *modules = key("_modules"), *params = key("_parameters"), *handle = key("_mpa_handle"), *config = key("config"),
             *mixer = key("mixer"), *norm = key("norm"), *weight = key("weight"), *bias = key("bias"), *A_log = key("A_log"), *D = key("D"),
             *in_proj = key("in_proj"), *conv1d = key("conv1d"), *x_proj = key("x_proj"), *dt_proj = key("dt_proj"), *out_proj = key("out_proj"),
             *dt_layernorm = key("dt_layernorm"), *eps = key("eps"), *use_mup = key("use_mup");
    PyObject* const hooks[4] = {key("_forward_hooks"), key("_forward_pre_hooks"), key("_backward_hooks"), key("_backward_pre_hooks")};
    PyObject* const sizes[7] = {key("d_model"), key("d_inner"), key("d_state"), key("dt_rank"), key("d_conv"), key("inner_layernorms"),
                                key("fused_softplus")};
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
// A number that no two states of any dictionaries share (PEP 509); where Python has none, never the same twice.
inline uint64_t state_of(PyObject* dict) {
#if PY_VERSION_HEX < 0x030C0000
    return reinterpret_cast<PyDictObject*>(dict)->ma_version_tag;
#else
    static uint64_t n = 0;
    return ++n;
#endif
}

inline bool empty_dict(PyObject* o) { return o && PyDict_Check(o) && PyDict_Size(o) == 0; }

// The exact Python classes that handles are made for, the methods of theirs that a native call stands in for, and
// torch's hooks on all modules.
struct Types {
    struct Method {
        Ref dict, name, was;  // the class's __dict__, and what was under the name
    };
    py::object block, norm, linear, conv;
    std::vector<Method> methods;
    std::vector<Ref> block_names, norm_names, linear_names;  // not to be found on an instance
    std::vector<Ref> global_hooks;
    bool plain() const {
        for (const Method& m : methods)
            if (get(m.dict.o, m.name.o) != m.was.o) return false;
        for (const Ref& h : global_hooks)
            if (!empty_dict(h.o)) return false;
        return true;
    }
};
inline Types* types = nullptr;  // set by register_types, kept for the interpreter's lifetime

// A module's instance dictionary, looked through again when it has changed (fifteen look-ups; a layer has seven).
struct Instance {
    uint64_t state = 0, params_state = 0;
    PyObject *params = nullptr, *hooks[4] = {};
    PyObject* pair[2] = {};  // what its _parameters hold under two names, in params_state
    // nothing on the module itself changes or watches its calls
    bool plain(PyObject* dict, const std::vector<Ref>& names) {
        if (!dict) return false;
        if (state_of(dict) != state) {
            state = 0;
            for (const Ref& n : names)
                if (get(dict, n.o)) return false;
            for (int i = 0; i < 4; ++i) hooks[i] = get(dict, keys().hooks[i]);
            params = get(dict, keys().params);
            if (!params || !PyDict_Check(params)) return false;
            state = state_of(dict);
        }
        for (PyObject* h : hooks)
            if (!empty_dict(h)) return false;
        return true;
    }
    void find(PyObject* first, PyObject* second) {  // (always the same two)
        if (state_of(params) == params_state) return;
        pair[0] = get(params, first);
        pair[1] = get(params, second);
        params_state = state_of(params);
    }
    // the instance dictionary of the plain submodule under `name`, or null
    PyObject* sub(PyObject* modules, PyObject* name, const py::object& type, const std::vector<Ref>& names) {
        PyObject* m = get(modules, name);
        if (!m || (PyObject*)Py_TYPE(m) != type.ptr()) return nullptr;
        PyObject* d = dict_of(m);
        return plain(d, names) ? d : nullptr;
    }
};

// The state a parameter was last seen in.  The tensor is not held beyond a call, not even weakly: a model that moves away
// takes its memory along, and its tensors can be swapped.  What tells another tensor at the same addresses from the old
// one is the old one's version counter, which is held: a tensor that is gone leaves it to us alone.
struct Param {
    const void* impl = nullptr;
    const void* data = nullptr;
    std::optional<c10::VariableVersion> counter;
    uint32_t version = 0;
    // Takes over what a module's _parameters hold under the name, None for no parameter; false if it is neither that nor a
    // plain tensor (pruning and parametrisation take the name away).  An inference tensor has no version counter and may
    // always have changed.
    bool take(PyObject* o, Tensor& now, bool& changed) {
        if (o == Py_None) {
            changed |= impl != nullptr;
            *this = Param{};
            return true;
        }
        if (!o || !THPVariable_CheckExact(o)) return false;
        now = THPVariable_Unpack(o);
        if (wrapped(now)) return false;
        const c10::TensorImpl* im = now.unsafeGetTensorImpl();
        const bool counted = !now.is_inference();
        if (counted && im == impl && counter && !counter->unique() && now.const_data_ptr() == data && now._version() == version) return true;
        changed = true;
        impl = im;
        data = now.const_data_ptr();
        counter.reset();
        if (counted) counter.emplace(im->version_counter());
        version = counted ? now._version() : 0;
        return true;
    }
};

enum { kInW, kInB, kConvW, kConvB, kXW, kXB, kDtW, kDtB, kALog, kD, kOutW, kOutB, kParams };

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
    Tensor own;
    Tensor form(const Tensor& p, bool old, std::vector<mpa_cast_job>& jobs) {
        if (!p.defined() || p.scalar_type() == at::kFloat) return p;
        derived(own, p.sizes(), at::kFloat, p);
        if (old) jobs.push_back(row_job(p, own));
        return own;
    }
};

inline c10::Stream current_stream(const c10::Device& device) { return c10::impl::VirtualGuardImpl(device.type()).getStream(device); }
inline bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }

// Orders the streams that read kept forms after the one that last wrote them, and tells the allocator of them.
// (A capture cannot wait for an event from outside; torch synchronises the device before it begins one.)
struct Written {
    std::shared_ptr<c10::Event> event;
    std::optional<c10::Stream> last;  // the stream that wrote, or one that has waited since
    bool unordered = false;           // written by a call that failed before its event
};
// The forming of the layers of one call: one event for all that is written, recorded by done().
class Forming {
public:
    explicit Forming(const c10::Device& device) : stream(current_stream(device)), capture(capturing()) {}
    Forming(const Forming&) = delete;
    ~Forming() {
        for (Written* w : wrote) w->unordered = true;
    }
    void done() {
        if (wrote.empty()) return;
        const auto event = std::make_shared<c10::Event>(stream.device_type());
        event->record(stream);
        for (Written* w : wrote) w->event = event;
        wrote.clear();
    }
    void before(const Written& w) const {
        if (w.event && w.last != stream && !capture) w.event->block(stream);
    }
    void after(Written& w, bool wrote_it, std::initializer_list<const Tensor*> forms) {
        if (w.last && w.last != stream)
            for (const Tensor* t : forms)
                if (t->defined()) t->record_stream(stream);
        if (capture) return;
        w.last = stream;
        if (wrote_it) wrote.push_back(&w);
    }
    const c10::Stream stream;
    const bool capture;

private:
    std::vector<Written*> wrote;
};

struct LayerSizes {
    int64_t d = 0, ED = 0, N = 0, R = 0, K = 0, Rp = 0;
    at::ScalarType dt = at::kFloat;
    c10::Device device{at::kCPU};
    int64_t padded_rows() const { return Rp == R ? R + 2 * N : (Rp + 2 * N + 63) / 64 * 64; }
};

// The parameters of a mixer and the forms of them that the kernels take.  A call takes one along when it lets go of the
// interpreter: handles change under the interpreter's lock, these not at all.
struct Weights : LayerSizes {
    Tensor p[kParams];
    Tensor conv_w, conv_b, dt_b, D;              // float32
    Tensor A;                        // -exp(A_log), float32
    Tensor xp, dtp;                  // x_proj and dt_proj, padded

    // x_proj and dt_proj in the shape the GEMM library serves best: the low-rank width R is the K of
    // dt_proj and R + 2N the rows of x_proj, both odd for its tiles (48 and 80 at width 768).  With R
    // rounded up to a multiple of 64 by zeros and the rows regrouped as [delta | 0 | B | C | 0], the two
    // products take 21 + 26 us instead of 25 + 38 us at 32768 rows in bfloat16.
    void pad_jobs(std::vector<mpa_cast_job>& jobs) const {
        const Tensor &xw = p[kXW], &dw = p[kDtW];
        jobs.push_back(cast_job(xw, xp, R, ED));
        jobs.push_back(cast_job(xw, xp, 2 * N, ED, R * ED, Rp * ED));
        jobs.push_back(cast_job(dw, dtp, ED, R));
    }

    // What a call with gradients takes in place of the kept forms: made in the call, on its stream, from the parameters
    // as they are, and held by its graph node; one launch.
    void form_for_training() {
        const Tensor& w = p[kInW];
        std::vector<mpa_cast_job> jobs;
        auto f32 = [&](const Tensor& q) {
            if (!q.defined() || q.scalar_type() == at::kFloat) return q;
            const Tensor t = empty(q.sizes(), at::kFloat, q);
            jobs.push_back(row_job(q, t));
            return t;
        };
        conv_w = f32(p[kConvW]);
        conv_b = f32(p[kConvB]);
        dt_b = f32(p[kDtB]);
        D = f32(p[kD]);
        A = empty({ED, N}, at::kFloat, w);
        jobs.push_back(cast_job(p[kALog], A, ED, N, 0, 0, MPA_CAST_NEG_EXP));
        if (Rp == R) {
            xp = p[kXW].detach();
            dtp = p[kDtW].detach();
        } else {
            const int64_t rows = padded_rows(), used = Rp + 2 * N;
            xp = empty({rows, ED}, dt, w);
            dtp = empty({ED, Rp}, dt, w);
            pad_jobs(jobs);
            jobs.push_back(zero_job(xp, Rp - R, ED, R * ED));
            if (rows > used) jobs.push_back(zero_job(xp, rows - used, ED, used * ED));
            jobs.push_back(zero_job(dtp, ED, Rp - R, R));
        }
        run_casts(jobs, w);
    }

    mpa_decode_layer desc(int64_t batch) const {
        mpa_decode_layer s{};
        s.batch = batch; s.d_model = d; s.dim = ED; s.dstate = N; s.dt_rank = R;
        s.d_conv = (int)K;
        s.io_dtype = dt == at::kFloat ? MPA_F32 : MPA_BF16;
        s.in_weight = ptr(p[kInW]); s.in_bias = ptr(p[kInB]);
        s.conv_weight = fptr(conv_w); s.conv_bias = fptr(conv_b);
        s.x_weight = ptr(p[kXW]); s.dt_weight = ptr(p[kDtW]);
        s.dt_bias = fptr(dt_b); s.A = fptr(A); s.D = fptr(D);
        s.out_weight = ptr(p[kOutW]); s.out_bias = ptr(p[kOutB]);
        return s;
    }
};

// (no two handles are ever at the same one)
inline uint64_t next_epoch() {
    static uint64_t last = 0;
    return ++last;
}

struct NormHandle;
struct MixerHandle : LayerSizes {
    bool decode_ok = false;   // the shapes are such as mpa_decode_layer_step takes
    bool forward_ok = false;  // ... as stack_forward and block_train take
    Ref modules;
    Instance self, in_proj, conv1d, x_proj, dt_proj, out_proj;
    Ref sizes[7];  // values of the config, by Keys::sizes
    uint64_t config_state = 0;
    Param p[kParams];
    bool fused_softplus = true;
    // Forms kept for calls without gradients, and the epoch they are of.  Version counters do not show every change
    // of a parameter (writes through .data), and a training loop makes one after each of its calls: a call with
    // gradients forms its own and begins an epoch.
    uint64_t epoch = next_epoch(), formed = 0, padded = 0;  // padded: that of xp and dtp
    Written written;
    F32 conv_w, conv_b, dt_b, D;
    Tensor A, xp, dtp;  // (xp and dtp: where the layer's own shapes are padded)

    explicit MixerHandle(PyObject* dict) : modules(get(dict, keys().modules)) {}
    // the dictionaries are those of this block (a shallow copy brings the handle of its original along)
    bool belongs_to(PyObject* dict) const { return get(dict, keys().modules) == modules.o; }

    // Whether the block with this __dict__ can run here with activations like x; its sizes and parameters.
    bool ready(PyObject* dict, const Tensor& x, Weights& w) {
        const Keys& k = keys();
        if (!self.plain(dict, types->block_names) || get(dict, k.dt_layernorm) != Py_None) return false;
        PyObject* mm = modules.o;
        if (!in_proj.sub(mm, k.in_proj, types->linear, types->linear_names) || !conv1d.sub(mm, k.conv1d, types->conv, types->linear_names) ||
            !x_proj.sub(mm, k.x_proj, types->linear, types->linear_names) || !dt_proj.sub(mm, k.dt_proj, types->linear, types->linear_names) ||
            !out_proj.sub(mm, k.out_proj, types->linear, types->linear_names))
            return false;
        bool changed = false;
        if (!read_config(get(dict, k.config), changed)) return false;
        auto take = [&](Instance& m, int i, PyObject* name_i, int j, PyObject* name_j) {
            m.find(name_i, name_j);
            return p[i].take(m.pair[0], w.p[i], changed) && p[j].take(m.pair[1], w.p[j], changed);
        };
        const bool there = take(in_proj, kInW, k.weight, kInB, k.bias) && take(conv1d, kConvW, k.weight, kConvB, k.bias) &&
                           take(x_proj, kXW, k.weight, kXB, k.bias) && take(dt_proj, kDtW, k.weight, kDtB, k.bias) &&
                           take(out_proj, kOutW, k.weight, kOutB, k.bias) && take(self, kALog, k.A_log, kD, k.D);
        if (changed) epoch = next_epoch();
        if (changed && !there) forget();
        decode_ok = forward_ok = false;
        if (there) look_over(w);
        static_cast<LayerSizes&>(w) = *this;
        return (decode_ok || forward_ok) && x.scalar_type() == dt && x.device() == device && x.size(-1) == d;
    }
    // (what has been taken over before a parameter was found missing is looked over again once it is back)
    void forget() {
        for (Param& q : p) q = Param{};
    }
    bool read_config(PyObject* config, bool& changed) {
        PyObject* dict = config ? dict_of(config) : nullptr;
        if (!dict) return false;
        const uint64_t state = state_of(dict);
        if (state == config_state) return PyObject_IsTrue(sizes[5].o) == 0;
        config_state = 0;
        PyObject* v[7];
        bool same = true;
        for (int i = 0; i < 7; ++i) {
            v[i] = get(dict, keys().sizes[i]);
            if (!v[i] || (i < 5 && !PyLong_Check(v[i]))) return false;
            same &= v[i] == sizes[i].o;
        }
        if (!same) {
            changed = true;
            int64_t* const to[] = {&d, &ED, &N, &R, &K};
            for (int i = 0; i < 5; ++i) *to[i] = PyLong_AsLongLong(v[i]);
            for (int i = 0; i < 7; ++i) sizes[i] = Ref(v[i]);
            Rp = (R + 63) / 64 * 64;
            fused_softplus = PyObject_IsTrue(sizes[6].o) == 1;
            xp = dtp = Tensor();  // (their zeros are elsewhere)
        }
        config_state = state;
        return PyObject_IsTrue(sizes[5].o) == 0;
    }

    void expire() { epoch = next_epoch(); }

    void look_over(const Weights& all) {
        const Tensor* const t = all.p;
        const Tensor& w = t[kInW];
        if (d <= 0 || R <= 0 || N <= 0 || !w.defined() || !w.is_cuda() || (w.scalar_type() != at::kFloat && w.scalar_type() != at::kBFloat16)) return;
        dt = w.scalar_type();
        device = w.device();
        for (int i : {kInW, kXW, kDtW, kOutW, kInB, kOutB}) {
            const Tensor& v = t[i];
            const bool optional = i == kInB || i == kOutB;
            if (!v.defined() && optional) continue;
            if (!v.defined() || v.scalar_type() != dt || v.device() != device || !v.is_contiguous()) return;
        }
        for (int i : {kConvW, kConvB, kDtB, kALog, kD})
            if (t[i].defined() && !small_ok(t[i], device)) return;
        if (!t[kConvW].defined() || !t[kALog].defined() || !t[kD].defined() || t[kXB].defined()) return;
        if (t[kInW].sizes() != at::IntArrayRef({2 * ED, d}) || t[kXW].sizes() != at::IntArrayRef({R + 2 * N, ED}) ||
            t[kDtW].sizes() != at::IntArrayRef({ED, R}) || t[kOutW].sizes() != at::IntArrayRef({d, ED}) ||
            t[kConvW].numel() != ED * K || t[kALog].sizes() != at::IntArrayRef({ED, N}) || t[kD].numel() != ED)
            return;
        for (const auto& [i, n] : {std::pair<int, int64_t>{kInB, 2 * ED}, {kConvB, ED}, {kDtB, ED}, {kOutB, d}})
            if (t[i].defined() && t[i].numel() != n) return;
        const int64_t vec = dt == at::kFloat ? 4 : 8;
        decode_ok = K >= 2 && K <= 4 && d % vec == 0 && ED % vec == 0 && N % 4 == 0 && N <= MPA_MAX_DSTATE && R <= 2048;
        for (int i : {kInW, kXW, kOutW}) decode_ok &= reinterpret_cast<uintptr_t>(p[i].data) % 16 == 0;
        forward_ok = K >= 2 && K <= 4 && N <= MPA_MAX_DSTATE && fused_softplus && d % vec == 0 && d <= 512 * vec && t[kDtB].defined();
    }
    static bool small_ok(const Tensor& t, const c10::Device& device) {
        return t.device() == device && t.is_contiguous() && (t.scalar_type() == at::kFloat || t.scalar_type() == at::kBFloat16);
    }

    // Fills w, as ready() left it, with the kept forms, up to date: xp and dtp among them for a sequence; and norm_w, as the norm
    // in front left it, if there is one.  Within a capture nothing runs yet: the next call still finds them old.
    void form(Forming& f, bool sequence, Weights& w, NormHandle* norm, Tensor* norm_w);
};

// The norm in front of a mixer.
struct NormHandle {
    bool changed = false;
    Instance norm;
    Ref modules, eps_seen;
    Param p;
    double eps = 0;
    F32 w;
    uint64_t formed = 0;  // epoch of the mixer's handle that w is of (the mixer's `written` covers it)

    explicit NormHandle(PyObject* dict) : modules(get(dict, keys().modules)) {}
    bool belongs_to(PyObject* dict) const { return get(dict, keys().modules) == modules.o; }
    bool ready(const MixerHandle& m, Tensor& t) {  // t: the norm's weight
        const Keys& k = keys();
        PyObject* const d = norm.sub(modules.o, k.norm, types->norm, types->norm_names);
        if (!d) return false;
        PyObject *const e = get(d, k.eps), *const gainless = get(d, k.use_mup);
        if (!e || !gainless) return false;
        if (e != eps_seen.o) {
            eps_seen = Ref(e);
            eps = py::handle(e).cast<double>();
        }
        if (PyObject_IsTrue(gainless) == 1) {
            changed |= p.impl != nullptr;
            p = Param{};
        } else if (norm.find(k.weight, k.bias); !p.take(norm.pair[0], t, changed)) {
            return false;
        }
        return !t.defined() || (t.numel() == m.d && MixerHandle::small_ok(t, m.device) && reinterpret_cast<uintptr_t>(p.data) % 16 == 0);
    }
};

inline void MixerHandle::form(Forming& f, bool sequence, Weights& w, NormHandle* norm, Tensor* norm_w) {
    f.before(written);
    if (written.unordered) expire();
    written.unordered = false;
    const bool small = formed != epoch, wide = sequence && padded != epoch, gain = norm && (norm->changed || norm->formed != epoch);
    std::vector<mpa_cast_job> jobs;
    if (norm) *norm_w = norm->w.form(*norm_w, gain, jobs);
    w.conv_w = conv_w.form(w.p[kConvW], small, jobs);
    w.conv_b = conv_b.form(w.p[kConvB], small, jobs);
    w.dt_b = dt_b.form(w.p[kDtB], small, jobs);
    w.D = D.form(w.p[kD], small, jobs);
    w.A = derived(A, {ED, N}, at::kFloat, w.p[kInW]);
    if (small) jobs.push_back(cast_job(w.p[kALog], A, ED, N, 0, 0, MPA_CAST_NEG_EXP));
    if (sequence) {
        const Tensor &xw = w.p[kXW], &dw = w.p[kDtW];
        w.xp = Rp == R ? xw : derived(xp, {padded_rows(), ED}, dt, xw);
        w.dtp = Rp == R ? dw : derived(dtp, {ED, Rp}, dt, dw);
        if (wide && Rp != R) w.pad_jobs(jobs);
    }
    run_casts(jobs, w.p[kInW]);
    const uint64_t of = f.capture ? 0 : epoch;
    if (gain) {
        norm->changed = f.capture;
        norm->formed = of;
    }
    if (small) formed = of;
    if (wide) padded = of;
    f.after(written, !jobs.empty(), {&conv_w.own, &conv_b.own, &dt_b.own, &D.own, &A, &xp, &dtp, norm ? &norm->w.own : &A});
}

// The products of a layer run on mpa_linear_run while they are small: it costs the host a quarter of a library call
// (18 us) and takes norms and residual adds along.  The line is steps x width^2, which the products' arithmetic goes with.
// Measured against library calls at 173 shapes of widths 64 to 2560 and 16 to 73728 steps (a layer of a stack without
// gradients; a mixer, forward and backward), times as fast:
//   bfloat16  below the line 0.96 to 2.0 and 0.99 to 1.7 (0.96 to 1.1 at the line itself), at twice the line 0.84 to 1.1
//   float32   a quarter of the rate, and every stage of a long K a latency.  Without gradients the line is that of width
//             704 up to width 512 and falls as its square from there (0.98 to 2.1; on the other side of it 0.72 to 1.2).  A mixer
//             with gradients makes three times the calls: 0.85 of the line up to width 1536 (1.00 to 1.9; on the other side 0.83 to 1.1).
// kLinearSteps bounds what was measured.
constexpr int64_t kLinearWorkBf16 = 2048LL * 768 * 768, kLinearWorkF32 = 1024LL * 704 * 704, kLinearSteps = 3072 * 768;
inline bool aligned(const void* p, size_t a) { return reinterpret_cast<uintptr_t>(p) % a == 0; }
inline bool below_line(bool bf16, bool training, int64_t T, int64_t d) {
    const int64_t work = T * d * d;
    if (bf16) return work <= kLinearWorkBf16;
    if (training) return work <= kLinearWorkF32 * 17 / 20 && d <= 1536;
    return work <= kLinearWorkF32 && (d <= 512 || work <= kLinearWorkF32 * 512 / d * 512 / d);
}
inline bool use_linear(at::ScalarType dt, bool training, int64_t T, int64_t d, int64_t ED, int64_t P, std::initializer_list<const Tensor*> operands) {
    const bool bf16 = dt == at::kBFloat16;
    if (!bf16 && dt != at::kFloat) return false;
    const int64_t vec = bf16 ? 8 : 4, span = (int64_t)1 << 28;  // (32-bit byte offsets in the kernel)
    bool ok = T * d <= kLinearSteps && below_line(bf16, training, T, d) && d % vec == 0 && ED % vec == 0 && P % vec == 0 &&
              ED * d < span && ED * P < span && T * std::max(ED, P) < span;
    for (const Tensor* t : operands) ok &= !t->defined() || aligned(t->const_data_ptr(), 16);
    return ok;
}
// The convolution of a mixer and x_proj of its output in one launch; false: not a case for it (mpa_conv1d_proj_fwd: bfloat16, four taps,
// up to 96 rows of x_proj, which is any rank up to 64 with up to 16 states).  Up to 24 * 2^20 activations: their 50 MB and the
// 100 MB they are read from are then in the last-level cache still when the kernel comes to them.  From memory it has too few
// loads in flight: in a forward pass of 8 x 3000 steps of width 768 it took 61 us where convolution and library product took 57; of
// 8 x 1000 steps 19 and 27.  (Buffers written just before, other memory between: 8 x 2000 x 1536 35 and 44 us, 8 x 2500 x 1536 53 and 51.)
constexpr int64_t kConvProjWork = 24LL << 20;
inline bool conv_proj(const mpa_conv_shape& s, const Weights& l, const void* x, const void* window, void* y, void* window_out, void* out, int64_t P,
                      void* stream) {
    const int64_t used = l.Rp + 2 * l.N;
    if (s.batch * s.seqlen * s.dim > kConvProjWork || !mpa_conv1d_proj_suits(&s, used) || !aligned(l.xp.const_data_ptr(), 16)) return false;
    check(mpa_conv1d_proj_fwd(&s, x, fptr(l.conv_w), fptr(l.conv_b), window, y, window_out, ptr(l.xp), used, out, P, P, stream),
          "mpa_conv1d_proj_fwd");
    return true;
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

// The wide float32 products of a layer on cut operands (mpa_split_run, mpa_split_product), where a product is long enough to pay
// for cutting its operands.  Measured against library products, widths 256 to 2560 and 128 to 32768 steps, each
// with the cutting of both operands: one product is 0.6 to 1.4 times as fast below 2.5 * 2^30 multiplications, 1.0 to 2.0 just
// above, 1.2 to 2.4 at 8 and 1.9 to 2.5 at 16 times 2^30.  A value is cut once and multiplied as often as the other operand has rows:
// with few steps against a wide weight cutting it is what costs, and below 300 (half the harmonic mean of T and M) one product of 2.5 to
// 5 * 2^30 is 0.6 to 1.0 times as fast (160 / 256 / 288 steps of width 2048 0.60 / 0.91 / 0.98, 352 1.22; 284 of 1536 0.86, 352 1.4; a
// stack of two layers, 160 / 284 steps of width 2048, without gradients 318 / 386 us with it and 237 / 348, at 320 steps 393 and 376, with
// gradients 1199 and 1230).
// The input gradient and both weight gradients together, one cutting for three products of which the library's weight
// gradients are its slowest: 1.04 to 2.1 from 2^31 for the input gradient on, 1.2 to 2.2 at four times that.
// (Time alone would take lower lines: 3 * 2^28 where both operands have 700 rows or more, 2^30 for three, 1.0 to 2.0 times as fast.  But a cut value is
// 2^-23 of itself, and operands that a float32 sum keeps whole, as a weight of ones and zeros does, come out 2^-24 off.)
constexpr int64_t kSplitOne = 5LL << 29, kSplitThree = 1LL << 31, kSplitRows = 300;
inline bool split_ok(at::ScalarType dt, int64_t T, int64_t M, int64_t K, std::initializer_list<const Tensor*> operands) {
    bool ok = dt == at::kFloat && T < 1 << 24 && M % 4 == 0 && K % 4 == 0;
    for (const Tensor* t : operands) ok &= !t->defined() || aligned(t->const_data_ptr(), 16);
    return ok;
}
inline bool use_split(at::ScalarType dt, int64_t T, int64_t M, int64_t K, std::initializer_list<const Tensor*> operands) {
    return T * M * K >= kSplitOne && T * M >= kSplitRows * (T + M) && split_ok(dt, T, M, K, operands);
}
inline bool use_split_three(at::ScalarType dt, int64_t T, int64_t M, int64_t K, std::initializer_list<const Tensor*> operands) {
    return T * M * K >= kSplitThree && split_ok(dt, T, M, K, operands);
}
// Operands of one launch; `hold` keeps their cut forms until the launches that read them are enqueued.
class Split {
public:
    Split(const Tensor& like, void* stream) : like_(like), stream_(stream) {}
    // element (row, i) at src[row * pitch + i], or by columns at src[i * pitch + row]
    int rows(const void* src, int64_t rows, int64_t k, int64_t pitch) { return add(src, rows, k, pitch, 0); }
    int cols(const void* src, int64_t rows, int64_t k, int64_t pitch) { return add(src, rows, k, pitch, 1); }
    void run() {
        for (mpa_split_operand& o : ops_) {
            if (o.split) continue;
            hold_.push_back(scratch(mpa_split_bytes(o.rows, o.k), like_));
            o.split = ptr(hold_.back());
        }
        check(mpa_split_run(ops_.data() + done_, (int)ops_.size() - done_, stream_), "mpa_split_run");
        done_ = (int)ops_.size();
    }
    // y (x's rows times w's rows)
    void product(int w, int x, const Tensor& bias, void* y, int64_t y_pitch) {
        jobs_.push_back(mpa_split_job{ops_[w], ops_[x], fptr(bias), static_cast<float*>(y), y_pitch});
    }
    void run_products() {
        const int n = (int)jobs_.size();
        const size_t nbytes = n ? mpa_split_product_workspace_bytes(jobs_.data(), n) : 0;
        const Tensor ws = scratch(nbytes, like_);
        if (n) check(mpa_split_product(jobs_.data(), n, ptr(ws), nbytes, stream_), "mpa_split_product");
        jobs_.clear();
    }

private:
    int add(const void* src, int64_t rows, int64_t k, int64_t pitch, int by_cols) {
        ops_.push_back(mpa_split_operand{static_cast<const float*>(src), rows, k, pitch, by_cols, 0, nullptr});
        return (int)ops_.size() - 1;
    }
    const Tensor& like_;
    void* const stream_;
    std::vector<mpa_split_operand> ops_;
    std::vector<mpa_split_job> jobs_;
    std::vector<Tensor> hold_;
    int done_ = 0;
};
// y = x . weight^T (+ bias) on cut operands; false: not a product for them
inline bool split_product(const Tensor& x, const Tensor& weight, const Tensor& bias, const Tensor& y, void* stream) {
    const int64_t M = weight.size(0), K = weight.size(1), T = x.numel() / K;
    if (!use_split(x.scalar_type(), T, M, K, {&x, &weight, &bias})) return false;
    Split s(x, stream);
    const int w = s.rows(ptr(weight), M, K, K), r = s.rows(ptr(x), T, K, K);
    s.run();
    s.product(w, r, bias, ptr(y), M);
    s.run_products();
    return true;
}

// y = x . weight^T, or x . weight (kxm), of matrices with dense rows.
inline void mm_into(const Tensor& y, const Tensor& x, const Tensor& weight, bool kxm, void* stream) {
    const mpa_gemm g{ptr(x), ptr(weight), ptr(y), x.size(0), y.size(1), x.size(1), x.stride(0), weight.stride(0), y.stride(0), kxm};
    if (x.scalar_type() == at::kBFloat16 && x.stride(1) == 1 && weight.stride(1) == 1 && mpa_gemm_faster(&g)) {
        check(mpa_gemm_run(&g, stream), "mpa_gemm_run");
    } else {
        Tensor out = y;
        at::mm_out(out, x, kxm ? weight : weight.t());
    }
}

template <typename H>
inline H* handle_in(PyObject* dict) {
    PyObject* o = get(dict, keys().handle);
    if (o && o != Py_None) {
        H* h = py::cast<H*>(py::handle(o));
        if (h->belongs_to(dict)) return h;
    }
    const py::object h = py::cast(new H(dict), py::return_value_policy::take_ownership);
    PyDict_SetItem(dict, keys().handle, h.ptr());
    return py::cast<H*>(h);
}

// The handle of a mixer that can run here and what it has of parameters, or null.
inline MixerHandle* ready_mixer(PyObject* mixer, const Tensor& x, Weights& w) {
    if (!mixer || (PyObject*)Py_TYPE(mixer) != types->block.ptr()) return nullptr;
    PyObject* dict = dict_of(mixer);
    MixerHandle* m = dict ? handle_in<MixerHandle>(dict) : nullptr;
    return m && m->ready(dict, x, w) ? m : nullptr;
}

// A residual block: its norm and its mixer, and what a call takes along of them.
struct Layer {
    NormHandle* n = nullptr;
    MixerHandle* m = nullptr;
    Weights w;
    Tensor norm_w;
    double eps = 0;
};
inline bool find_layer(PyObject* block, const Tensor& x, Layer& l) {
    PyObject* dict = dict_of(block);
    l.m = ready_mixer(get(get(dict, keys().modules), keys().mixer), x, l.w);
    if (!l.m) return false;
    l.n = handle_in<NormHandle>(dict);
    if (!l.n->ready(*l.m, l.norm_w)) return false;
    l.eps = l.n->eps;
    return true;
}

// Whether a native call may run at all: nothing replaces or rewrites the calls it stands in for (autocast does), and x is
// an ordinary tensor without a tangent.
inline bool native_call(const Tensor& x) {
    return types && types->plain() && !at::autocast::is_autocast_enabled(at::kCUDA) && !forward_mode() && x.is_cuda() && !wrapped(x);
}

inline bool fits(const Tensor& t, at::IntArrayRef shape, at::ScalarType dt, const c10::Device& dev) {
    return t.scalar_type() == dt && t.device() == dev && t.sizes() == shape && t.is_contiguous() &&
           reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
}

}  // namespace mpa_host
