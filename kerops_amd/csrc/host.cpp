// Native call path of the ops: everything an op's Python function does for its common call (checks of the arguments, live
// launch shapes, outputs, scratch memory, the library call), in one C++ call.  A small volume's kernel runs for 2 to 5 us, the
// Python function of its op took 8 to 19 us, so short calls waited for Python.  Host time per call in us, Python / here (a
// launch is 2.6 of it, and ops with a reduction launch twice): DWConv 8.8 / 4.9, DWConvStats 14.2 / 9.6, DWConvBackward 15.0 /
// 9.1, Stats 14.7 / 8.6, AddStats 17.2 / 10.0, AddStatsBackward 11.2 / 5.5, ApplyBNReLUBackward 17.8 / 10.2, AvgPoolCeilStats
// 18.4 / 9.2, ReLULinearAdd 8.3 / 4.5, ReLULinearBackward 15.4 / 8.5, DWSepBlockInt8 27.0 / 15.1, QuantUint8Window 8.7 / 4.9.
//
// The Python functions stay what defines an op.  A function here takes a call only if nothing about it is unusual and
// returns None otherwise, whereupon the caller goes on with the Python function: wrong shapes, types or devices (it
// raises the op's own error), copies (a weight that is not contiguous), tensor subclasses, torch function and dispatch
// modes, tracing, vmap, tensors of another than the current device, knobs passed by keyword, a replaced function, configurator
// or module-level name that the Python function of the call would read (`watch`).  Launch tables are read on every call.
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <ATen/ops/empty_strided.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <array>
#include <climits>
#include <initializer_list>
#include <optional>
#include <utility>
#include <vector>

#include "../../include/kerops_hip.h"

namespace {

using at::Tensor;

// ---- the library's entry points, given by the binding that has loaded it and checked its version ----
#define KEROPS_ENTRIES(X)                                                                                              \
    X(dwconv_fwd_f16) X(dwconv_stats_workspace_bytes) X(dwconv_stats_f16) X(dwconv_bwd_workspace_bytes)                 \
    X(dwconv_bwd_f16_out) X(dwconv_wgrad_workspace_bytes) X(dwconv_wgrad_f16_out) X(stats_workspace_bytes) X(stats_f16) \
    X(stats_bwd_f16) X(add_stats_f16) X(add_stats_bwd_f16) X(bnrelu_fwd_f16) X(bnrelu_bwd_f16)                          \
    X(avgpool_ceil_stats_workspace_bytes) X(avgpool_ceil_stats_f16) X(bnrelu_avgpool_ceil_stats_f16)                    \
    X(avgpool_ceil_stats_bwd_f16) X(quant_u8_window) X(dequant_u8_window) X(quant_i8_sym_f16) X(pointwise_f16)          \
    X(bnrelu_pointwise_f16) X(lin_brelu_lin_add_f16) X(lin_brelu_lin_bwd_workspace_bytes) X(lin_brelu_lin_bwd_f16_out)  \
    X(relu_linear_bwd_workspace_bytes) X(relu_linear_bwd_f16_out) X(bnrelu_linear_bwd_workspace_bytes)                  \
    X(bnrelu_linear_bwd_f16) X(dwsep_block_workspace_bytes) X(dwsep_block_f16)
struct {
#define X(name) decltype(&kerops_##name) name;
    KEROPS_ENTRIES(X)
#undef X
} lib;

// ---- what a call relies on beside its arguments ----
#define KEROPS_OPS(X)                                                                                                  \
    X(DWConv) X(DWConvStats) X(DWConvBackward) X(DWConvWGRAD) X(Stats) X(StatsBackward) X(AddStats) X(AddStatsBackward) \
    X(ApplyBNReLU) X(ApplyBNReLUBackward) X(AvgPoolCeilStats) X(ApplyBNReLUAvgPoolCeilStats) X(AvgPoolCeilStatsBackward) \
    X(ReLULinearAdd) X(ReLULinearBackward) X(ApplyBNReLULinearAdd) X(ApplyBNReLULinearBackward) X(LinBReLULinAdd)        \
    X(LinBReLULinBackward) X(QuantUint8Window) X(DequantUint8Window) X(QuantInt8Sym) X(DWSepBlock)
enum Op {
#define X(name) op_##name,
    KEROPS_OPS(X)
#undef X
    kOps
};

// The entries of one dictionary that have to be what they were.  A dictionary's version (no two states of any dictionaries
// share one) says that nothing was written to it since they were last compared.
struct Watched {
    PyObject* dict;  // nullptr: the op's configurators of the moment
    std::vector<std::pair<PyObject*, PyObject*>> entries;
    uint64_t version = 0;
};
struct Relied {
    PyObject* op_dict = nullptr;  // the ConfiguredFunction's attributes (nullptr: a plain function)
    std::vector<Watched> dicts;
};
std::array<Relied, kOps> relied;
std::array<PyObject*, kOps> op_names;
// module dictionaries whose live entries are launch shapes
PyObject *stream_table, *hardware_conf, *fwd_conf, *wgrad_conf, *lib_module;
PyObject *k_table, *k_small_bytes, *k_small, *k_default, *k_blocks, *k_warps, *k_segment, *k_l1, *k_tile_w, *k_tile_d, *k_lane,
    *k_waves, *k_fwd_variants, *k_wgrad_variants, *k_out_dtype, *k_configurators;

bool as_int(PyObject* o, int64_t& v)
{
    if (!o || !PyLong_CheckExact(o)) return false;
    int overflow = 0;
    v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return !overflow;
}

bool as_knob(PyObject* o, int32_t& v)
{
    int64_t w;
    if (!as_int(o, w) || w < INT_MIN || w > INT_MAX) return false;
    v = (int32_t)w;
    return true;
}

// nothing between this thread and a plain call: no torch function mode, no dispatch mode, tracer or functorch level
bool plain_thread()
{
    using c10::DispatchKey;
    static const uint64_t usual = c10::DispatchKeySet({DispatchKey::BackendSelect, DispatchKey::ADInplaceOrView,
                                                       DispatchKey::AutocastCUDA, DispatchKey::AutocastCPU})
                                      .raw_repr();
    return at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
           (c10::impl::tls_local_dispatch_key_set().included_.raw_repr() & ~usual) == 0;
}

bool as_before(PyObject* dict, Watched& w)
{
#if PY_VERSION_HEX < 0x030C0000
    const uint64_t version = ((PyDictObject*)dict)->ma_version_tag;
    if (version == w.version) return true;
#endif
    for (const auto& [key, value] : w.entries)
        if (PyDict_GetItem(dict, key) != value) return false;
#if PY_VERSION_HEX < 0x030C0000
    w.version = version;
#endif
    return true;
}

bool steady(Op op)
{
    Relied& r = relied[op];
    PyObject* configurators = r.op_dict ? PyDict_GetItem(r.op_dict, k_configurators) : nullptr;
    if (r.op_dict && !(configurators && PyDict_CheckExact(configurators))) return false;
    for (Watched& w : r.dicts)
        if (!as_before(w.dict ? w.dict : configurators, w)) return false;
    return !r.dicts.empty() && plain_thread();
}

// ---- arguments ----
// a torch.Tensor or Parameter (no subclass) that is an ordinary strided tensor on the GPU
const Tensor* gpu_tensor(PyObject* o)
{
    using c10::DispatchKey;
    static const uint64_t usual = c10::DispatchKeySet({DispatchKey::CUDA, DispatchKey::AutogradCUDA, DispatchKey::AutocastCUDA,
                                                       DispatchKey::ADInplaceOrView})
                                      .raw_repr();
    if (!THPVariable_CheckExact(o)) return nullptr;
    const Tensor& t = THPVariable_Unpack(o);
    return (t.key_set().raw_repr() & ~usual) == 0 && t.is_cuda() ? &t : nullptr;
}

struct Where {
    std::optional<c10::hip::HIPStream> stream;  // of the current device (asked only once there is a tensor on the GPU)
    bool holds(std::initializer_list<const Tensor*> ts)
    {
        for (const Tensor* t : ts)
            if (!t) return false;
        stream = c10::hip::getCurrentHIPStream();
        for (const Tensor* t : ts)
            if (t->get_device() != stream->device_index()) return false;
        return true;
    }
    void* handle() const { return (void*)stream->stream(); }
};

bool power_of_2(int64_t n) { return n >= 1 && (n & (n - 1)) == 0; }

struct Volume {  // (N, C, H, W, D), fp16, channels_last_3d
    const Tensor* t = nullptr;
    int64_t c, v;  // channels, voxels
    int32_t n, h, w, d;
    explicit Volume(PyObject* o)
    {
        const Tensor* p = gpu_tensor(o);
        if (!p || p->dim() != 5 || p->scalar_type() != at::kHalf || !p->is_contiguous(at::MemoryFormat::ChannelsLast3d)) return;
        const auto s = p->sizes();
        for (int64_t e : s)
            if (e > INT_MAX) return;
        c = s[1];
        if (c < 1) return;
        v = p->numel() / c;
        n = (int32_t)s[0], h = (int32_t)s[2], w = (int32_t)s[3], d = (int32_t)s[4];
        t = p;
    }
    explicit operator bool() const { return t != nullptr; }
    bool same_space(const Volume& o) const { return n == o.n && h == o.h && w == o.w && d == o.d; }
    bool same_shape(const Volume& o) const { return c == o.c && same_space(o); }
};

bool is_matrix(const Tensor* t, at::IntArrayRef sizes)
{
    return t && t->scalar_type() == at::kHalf && t->sizes() == sizes && t->is_contiguous();
}
bool is_taps(const Tensor* t, int64_t c) { return is_matrix(t, {3, 3, 3, c}); }
bool is_affine(const Tensor* t, int64_t c)
{
    return t && t->scalar_type() == at::kFloat && t->numel() == c && t->is_contiguous();
}
bool built_linear(int64_t c) { return c == 16 || c == 32 || c == 64 || c == 128; }

// keyword arguments: none, or out_dtype = fp16 or fp32
bool out_dtype(PyObject* const* end, PyObject* kw, at::ScalarType& type)
{
    if (!kw) return true;
    if (PyTuple_GET_SIZE(kw) != 1 || PyUnicode_Compare(PyTuple_GET_ITEM(kw, 0), k_out_dtype) != 0 || !THPDtype_Check(end[0]))
        return false;
    type = ((THPDtype*)end[0])->scalar_type;
    return type == at::kHalf || type == at::kFloat;
}

// ---- live launch shapes ----
struct Shape {
    int32_t blocks = 0, warps = 0, segment = 0;
};

// stream_table._find and _common.stream_waves for values that are built
bool stream_shape(Op op, int64_t channels, int64_t bytes, Shape& s)
{
    PyObject* table = PyDict_GetItem(stream_table, k_table);
    int64_t small_bytes;
    if (!table || !PyDict_CheckExact(table) || !as_int(PyDict_GetItem(stream_table, k_small_bytes), small_bytes)) return false;
    PyObject* entry = PyDict_GetItem(table, op_names[op]);
    if (!entry) return true;
    if (!PyDict_CheckExact(entry)) return false;
    PyObject* found = bytes < small_bytes ? PyDict_GetItem(entry, k_small) : nullptr;
    if (!found && channels) {
        PyObject* key = PyUnicode_FromFormat("%lld", (long long)channels);
        if (!key) {
            PyErr_Clear();
            return false;
        }
        found = PyDict_GetItem(entry, key);
        Py_DECREF(key);
    }
    if (!found) found = PyDict_GetItem(entry, k_default);
    if (!found) return true;
    return PyDict_CheckExact(found) && as_knob(PyDict_GetItem(found, k_blocks), s.blocks) &&
           as_knob(PyDict_GetItem(found, k_warps), s.warps) && as_knob(PyDict_GetItem(found, k_segment), s.segment) &&
           (s.warps == 0 || s.warps == 4 || s.warps == 8 || s.warps == 16);
}

// the entry of a per-channel dictionary of a conv module
PyObject* conv_entry(PyObject* module, PyObject* name, PyObject* channels)
{
    PyObject* table = PyDict_GetItem(module, name);
    return table && PyDict_CheckExact(table) ? PyDict_GetItem(table, channels) : nullptr;
}

// (patch W, patch D, kernel family) that the op's configurators give, if the library is built with it
bool conv_shape(PyObject* module, PyObject* variants, int64_t c, bool deep, int32_t& tw, int32_t& td, int32_t& lane)
{
    PyObject* channels = PyLong_FromLongLong(c);
    bool ok = false;
    int64_t waves;
    if (channels && as_int(conv_entry(module, k_waves, channels), waves) && waves > 0 &&
        as_knob(conv_entry(module, k_tile_w, channels), tw) && as_knob(conv_entry(module, k_tile_d, channels), td) &&
        as_knob(conv_entry(module, k_lane, channels), lane)) {
        if (deep) td = 64;
        PyObject* built = conv_entry(module, variants, channels);
        PyObject* shape = built ? Py_BuildValue("(iii)", tw, td, lane) : nullptr;
        ok = shape && power_of_2(td) && PySequence_Contains(built, shape) == 1;
        Py_XDECREF(shape);
    }
    Py_XDECREF(channels);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        ok = false;
    }
    return ok;
}

// ---- results ----
Tensor vector32(const Tensor& like, int64_t n) { return at::empty({n}, like.options().dtype(at::kFloat)); }
// as torch.empty([n, h, w, d, c]).permute(0, 4, 1, 2, 3)
Tensor volume(const Tensor& like, int64_t n, int64_t c, int64_t h, int64_t w, int64_t d)
{
    const auto at_least_1 = [](int64_t e) { return e > 1 ? e : 1; };
    const int64_t sd = at_least_1(c), sw = sd * at_least_1(d), sh = sw * at_least_1(w), sn = sh * at_least_1(h);
    return at::empty_strided({n, c, h, w, d}, {sn, 1, sh, sw, sd}, like.options());
}
at::DataPtr scratch(int64_t bytes) { return c10::hip::HIPCachingAllocator::get()->allocate(bytes > 16 ? (size_t)bytes : 16); }
int32_t dtype_tag(at::ScalarType t) { return t == at::kHalf ? 0 : t == at::kFloat ? 1 : t == at::kBFloat16 ? 2 : -1; }

struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

struct Fault {
    const char* name = nullptr;
    int64_t code = 0;
};

PyObject* wrapped(std::initializer_list<Tensor> ts)
{
    if (ts.size() == 1) return THPVariable_Wrap(*ts.begin());
    PyObject* out = PyTuple_New((Py_ssize_t)ts.size());
    if (!out) return nullptr;
    Py_ssize_t i = 0;
    for (const Tensor& t : ts) {
        PyObject* o = THPVariable_Wrap(t);
        if (!o) {
            Py_DECREF(out);
            return nullptr;
        }
        PyTuple_SET_ITEM(out, i++, o);
    }
    return out;
}

// the binding's own exception, with the library's text for this thread
PyObject* raise(const Fault& f)
{
    PyObject* r = PyObject_CallMethod(lib_module, "fail", "sL", f.name, (long long)f.code);
    Py_XDECREF(r);
    return nullptr;
}

// FAULT: leaves the surrounding function object with an error code of the library
#define CHECKED(entry, ...)                                    \
    if (const int rc_ = lib.entry(__VA_ARGS__); rc_ != 0) {    \
        return Fault{"kerops_" #entry, rc_};                   \
    }
#define SIZED(bytes, entry, ...)                               \
    const int64_t bytes = lib.entry(__VA_ARGS__);              \
    if (bytes < 0) return Fault{"kerops_" #entry, bytes};

// body: allocates and launches, without the interpreter lock
template <class F>
bool run(F&& body, Fault& fault)
{
    NoGil unlocked;
    fault = body();
    return fault.name == nullptr;
}
#define RUN(...)                              \
    Fault fault;                              \
    if (!run(__VA_ARGS__, fault)) return raise(fault);

#define OP(name) \
    PyObject* name##_body(PyObject* const* a, Py_ssize_t n, [[maybe_unused]] PyObject* kw)
#define DECLINE return nullptr

OP(DWConv)
{
    if (n != 2 || kw || !steady(op_DWConv)) DECLINE;
    const Volume x(a[0]);
    const Tensor* wt = gpu_tensor(a[1]);
    Where at;
    int32_t tw, td, lane;
    if (!x || !power_of_2(x.c) || !is_taps(wt, x.c) || !at.holds({x.t, wt}) ||
        !conv_shape(fwd_conf, k_fwd_variants, x.c, x.c == 8 && x.d > 32, tw, td, lane))
        DECLINE;
    Tensor y;
    RUN([&]() -> Fault {
        y = at::empty_like(*x.t);
        CHECKED(dwconv_fwd_f16, x.t->data_ptr(), wt->data_ptr(), y.data_ptr(), x.n, x.h, x.w, x.d, (int32_t)x.c, tw, td, 0, lane,
                at.handle())
        return {};
    })
    return wrapped({y});
}

OP(DWConvStats)
{
    if (n != 2 || kw || !steady(op_DWConvStats)) DECLINE;
    const Volume x(a[0]);
    const Tensor* wt = gpu_tensor(a[1]);
    Where at;
    if (!x || !power_of_2(x.c) || !is_taps(wt, x.c) || !at.holds({x.t, wt})) DECLINE;
    const int32_t c = (int32_t)x.c;
    Tensor y, mean, sqmean;
    RUN([&]() -> Fault {
        SIZED(bytes, dwconv_stats_workspace_bytes, x.n, x.h, x.w, x.d, c)
        y = at::empty_like(*x.t), mean = vector32(*x.t, c), sqmean = vector32(*x.t, c);
        const at::DataPtr ws = scratch(bytes);
        CHECKED(dwconv_stats_f16, x.t->data_ptr(), wt->data_ptr(), y.data_ptr(), (float*)mean.data_ptr(), (float*)sqmean.data_ptr(),
                ws.get(), bytes, x.n, x.h, x.w, x.d, c, at.handle())
        return {};
    })
    return wrapped({y, mean, sqmean});
}

OP(DWConvBackward)
{
    at::ScalarType type = at::kHalf;
    if (n != 3 || !steady(op_DWConvBackward) || !out_dtype(a + n, kw, type)) DECLINE;
    const Volume x(a[0]), g(a[1]);
    const Tensor* wt = gpu_tensor(a[2]);
    Where at;
    if (!x || !g || !x.same_shape(g) || !power_of_2(x.c) || x.c < 8 || x.c > 128 || !is_taps(wt, x.c) || !at.holds({x.t, g.t, wt}))
        DECLINE;
    const int32_t c = (int32_t)x.c;
    Tensor dx, dw;
    RUN([&]() -> Fault {
        SIZED(bytes, dwconv_bwd_workspace_bytes, x.n, x.h, x.w, x.d, c, 0)
        dx = at::empty_like(*x.t), dw = at::empty({3, 3, 3, c}, x.t->options().dtype(type));
        const at::DataPtr ws = scratch(bytes);
        CHECKED(dwconv_bwd_f16_out, x.t->data_ptr(), g.t->data_ptr(), wt->data_ptr(), dx.data_ptr(), dw.data_ptr(), dtype_tag(type),
                ws.get(), bytes, x.n, x.h, x.w, x.d, c, 0, at.handle())
        return {};
    })
    return wrapped({dx, dw});
}

OP(DWConvWGRAD)
{
    at::ScalarType type = at::kHalf;
    if (n != 2 || !steady(op_DWConvWGRAD) || !out_dtype(a + n, kw, type)) DECLINE;
    const Volume x(a[0]), g(a[1]);
    Where at;
    int32_t tw, td, lane;
    if (!x || !g || !x.same_shape(g) || !power_of_2(x.c) || x.c < 8 || x.c > 128 || !at.holds({x.t, g.t}) ||
        !conv_shape(wgrad_conf, k_wgrad_variants, x.c, false, tw, td, lane))
        DECLINE;
    const int32_t c = (int32_t)x.c;
    Tensor dw;
    RUN([&]() -> Fault {
        SIZED(bytes, dwconv_wgrad_workspace_bytes, x.n, x.h, x.w, x.d, c, tw, td, 0, lane)
        const at::DataPtr ws = scratch(bytes);
        dw = at::empty({3, 3, 3, c}, x.t->options().dtype(type));
        CHECKED(dwconv_wgrad_f16_out, x.t->data_ptr(), g.t->data_ptr(), dw.data_ptr(), dtype_tag(type), ws.get(), bytes, x.n, x.h,
                x.w, x.d, c, tw, td, 0, lane, at.handle())
        return {};
    })
    return wrapped({dw});
}

OP(Stats)
{
    if (n != 1 || kw || !steady(op_Stats)) DECLINE;
    const Volume x(a[0]);
    Where at;
    Shape s;
    if (!x || !power_of_2(x.c) || !at.holds({x.t}) || !stream_shape(op_Stats, x.c, 2 * x.v * x.c, s)) DECLINE;
    const int32_t c = (int32_t)x.c;
    Tensor mean, sqmean;
    RUN([&]() -> Fault {
        SIZED(bytes, stats_workspace_bytes, x.v, c, s.blocks)
        const at::DataPtr ws = scratch(bytes);
        mean = vector32(*x.t, c), sqmean = vector32(*x.t, c);
        CHECKED(stats_f16, x.t->data_ptr(), (float*)mean.data_ptr(), (float*)sqmean.data_ptr(), x.v, c, ws.get(), bytes, s.blocks,
                s.warps, s.segment, at.handle())
        return {};
    })
    return wrapped({mean, sqmean});
}

OP(StatsBackward)
{
    if (n != 3 || kw || !steady(op_StatsBackward)) DECLINE;
    const Volume x(a[0]);
    const Tensor *gm = gpu_tensor(a[1]), *gs = gpu_tensor(a[2]);
    Where at;
    Shape s;
    if (!x || !power_of_2(x.c) || !is_affine(gm, x.c) || !is_affine(gs, x.c) || !at.holds({x.t, gm, gs}) ||
        !stream_shape(op_StatsBackward, x.c, 2 * x.v * x.c, s))
        DECLINE;
    Tensor dx;
    RUN([&]() -> Fault {
        dx = at::empty_like(*x.t);
        CHECKED(stats_bwd_f16, x.t->data_ptr(), (const float*)gm->data_ptr(), (const float*)gs->data_ptr(), dx.data_ptr(), x.v,
                (int32_t)x.c, s.blocks, s.warps, s.segment, at.handle())
        return {};
    })
    return wrapped({dx});
}

OP(AddStats)
{
    // (in place, the third argument, is left to the Python function)
    if (n != 2 || kw || !steady(op_AddStats)) DECLINE;
    const Volume x(a[0]), y(a[1]);
    Where at;
    Shape s;
    if (!x || !y || !x.same_shape(y) || !power_of_2(x.c) || !at.holds({x.t, y.t}) ||
        !stream_shape(op_AddStats, x.c, 2 * x.v * x.c, s))
        DECLINE;
    const int32_t c = (int32_t)x.c;
    Tensor z, mean, sqmean;
    RUN([&]() -> Fault {
        z = at::empty_like(*x.t);
        SIZED(bytes, stats_workspace_bytes, x.v, c, s.blocks)
        const at::DataPtr ws = scratch(bytes);
        mean = vector32(*x.t, c), sqmean = vector32(*x.t, c);
        CHECKED(add_stats_f16, x.t->data_ptr(), y.t->data_ptr(), z.data_ptr(), (float*)mean.data_ptr(), (float*)sqmean.data_ptr(), x.v,
                c, ws.get(), bytes, s.blocks, s.warps, s.segment, at.handle())
        return {};
    })
    return wrapped({z, mean, sqmean});
}

OP(AddStatsBackward)
{
    if (n != 4 || kw || !steady(op_AddStatsBackward)) DECLINE;
    const Volume g(a[0]), z(a[3]);
    const Tensor *gm = gpu_tensor(a[1]), *gs = gpu_tensor(a[2]);
    Where at;
    Shape s;
    if (!g || !z || !g.same_shape(z) || !power_of_2(g.c) || !is_affine(gm, g.c) || !is_affine(gs, g.c) ||
        !at.holds({g.t, z.t, gm, gs}) || !stream_shape(op_AddStatsBackward, g.c, 2 * g.v * g.c, s))
        DECLINE;
    Tensor dx;
    RUN([&]() -> Fault {
        dx = at::empty_like(*g.t);
        CHECKED(add_stats_bwd_f16, g.t->data_ptr(), (const float*)gm->data_ptr(), (const float*)gs->data_ptr(), z.t->data_ptr(),
                dx.data_ptr(), g.v, (int32_t)g.c, s.blocks, s.warps, s.segment, at.handle())
        return {};
    })
    return wrapped({dx});
}

OP(ApplyBNReLU)
{
    if (n != 3 || kw || !steady(op_ApplyBNReLU)) DECLINE;
    const Volume x(a[0]);
    const Tensor *wt = gpu_tensor(a[1]), *b = gpu_tensor(a[2]);
    Where at;
    Shape s;
    if (!x || !power_of_2(x.c) || !is_affine(wt, x.c) || !is_affine(b, x.c) || !at.holds({x.t, wt, b}) ||
        !stream_shape(op_ApplyBNReLU, x.c, 2 * x.v * x.c, s))
        DECLINE;
    Tensor y;
    RUN([&]() -> Fault {
        y = at::empty_like(*x.t);
        CHECKED(bnrelu_fwd_f16, x.t->data_ptr(), (const float*)wt->data_ptr(), (const float*)b->data_ptr(), y.data_ptr(), x.v,
                (int32_t)x.c, s.blocks, s.warps, s.segment, at.handle())
        return {};
    })
    return wrapped({y});
}

OP(ApplyBNReLUBackward)
{
    if (n != 4 || kw || !steady(op_ApplyBNReLUBackward)) DECLINE;
    const Volume x(a[0]), g(a[3]);
    const Tensor *wt = gpu_tensor(a[1]), *b = gpu_tensor(a[2]);
    Where at;
    Shape s;
    if (!x || !g || !x.same_shape(g) || !power_of_2(x.c) || !is_affine(wt, x.c) || !is_affine(b, x.c) ||
        !at.holds({x.t, g.t, wt, b}) || !stream_shape(op_ApplyBNReLUBackward, x.c, 2 * x.v * x.c, s))
        DECLINE;
    const int32_t c = (int32_t)x.c;
    Tensor dx, dw, db;
    RUN([&]() -> Fault {
        dx = at::empty_like(*x.t), dw = at::empty_like(*wt), db = at::empty_like(*b);
        SIZED(bytes, stats_workspace_bytes, x.v, c, s.blocks)
        const at::DataPtr ws = scratch(bytes);
        CHECKED(bnrelu_bwd_f16, x.t->data_ptr(), (const float*)wt->data_ptr(), (const float*)b->data_ptr(), g.t->data_ptr(),
                dx.data_ptr(), (float*)dw.data_ptr(), (float*)db.data_ptr(), x.v, c, ws.get(), bytes, s.blocks, s.warps, s.segment,
                at.handle())
        return {};
    })
    return wrapped({dx, dw, db});
}

OP(AvgPoolCeilStats)
{
    if (n != 1 || kw || !steady(op_AvgPoolCeilStats)) DECLINE;
    const Volume x(a[0]);
    Where at;
    Shape s;
    int64_t l1;
    if (!x || !power_of_2(x.c) || !at.holds({x.t}) || !stream_shape(op_AvgPoolCeilStats, x.c, 2 * x.v * x.c, s) ||
        !as_int(PyDict_GetItem(hardware_conf, k_l1), l1) || l1 < 0 || x.d * x.c > l1 / 2)
        DECLINE;
    const int32_t c = (int32_t)x.c;
    Tensor y, mean, sqmean;
    RUN([&]() -> Fault {
        y = volume(*x.t, x.n, c, (x.h + 1LL) / 2, (x.w + 1LL) / 2, (x.d + 1LL) / 2);
        mean = vector32(*x.t, c), sqmean = vector32(*x.t, c);
        SIZED(bytes, avgpool_ceil_stats_workspace_bytes, x.n, x.h, x.w, x.d, c, s.blocks)
        const at::DataPtr ws = scratch(bytes);
        CHECKED(avgpool_ceil_stats_f16, x.t->data_ptr(), y.data_ptr(), (float*)mean.data_ptr(), (float*)sqmean.data_ptr(), x.n, x.h,
                x.w, x.d, c, ws.get(), bytes, s.blocks, s.warps, s.segment, at.handle())
        return {};
    })
    return wrapped({y, mean, sqmean});
}

OP(ApplyBNReLUAvgPoolCeilStats)
{
    if (n != 3 || kw || !steady(op_ApplyBNReLUAvgPoolCeilStats)) DECLINE;
    const Volume x(a[0]);
    const Tensor *wt = gpu_tensor(a[1]), *b = gpu_tensor(a[2]);
    Where at;
    Shape s;
    if (!x || !power_of_2(x.c) || !is_affine(wt, x.c) || !is_affine(b, x.c) || !at.holds({x.t, wt, b}) ||
        !stream_shape(op_ApplyBNReLUAvgPoolCeilStats, x.c, 2 * x.v * x.c, s))
        DECLINE;
    const int32_t c = (int32_t)x.c;
    Tensor y, mean, sqmean;
    RUN([&]() -> Fault {
        y = volume(*x.t, x.n, c, (x.h + 1LL) / 2, (x.w + 1LL) / 2, (x.d + 1LL) / 2);
        mean = vector32(*x.t, c), sqmean = vector32(*x.t, c);
        SIZED(bytes, avgpool_ceil_stats_workspace_bytes, x.n, x.h, x.w, x.d, c, s.blocks)
        const at::DataPtr ws = scratch(bytes);
        CHECKED(bnrelu_avgpool_ceil_stats_f16, x.t->data_ptr(), (const float*)wt->data_ptr(), (const float*)b->data_ptr(),
                y.data_ptr(), (float*)mean.data_ptr(), (float*)sqmean.data_ptr(), x.n, x.h, x.w, x.d, c, ws.get(), bytes, s.blocks,
                s.warps, s.segment, at.handle())
        return {};
    })
    return wrapped({y, mean, sqmean});
}

OP(AvgPoolCeilStatsBackward)
{
    if (n != 5 || kw || !steady(op_AvgPoolCeilStatsBackward) || !PyTuple_Check(a[4]) || PyTuple_GET_SIZE(a[4]) != 5) DECLINE;
    int64_t e[5];  // N, C, H, W, D of the gradient that the op writes
    for (int i = 0; i < 5; ++i)
        if (!as_int(PyTuple_GET_ITEM(a[4], i), e[i]) || e[i] < 0 || e[i] > INT_MAX) DECLINE;
    const Volume g(a[0]), y(a[3]);
    const Tensor *gm = gpu_tensor(a[1]), *gs = gpu_tensor(a[2]);
    Where at;
    Shape s;
    int64_t l1;
    if (!g || !y || !g.same_shape(y) || g.c != e[1] || !power_of_2(g.c) || g.n != e[0] || g.h != (e[2] + 1) / 2 ||
        g.w != (e[3] + 1) / 2 || g.d != (e[4] + 1) / 2 || !is_affine(gm, g.c) || !is_affine(gs, g.c) ||
        !at.holds({g.t, y.t, gm, gs}) || !as_int(PyDict_GetItem(hardware_conf, k_l1), l1) || l1 < 0 || e[4] * e[1] > l1 / 2 ||
        !stream_shape(op_AvgPoolCeilStatsBackward, g.c, 2 * e[0] * e[1] * e[2] * e[3] * e[4], s))
        DECLINE;
    Tensor dx;
    RUN([&]() -> Fault {
        dx = volume(*g.t, e[0], e[1], e[2], e[3], e[4]);
        CHECKED(avgpool_ceil_stats_bwd_f16, g.t->data_ptr(), (const float*)gm->data_ptr(), (const float*)gs->data_ptr(),
                y.t->data_ptr(), dx.data_ptr(), (int32_t)e[0], (int32_t)e[2], (int32_t)e[3], (int32_t)e[4], (int32_t)e[1], s.blocks,
                s.warps, s.segment, at.handle())
        return {};
    })
    return wrapped({dx});
}

OP(ReLULinearAdd)
{
    if (n != 3 || kw || !steady(op_ReLULinearAdd)) DECLINE;
    const Volume x(a[0]), add(a[2]);
    const Tensor* wt = gpu_tensor(a[1]);
    Where at;
    if (!x || !add || !x.same_space(add) || !built_linear(x.c) || !built_linear(add.c) || !is_matrix(wt, {x.c, add.c}) ||
        !at.holds({x.t, wt, add.t}))
        DECLINE;
    Tensor y;
    RUN([&]() -> Fault {
        y = at::empty_like(*add.t);
        CHECKED(pointwise_f16, x.t->data_ptr(), wt->data_ptr(), add.t->data_ptr(), y.data_ptr(), x.v, (int32_t)x.c, (int32_t)add.c, 1,
                at.handle())
        return {};
    })
    return wrapped({y});
}

OP(ReLULinearBackward)
{
    at::ScalarType type = at::kHalf;
    if (n != 3 || !steady(op_ReLULinearBackward) || !out_dtype(a + n, kw, type)) DECLINE;
    const Volume x(a[0]), g(a[1]);
    const Tensor* wt = gpu_tensor(a[2]);
    Where at;
    if (!x || !g || !x.same_space(g) || !built_linear(x.c) || !built_linear(g.c) || !is_matrix(wt, {x.c, g.c}) ||
        !at.holds({x.t, g.t, wt}))
        DECLINE;
    const int32_t ci = (int32_t)x.c, co = (int32_t)g.c;
    Tensor dx, dw;
    RUN([&]() -> Fault {
        SIZED(bytes, relu_linear_bwd_workspace_bytes, g.v, ci, co)
        const at::DataPtr ws = scratch(bytes);
        dx = at::empty_like(*x.t), dw = at::empty({ci, co}, x.t->options().dtype(type));
        CHECKED(relu_linear_bwd_f16_out, x.t->data_ptr(), g.t->data_ptr(), wt->data_ptr(), dx.data_ptr(), dw.data_ptr(),
                dtype_tag(type), ws.get(), bytes, g.v, ci, co, at.handle())
        return {};
    })
    return wrapped({dx, dw});
}

OP(ApplyBNReLULinearAdd)
{
    if (n != 5 || kw || !steady(op_ApplyBNReLULinearAdd)) DECLINE;
    const Volume x(a[0]), add(a[4]);
    const Tensor *scale = gpu_tensor(a[1]), *shift = gpu_tensor(a[2]), *wt = gpu_tensor(a[3]);
    Where at;
    if (!x || !add || !x.same_space(add) || !built_linear(x.c) || !built_linear(add.c) || !is_matrix(wt, {x.c, add.c}) ||
        !is_affine(scale, x.c) || !is_affine(shift, x.c) || !at.holds({x.t, scale, shift, wt, add.t}))
        DECLINE;
    Tensor y;
    RUN([&]() -> Fault {
        y = at::empty_like(*add.t);
        CHECKED(bnrelu_pointwise_f16, x.t->data_ptr(), (const float*)scale->data_ptr(), (const float*)shift->data_ptr(),
                wt->data_ptr(), add.t->data_ptr(), y.data_ptr(), x.v, (int32_t)x.c, (int32_t)add.c, at.handle())
        return {};
    })
    return wrapped({y});
}

OP(ApplyBNReLULinearBackward)
{
    if (n != 5 || kw || !steady(op_ApplyBNReLULinearBackward)) DECLINE;
    const Volume x(a[0]), g(a[3]);
    const Tensor *scale = gpu_tensor(a[1]), *shift = gpu_tensor(a[2]), *wt = gpu_tensor(a[4]);
    Where at;
    if (!x || !g || !x.same_space(g) || !built_linear(x.c) || !built_linear(g.c) || !is_matrix(wt, {x.c, g.c}) ||
        !is_affine(scale, x.c) || !is_affine(shift, x.c) || !at.holds({x.t, scale, shift, g.t, wt}))
        DECLINE;
    const int32_t ci = (int32_t)x.c, co = (int32_t)g.c;
    Tensor dx, dw, affine;
    RUN([&]() -> Fault {
        SIZED(bytes, bnrelu_linear_bwd_workspace_bytes, x.v, ci, co)
        const at::DataPtr ws = scratch(bytes);
        dx = at::empty_like(*x.t), dw = at::empty_like(*wt), affine = at::empty({2, ci}, x.t->options().dtype(at::kFloat));
        CHECKED(bnrelu_linear_bwd_f16, x.t->data_ptr(), (const float*)scale->data_ptr(), (const float*)shift->data_ptr(),
                g.t->data_ptr(), wt->data_ptr(), dx.data_ptr(), dw.data_ptr(), 0, (float*)affine.data_ptr(), ws.get(), bytes, x.v, ci,
                co, at.handle())
        return {};
    })
    return wrapped({dx, affine.select(0, 0), affine.select(0, 1), dw});
}

OP(LinBReLULinAdd)
{
    if (n != 5 || kw || !steady(op_LinBReLULinAdd)) DECLINE;
    const Volume x(a[0]), add(a[4]);
    const Tensor *up = gpu_tensor(a[1]), *down = gpu_tensor(a[2]), *bias = gpu_tensor(a[3]);
    Where at;
    if (!x || !add || !x.same_shape(add) || !(x.c == 16 || x.c == 32 || x.c == 64) || !is_matrix(up, {x.c, 2 * x.c}) ||
        !is_matrix(down, {2 * x.c, x.c}) || !is_matrix(bias, {2 * x.c}) || !at.holds({x.t, up, down, bias, add.t}))
        DECLINE;
    Tensor y;
    RUN([&]() -> Fault {
        y = at::empty_like(*x.t);
        CHECKED(lin_brelu_lin_add_f16, x.t->data_ptr(), up->data_ptr(), down->data_ptr(), bias->data_ptr(), add.t->data_ptr(),
                y.data_ptr(), x.v, (int32_t)x.c, at.handle())
        return {};
    })
    return wrapped({y});
}

OP(LinBReLULinBackward)
{
    at::ScalarType type = at::kHalf;
    if (n != 5 || !steady(op_LinBReLULinBackward) || !out_dtype(a + n, kw, type)) DECLINE;
    const Volume x(a[0]), g(a[1]);
    const Tensor *up = gpu_tensor(a[2]), *down = gpu_tensor(a[3]), *bias = gpu_tensor(a[4]);
    Where at;
    if (!x || !g || !x.same_shape(g) || !(x.c == 16 || x.c == 32 || x.c == 64) || !is_matrix(up, {x.c, 2 * x.c}) ||
        !is_matrix(down, {2 * x.c, x.c}) || !is_matrix(bias, {2 * x.c}) || !at.holds({x.t, g.t, up, down, bias}))
        DECLINE;
    const int32_t c = (int32_t)x.c;
    Tensor dx, dup, ddown, dbias;
    RUN([&]() -> Fault {
        SIZED(bytes, lin_brelu_lin_bwd_workspace_bytes, x.v, c)
        const at::DataPtr ws = scratch(bytes);
        const auto res = x.t->options().dtype(type);
        dx = at::empty_like(*x.t), dup = at::empty({c, 2 * c}, res), ddown = at::empty({2 * c, c}, res);
        dbias = at::empty({2 * c}, res);
        CHECKED(lin_brelu_lin_bwd_f16_out, x.t->data_ptr(), g.t->data_ptr(), up->data_ptr(), down->data_ptr(), bias->data_ptr(),
                dx.data_ptr(), dup.data_ptr(), ddown.data_ptr(), dbias.data_ptr(), dtype_tag(type), ws.get(), bytes, x.v, c, at.handle())
        return {};
    })
    return wrapped({dx, dup, ddown, dbias});
}

// a flat stream: any dense layout (quantization._dense)
bool dense(const Tensor& t)
{
    return t.is_contiguous() || (t.dim() == 5 && t.is_contiguous(at::MemoryFormat::ChannelsLast3d)) ||
           (t.dim() == 4 && t.is_contiguous(at::MemoryFormat::ChannelsLast));
}

bool as_window(PyObject* o, float& w)
{
    if (!PyFloat_CheckExact(o)) return false;
    w = (float)PyFloat_AS_DOUBLE(o);
    return true;
}

OP(QuantUint8Window)
{
    if (n != 2 || kw || !steady(op_QuantUint8Window)) DECLINE;
    const Tensor* x = gpu_tensor(a[0]);
    Where at;
    Shape s;
    float window;
    if (!x || dtype_tag(x->scalar_type()) < 0 || !dense(*x) || !as_window(a[1], window) || !at.holds({x}) ||
        !stream_shape(op_QuantUint8Window, x->dim() == 5 ? x->size(1) : 0, x->numel() * (int64_t)x->element_size(), s))
        DECLINE;
    Tensor q;
    RUN([&]() -> Fault {
        q = at::empty_like(*x, x->options().dtype(at::kByte));
        CHECKED(quant_u8_window, x->data_ptr(), dtype_tag(x->scalar_type()), (uint8_t*)q.data_ptr(), x->numel(), window, s.blocks,
                s.warps, s.segment, at.handle())
        return {};
    })
    return wrapped({q});
}

OP(DequantUint8Window)
{
    if (n != 3 || kw || !steady(op_DequantUint8Window) || !THPDtype_Check(a[1])) DECLINE;
    const Tensor* x = gpu_tensor(a[0]);
    const at::ScalarType type = ((THPDtype*)a[1])->scalar_type;
    Where at;
    Shape s;
    float window;
    if (!x || x->scalar_type() != at::kByte || dtype_tag(type) < 0 || !dense(*x) || !as_window(a[2], window) || !at.holds({x}) ||
        !stream_shape(op_DequantUint8Window, x->dim() == 5 ? x->size(1) : 0, x->numel(), s))
        DECLINE;
    Tensor y;
    RUN([&]() -> Fault {
        y = at::empty_like(*x, x->options().dtype(type));
        CHECKED(dequant_u8_window, (const uint8_t*)x->data_ptr(), y.data_ptr(), dtype_tag(type), x->numel(), window, s.blocks, s.warps,
                s.segment, at.handle())
        return {};
    })
    return wrapped({y});
}

OP(QuantInt8Sym)
{
    if (n != 2 || kw || !steady(op_QuantInt8Sym)) DECLINE;
    const Tensor *y = gpu_tensor(a[0]), *absmax = gpu_tensor(a[1]);
    Where at;
    Shape s;
    if (!y || y->scalar_type() != at::kHalf || !dense(*y) || !is_affine(absmax, 1) || !at.holds({y, absmax}) ||
        !stream_shape(op_QuantInt8Sym, y->dim() == 5 ? y->size(1) : 0, y->numel() * 2, s))
        DECLINE;
    Tensor q, scale;
    RUN([&]() -> Fault {
        q = at::empty_like(*y, y->options().dtype(at::kChar)), scale = at::empty_like(*absmax);
        CHECKED(quant_i8_sym_f16, y->data_ptr(), (const float*)absmax->data_ptr(), (int8_t*)q.data_ptr(), (float*)scale.data_ptr(),
                y->numel(), s.blocks, s.warps, s.segment, at.handle())
        return {};
    })
    return wrapped({q, scale});
}

OP(DWSepBlock)
{
    if (n != 5 || kw || !steady(op_DWSepBlock)) DECLINE;
    const Volume x(a[0]);
    const Tensor *dw = gpu_tensor(a[1]), *scale = gpu_tensor(a[2]), *shift = gpu_tensor(a[3]), *pw = gpu_tensor(a[4]);
    Where at;
    if (!x || !is_taps(dw, x.c) || !is_affine(scale, x.c) || !is_affine(shift, x.c) || !pw || pw->dim() != 2 ||
        !is_matrix(pw, {x.c, pw->size(1)}) || pw->size(1) > INT_MAX || !at.holds({x.t, dw, scale, shift, pw}))
        DECLINE;
    const int32_t ci = (int32_t)x.c, co = (int32_t)pw->size(1);
    Tensor y, absmax;
    RUN([&]() -> Fault {
        SIZED(bytes, dwsep_block_workspace_bytes, x.n, x.h, x.w, x.d, ci, co)
        const at::DataPtr ws = scratch(bytes);
        y = volume(*x.t, x.n, co, x.h, x.w, x.d), absmax = vector32(*x.t, 1);
        CHECKED(dwsep_block_f16, x.t->data_ptr(), dw->data_ptr(), (const float*)scale->data_ptr(), (const float*)shift->data_ptr(),
                pw->data_ptr(), y.data_ptr(), (float*)absmax.data_ptr(), x.n, x.h, x.w, x.d, ci, co, ws.get(), bytes, at.handle())
        return {};
    })
    return wrapped({y, absmax});
}

// ---- module ----
#define X(name)                                                                                       \
    PyObject* name##_call(PyObject*, PyObject* const* a, Py_ssize_t n, PyObject* kw)                  \
    {                                                                                                 \
        HANDLE_TH_ERRORS                                                                              \
        PyObject* out = name##_body(a, n, kw);                                                        \
        if (!out && !PyErr_Occurred()) Py_RETURN_NONE;                                                \
        return out;                                                                                   \
        END_HANDLE_TH_ERRORS                                                                          \
    }
KEROPS_OPS(X)
#undef X

// setup(entry points {name: address}, {op: (attributes of its ConfiguredFunction or None, [(dictionary, or None for the
// configurators, key, value), ...])}, binding module, dictionaries of stream_table, hardware_conf, ops.conv.dwconv and
// ops.conv.dwconv_wgrad)
PyObject* setup(PyObject*, PyObject* args)
{
    PyObject *entries, *watch, *module, *stream, *hardware, *fwd, *wgrad;
    if (!PyArg_ParseTuple(args, "O!O!OO!O!O!O!", &PyDict_Type, &entries, &PyDict_Type, &watch, &module, &PyDict_Type, &stream,
                          &PyDict_Type, &hardware, &PyDict_Type, &fwd, &PyDict_Type, &wgrad))
        return nullptr;
    int64_t address;
#define X(name)                                                                                                          \
    if (!as_int(PyDict_GetItemString(entries, "kerops_" #name), address) || !address)                                    \
        return PyErr_Format(PyExc_RuntimeError, "no address of kerops_%s", #name);                                       \
    lib.name = (decltype(lib.name))(uintptr_t)address;
    KEROPS_ENTRIES(X)
#undef X
    // (references are kept for the life of the process)
    Py_INCREF(module), Py_INCREF(stream), Py_INCREF(hardware), Py_INCREF(fwd), Py_INCREF(wgrad);
    lib_module = module, stream_table = stream, hardware_conf = hardware, fwd_conf = fwd, wgrad_conf = wgrad;
    for (int op = 0; op < kOps; ++op) {
        PyObject *item = PyDict_GetItem(watch, op_names[op]), *op_dict, *list;
        if (!item) return PyErr_Format(PyExc_RuntimeError, "nothing to watch for %U", op_names[op]);
        if (!PyArg_ParseTuple(item, "OO!", &op_dict, &PyList_Type, &list)) return nullptr;
        Relied r;
        if (op_dict != Py_None) r.op_dict = op_dict, Py_INCREF(op_dict);
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(list); ++i) {
            PyObject *dict, *key, *value;
            if (!PyArg_ParseTuple(PyList_GET_ITEM(list, i), "OOO", &dict, &key, &value)) return nullptr;
            if (dict == Py_None && r.op_dict) dict = nullptr;
            else if (!PyDict_Check(dict)) return PyErr_Format(PyExc_RuntimeError, "%U: not a dictionary", op_names[op]);
            size_t d = 0;
            while (d < r.dicts.size() && r.dicts[d].dict != dict) ++d;
            if (d == r.dicts.size()) {
                Py_XINCREF(dict);
                r.dicts.push_back({dict, {}});
            }
            Py_INCREF(key), Py_INCREF(value);
            r.dicts[d].entries.emplace_back(key, value);
        }
        relied[op] = std::move(r);
    }
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"setup", setup, METH_VARARGS, nullptr},
#define X(name) {#name, (PyCFunction)(void (*)())name##_call, METH_FASTCALL | METH_KEYWORDS, nullptr},
    KEROPS_OPS(X)
#undef X
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef definition = {PyModuleDef_HEAD_INIT, "kerops_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_kerops_host()
{
    const auto name = [](const char* s) { return PyUnicode_InternFromString(s); };
#define X(op) op_names[op_##op] = name(#op);
    KEROPS_OPS(X)
#undef X
    k_table = name("_table"), k_small_bytes = name("SMALL_BYTES"), k_small = name("small"), k_default = name("default");
    k_blocks = name("blocks"), k_warps = name("num_warps"), k_segment = name("segment"), k_l1 = name("L1_CACHE_BYTES");
    k_tile_w = name("_TILE_W"), k_tile_d = name("_TILE_D"), k_lane = name("_LANE_C"), k_waves = name("_WAVES");
    k_fwd_variants = name("FWD_VARIANTS"), k_wgrad_variants = name("WGRAD_VARIANTS"), k_out_dtype = name("out_dtype");
    k_configurators = name("configurators");
    PyObject* m = PyModule_Create(&definition);
    // what the binding compares before it calls anything else: the layouts of torch's and the interpreter's objects that
    // this file was compiled with are those of these versions only
    if (m && (PyModule_AddIntConstant(m, "HEADER_VERSION", KEROPS_HIP_VERSION) != 0 ||
              PyModule_AddStringConstant(m, "TORCH_VERSION", KEROPS_TORCH_VERSION) != 0 ||
              PyModule_AddIntConstant(m, "PYTHON_VERSION", PY_VERSION_HEX >> 16) != 0))
        Py_CLEAR(m);
    return m;
}
