// Host side of the package's hot calls as a CPython extension (`arcq_vit_amd._arcq_host`): what a forward does between
// the Python call and the kernel launches -- argument checks, the cached fp32 / contiguous views of a layer's buffers,
// output and scratch allocation, the current stream, the call into libarcq_hip.so.
//
// Why it exists: these calls are a few kernels of 5-15 us each, and the same work written in Python (attribute and
// data_ptr reads, torch.empty / reshape / torch.cuda.device, a ctypes call with some twenty arguments) costs 15-25 us
// per layer, so that up to a few hundred rows -- and, in whole models, up to a batch of about twenty -- the GPU waited
// for the host.  Measured per layer call on one box: 18 us in Python, 6 us here.
//
// Every function returns None where a call is not the plain case (an argument of another type, layout or device, a
// module with hooks, a shape the library does not run): the Python code behind it then validates, converts and raises
// as it always did.  Nothing here synchronises, but for what is done once per layer: its FP8 multiplier is read back, and the
// first call from a second stream waits for the copies that the first one makes.  What a call needs of its modules is read
// first, under the GIL; allocations, torch operations and launches follow without it, so that threads on streams of their
// own run side by side.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <algorithm>
#include <cstring>
#include <memory>
#include <optional>
#include <stdexcept>
#include <string>
#include <vector>

#include "arcq_hip.h"

namespace {

using at::Tensor;

// ---- names --------------------------------------------------------------------------------------------------------
#define ARCQ_NAMES(X)                                                                                                     \
    X(_buffers) X(_modules) X(_parameters) X(_host_plan) X(_weight_buffer) X(_x_hat_buffer) X(out_dtype) X(fp8_operands) \
    X(in_features) X(out_features) X(bits) X(group_size) X(act_group_size) X(in_channels) X(out_channels) X(kernel_size)                  \
    X(packed_weight_codes) X(weight_codebook) X(weight_center)                                                            \
    X(weight_scale) X(weight_code_sum) X(activation_codebook) X(activation_thresholds) X(bias_tensor) X(bias)             \
    X(product_table) X(weight_codes_u8) X(weight_dequant) X(runtime_code_format)                                          \
    X(weight) X(eps) X(normalized_shape) X(elementwise_affine) X(norm1) X(norm2) X(attn) X(mlp) X(qkv) X(proj) X(fc1)     \
    X(fc2) X(act) X(fuse_elementwise) X(chain_mlp) X(num_heads) X(own_kernel) X(approximate) X(none) X(forward)           \
    X(_forward_hooks) X(_forward_pre_hooks) X(_backward_hooks) X(_backward_pre_hooks) X(mix)                              \
    X(_global_forward_hooks) X(_global_forward_pre_hooks) X(_global_backward_hooks) X(_global_backward_pre_hooks)
struct Names {
#define X(n) PyObject *n;
    ARCQ_NAMES(X)
#undef X
} S;

PyObject *g_torch_module = nullptr;      // torch.nn.modules.module (the global hook dictionaries)
PyObject *g_layer_type = nullptr;        // ARCQPackedLinearOnTheFly
PyObject *g_attention_type = nullptr, *g_mlp_type = nullptr;
PyObject *g_gelu_type = nullptr, *g_layernorm_type = nullptr;
PyObject *g_fp8_multiplier = nullptr;    // ops.fp8_weight_multiplier
PyObject *g_half = nullptr, *g_float = nullptr;      // torch.float16, torch.float32

struct Failure {};      // a Python exception is set

// The part of a call that touches no Python object.
struct NoGil {
    PyThreadState *state = PyEval_SaveThread();
    NoGil() = default;
    NoGil(const NoGil &) = delete;
    ~NoGil() { PyEval_RestoreThread(state); }
};

inline void check(int rc)
{
    if (rc == 0) return;
    const char *msg = arcq_last_error();
    throw std::runtime_error(msg && msg[0] ? std::string(msg) : "libarcq_hip call failed with code " + std::to_string(rc));
}

inline PyObject *dict_of(PyObject *o)
{
    PyObject **d = _PyObject_GetDictPtr(o);
    return d ? *d : nullptr;
}
// A borrowed reference.  (The keys are interned strings, whose lookup cannot fail.)
inline PyObject *get(PyObject *dict, PyObject *key) { return dict ? PyDict_GetItemWithError(dict, key) : nullptr; }
// What `if o:` decides; an absent attribute is false.  (May run code of a class's own __bool__.)
inline bool is_true(PyObject *o)
{
    if (o == Py_True) return true;
    if (!o || o == Py_False || o == Py_None) return false;
    Py_INCREF(o);
    const int r = PyObject_IsTrue(o);
    Py_DECREF(o);
    if (r < 0) throw Failure{};
    return r == 1;
}
inline bool get_int(PyObject *dict, PyObject *key, int64_t &out)
{
    PyObject *v = get(dict, key);
    if (!v || !PyLong_CheckExact(v)) return false;
    out = PyLong_AsLongLong(v);
    return true;
}
inline const Tensor *as_tensor(PyObject *o) { return o && THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// Inference tensors have no version: a change in place leaves no trace on them, and nothing derived from one is kept.
inline bool has_version(const Tensor &t) { return t.unsafeGetTensorImpl()->version_counter().enabled(); }
inline Tensor empty(at::IntArrayRef sizes, at::ScalarType type, c10::Device device)
{
    return Tensor(at::detail::empty_cuda(sizes, type, device, std::nullopt));
}
inline void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
inline bool here(const Tensor &t) { return t.is_cuda() && t.device().index() == c10::hip::current_device(); }
inline bool f16(const Tensor &t) { return t.scalar_type() == at::kHalf; }
inline bool f32(const Tensor &t) { return t.scalar_type() == at::kFloat; }
// The library's code of a tensor's type.  It knows two: every tensor that an operation of torch's made (autocast chooses the
// type of some) goes through as_operand first.
inline int code_of(const Tensor &t)
{
    TORCH_CHECK(f16(t) || f32(t), "expected a float16 or float32 tensor, got ", t.scalar_type());
    return f16(t) ? ARCQ_F16 : ARCQ_F32;
}
inline Tensor as_operand(const Tensor &t) { return (f16(t) || f32(t) ? t : t.to(at::kHalf)).contiguous(); }
inline bool aligned16(const void *p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }
inline bool aligned16(const Tensor &t) { return aligned16(t.const_data_ptr()); }
inline const float *fptr(const Tensor &t) { return static_cast<const float *>(t.const_data_ptr()); }
inline const uint8_t *bptr(const Tensor &t) { return static_cast<const uint8_t *>(t.const_data_ptr()); }

// ---- a layer's buffers, as the library takes them -------------------------------------------------------------------
// One buffer as it was last seen: compared at every call, and converted only where the library does not take it as it lies.
// The memory stays the module's to give back: the storage is held weakly, which is enough for its address to name it.
struct Slot {
    std::optional<c10::weak_intrusive_ptr<c10::StorageImpl>> storage;
    const c10::StorageImpl *named = nullptr;
    Tensor copy;              // fp32 / contiguous, where the tensor is not
    bool tracked = true;      // changes in place show in its version
    uint32_t version = 0;
    const void *data = nullptr;
    at::ScalarType type = at::kByte;
    at::DimVector sizes, strides;
    bool same(const Tensor &t) const
    {
        const c10::TensorImpl *impl = t.unsafeGetTensorImpl();
        const auto &vc = impl->version_counter();
        return named == impl->unsafe_storage().unsafeGetStorageImpl() && data == t.const_data_ptr() && type == t.scalar_type() &&
               t.sizes().equals(sizes) && t.strides().equals(strides) &&
               (tracked ? vc.enabled() && vc.current_version() == version : !vc.enabled() && !copy.defined());
    }
    void set(const Tensor &t, bool as_f32, bool align = false)
    {
        storage.emplace(t.storage().getWeakStorageImpl());
        named = storage->_unsafe_get_target();
        tracked = has_version(t);
        version = tracked ? t.unsafeGetTensorImpl()->version_counter().current_version() : 0;
        data = t.const_data_ptr();
        type = t.scalar_type();
        sizes = t.sizes();
        strides = t.strides();
        const Tensor use = (as_f32 ? t.detach().to(at::kFloat) : t.detach()).contiguous();
        if (use.const_data_ptr() != data) copy = use;
        else if (align && !aligned16(data)) copy = use.clone();
    }
    const void *ptr() const { return copy.defined() ? copy.const_data_ptr() : data; }
    int64_t numel() const { return c10::multiply_integers(sizes); }
};
// Copies made while the stream is captured belong to the graph: nothing has run that fills them, and their memory is the graph's.
// Such a call uses them and keeps nothing.
inline bool capturing() { return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None; }
// The stream that fills a set of copies, until they are known to be filled: the first call from another stream waits for it.
// (A capture begins with a synchronised device, and may not wait.)
struct FilledOn {
    std::optional<c10::hip::HIPStream> stream;
    void settle()
    {
        if (!stream || *stream == c10::hip::getCurrentHIPStream(stream->device_index()) || capturing()) return;
        stream->synchronize();
        stream.reset();
    }
};
// References to Python objects for the length of a call (the GIL is held where it is made and where it ends).
struct Refs {
    c10::SmallVector<PyObject *, 64> held;      // (a block: four layers, two LayerNorms, nine modules)
    Refs() = default;
    Refs(const Refs &) = delete;
    ~Refs() { for (PyObject *o : held) Py_DECREF(o); }
    void add(PyObject *o)
    {
        Py_INCREF(o);
        held.push_back(o);
    }
};
struct LayerNormParams {
    Slot w, b;
    Tensor no_bias;           // zeros, for a LayerNorm without one
    FilledOn filled;
    bool copied() const { return w.copy.defined() || b.copy.defined() || no_bias.defined(); }
    bool has_bias() const { return !no_bias.defined(); }
    const float *weight() const { return static_cast<const float *>(w.ptr()); }
    const float *bias() const { return has_bias() ? static_cast<const float *>(b.ptr()) : fptr(no_bias); }
};
constexpr int kMaxSlots = 11;
struct Plan {
    c10::DeviceIndex device = -1;
    int64_t K = 0, N = 0, bits = 0, gs = 0;
    Slot slot[kMaxSlots];
    const void *p[kMaxSlots] = {};
    FilledOn filled;
    double fp8_mult = NAN;
    std::vector<LayerNormParams> ln;
};

// The plan of one module, kept in its __dict__.  `owner` is the module it was made for: copy.copy and DataParallel's replicas
// copy the __dict__ and with it the reference, and a module that finds another one's plan makes its own.  (An address can be
// compared here: a plan is used only by the living module at it, and every other holder replaces it before the first use.)
// A plan is not changed by later calls on other buffers: those publish a new one, and a call in flight keeps the one it
// began with -- Python code that runs in the middle of a call lets other threads call the same module.
struct PlanObject {
    PyObject_HEAD
    std::shared_ptr<Plan> plan;
    const void *owner;
};
PyObject *plan_new(PyTypeObject *type, PyObject *, PyObject *)
{
    PlanObject *o = reinterpret_cast<PlanObject *>(type->tp_alloc(type, 0));
    if (o) new (&o->plan) std::shared_ptr<Plan>();
    return reinterpret_cast<PyObject *>(o);
}
void plan_dealloc(PyObject *o)
{
    reinterpret_cast<PlanObject *>(o)->plan.~shared_ptr();
    Py_TYPE(o)->tp_free(o);
}
PyObject *plan_reduce(PyObject *, PyObject *)       // copies and pickles hold None in its place
{
    return Py_BuildValue("O()", reinterpret_cast<PyObject *>(Py_TYPE(Py_None)));
}
PyMethodDef plan_methods[] = {{"__reduce__", plan_reduce, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyTypeObject PlanType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// The three kinds of module: their buffers in the order of Plan::slot.
enum { A_THR, A_CB, W_PACKED, W_CB, W_CENTER, W_SCALE, W_SUM, W_BIAS, P_TABLE, P_CODES, P_DENSE };
enum class Kind { OnTheFly, Packed, Conv };

// Whether the buffers hold what the kernels will read for the layer's sizes: a buffer may have been replaced since the module
// checked them.  `indexed`: the index-space formats, whose quantizer takes no other length of a codebook.
bool shapes_ok(const Plan &p, const Tensor *const *t, bool indexed)
{
    if (p.bits < 2 || p.bits > 4 || p.gs <= 0 || p.K <= 0 || p.N <= 0 || p.K % p.gs != 0) return false;
    const int64_t levels = int64_t(1) << p.bits, meta = p.N * (p.K / p.gs);
    if (t[W_PACKED]->dim() != 2 || t[W_PACKED]->size(0) != p.N || t[W_PACKED]->size(1) != (p.K * p.bits + 7) / 8) return false;
    if (t[A_CB]->numel() < levels || t[W_CB]->numel() < levels || t[A_THR]->numel() < levels - 1) return false;
    if (indexed && (t[A_CB]->numel() != levels || t[A_THR]->numel() != levels - 1)) return false;
    for (int i : {W_CENTER, W_SCALE, W_SUM})
        if (t[i]->numel() < meta) return false;
    return t[W_BIAS]->numel() == 0 || t[W_BIAS]->numel() >= p.N;
}
// `refs` takes the module and its buffers for the length of the call: the plan itself does not keep them.
std::shared_ptr<Plan> plan_of(PyObject *module, Kind kind, Refs &refs, PyObject *&dict)
{
    dict = dict_of(module);
    PyObject *buffers = get(dict, S._buffers);
    if (!buffers || !PyDict_Check(buffers)) return nullptr;
    PyObject *po = get(dict, S._host_plan);
    std::shared_ptr<Plan> plan;
    if (po && Py_TYPE(po) == &PlanType && reinterpret_cast<PlanObject *>(po)->owner == module)
        plan = reinterpret_cast<PlanObject *>(po)->plan;
    PyObject *const names[kMaxSlots] = {S.activation_thresholds, S.activation_codebook, S.packed_weight_codes, S.weight_codebook,
                                        S.weight_center, S.weight_scale, S.weight_code_sum,
                                        kind == Kind::OnTheFly ? S.bias_tensor : S.bias, S.product_table, S.weight_codes_u8,
                                        S.weight_dequant};
    const int n = kind == Kind::Packed ? 11 : 8;
    const Tensor *t[kMaxSlots];
    bool same = plan != nullptr;
    refs.add(module);
    for (int i = 0; i < n; ++i) {
        PyObject *o = get(buffers, names[i]);
        t[i] = as_tensor(o);
        if (!t[i]) return nullptr;
        refs.add(o);
        same = same && plan->slot[i].same(*t[i]);
    }
    if (same) {
        plan->filled.settle();
        return plan;
    }
    plan = std::make_shared<Plan>();
    const c10::Device dev = t[W_PACKED]->device();
    for (int i = 0; i < n; ++i) {
        if (t[i]->numel() == 0) continue;
        if (!t[i]->is_cuda() || t[i]->device() != dev) return nullptr;
    }
    if (!t[W_PACKED]->is_cuda() || t[W_PACKED]->scalar_type() != at::kByte) return nullptr;
    if (kind == Kind::Conv) {
        int64_t c;                       // (the call below serves 16 x 16 patches only)
        if (!get_int(dict, S.in_channels, c) || !get_int(dict, S.out_channels, plan->N)) return nullptr;
        plan->K = 256 * c;
    } else if (!get_int(dict, S.in_features, plan->K) || !get_int(dict, S.out_features, plan->N)) {
        return nullptr;
    }
    if (!get_int(dict, S.bits, plan->bits) || !get_int(dict, S.group_size, plan->gs)) return nullptr;
    if (!shapes_ok(*plan, t, kind == Kind::Packed)) return nullptr;
    for (int i = 0; i < n; ++i) {
        plan->slot[i].set(*t[i], i != W_PACKED && i != P_CODES && i != P_DENSE);
        plan->p[i] = t[i]->numel() ? plan->slot[i].ptr() : nullptr;
    }
    plan->device = dev.index();
    if (std::any_of(plan->slot, plan->slot + n, [](const Slot &s) { return s.copy.defined(); })) {
        if (capturing()) return plan;
        plan->filled.stream = c10::hip::getCurrentHIPStream(plan->device);
    }
    PlanObject *fresh = reinterpret_cast<PlanObject *>(plan_new(&PlanType, nullptr, nullptr));
    if (!fresh) throw Failure{};
    fresh->plan = plan;
    fresh->owner = module;
    const int rc = PyDict_SetItem(dict, S._host_plan, reinterpret_cast<PyObject *>(fresh));
    Py_DECREF(fresh);
    if (rc != 0) throw Failure{};
    return plan;
}

// A LayerNorm in front of a layer's stage 1, as the library takes it; `weight_copy` and `bias_copy` keep what is not the module's.
struct FusedLayerNorm {
    const float *weight, *bias;
    float eps;
    Tensor weight_copy, bias_copy;
};
// fp32 copies of its weight and bias are made once per layer and parameter version.  False: not the plain case.
bool read_fused_layernorm(Plan &plan, PyObject *ln, Refs &refs, FusedLayerNorm &out)
{
    PyObject *d = dict_of(ln);
    PyObject *params = get(d, S._parameters);
    PyObject *e = get(d, S.eps), *shape = get(d, S.normalized_shape);
    const Tensor *w = as_tensor(get(params, S.weight));
    PyObject *bo = get(params, S.bias);
    const Tensor *b = as_tensor(bo);
    if (!w || !e || !PyFloat_Check(e) || !shape || !PyTuple_Check(shape) || PyTuple_GET_SIZE(shape) != 1) return false;
    if (!b && bo != Py_None) return false;
    refs.add(get(params, S.weight));
    refs.add(bo);
    out.eps = static_cast<float>(PyFloat_AS_DOUBLE(e));
    LayerNormParams p;
    LayerNormParams *found = nullptr;
    for (auto &q : plan.ln)
        if (q.w.same(*w) && q.has_bias() == (b != nullptr) && (!b || q.b.same(*b))) found = &q;
    if (!found) {
        if (!w->is_cuda() || w->device().index() != plan.device || w->numel() != plan.K || w->dim() != 1) return false;
        if (b && (b->device() != w->device() || b->numel() != plan.K)) return false;
        p.w.set(*w, true, true);
        if (b) p.b.set(*b, true, true);
        else p.no_bias = at::zeros({plan.K}, w->options().dtype(at::kFloat).requires_grad(false));
        found = &p;
        if (!p.copied() || !capturing()) {
            if (p.copied()) p.filled.stream = c10::hip::getCurrentHIPStream(plan.device);
            if (plan.ln.size() >= 4) plan.ln.clear();        // (a layer has one LayerNorm in front of it; a bound, not a policy)
            plan.ln.push_back(std::move(p));
            found = &plan.ln.back();
        }
    }
    found->filled.settle();
    out.weight = found->weight(), out.weight_copy = found->w.copy;
    out.bias = found->bias(), out.bias_copy = found->has_bias() ? found->b.copy : found->no_bias;
    return true;
}

// ---- one on-the-fly layer -------------------------------------------------------------------------------------------
struct Layer {                   // what a call needs of an ARCQPackedLinearOnTheFly
    std::shared_ptr<Plan> plan;
    std::optional<at::ScalarType> out;      // none: a type the library does not write
    bool fp8 = false;
    float fp8_mult = 1.0f;
    bool lends = false;                     // has a _weight_buffer ...
    const Tensor *weight_buffer = nullptr, *x_hat_buffer = nullptr;       // ... that may be no tensor
};

// The power of two inside a layer's FP8 weights (reads the metadata back to the host: once per layer and set of buffers).
float fp8_multiplier(Plan &p, PyObject *dict)
{
    const bool tracked = p.slot[W_CB].tracked && p.slot[W_CENTER].tracked && p.slot[W_SCALE].tracked && p.slot[W_SUM].tracked;
    if (tracked && !std::isnan(p.fp8_mult)) return static_cast<float>(p.fp8_mult);
    PyObject *b = get(dict, S._buffers);
    PyObject *r = PyObject_CallFunctionObjArgs(g_fp8_multiplier, get(b, S.weight_codebook), get(b, S.weight_center), get(b, S.weight_scale),
                                               get(b, S.weight_code_sum), nullptr);
    if (!r) throw Failure{};
    const double mult = PyFloat_AsDouble(r);
    Py_DECREF(r);
    if (PyErr_Occurred()) throw Failure{};
    p.fp8_mult = mult;
    return static_cast<float>(mult);
}

bool read_layer(PyObject *module, Refs &refs, Layer &l)
{
    PyObject *dict;
    l.plan = plan_of(module, Kind::OnTheFly, refs, dict);
    if (!l.plan) return false;
    PyObject *od = get(dict, S.out_dtype);
    if (od == g_half) l.out = at::kHalf;
    else if (od == g_float) l.out = at::kFloat;
    PyObject *wo = get(dict, S._weight_buffer);
    l.lends = wo && wo != Py_None;
    PyObject *xo = get(dict, S._x_hat_buffer);
    if ((l.weight_buffer = as_tensor(wo))) refs.add(wo);
    if ((l.x_hat_buffer = as_tensor(xo))) refs.add(xo);
    l.fp8 = is_true(get(dict, S.fp8_operands));
    if (l.fp8 && l.plan->gs == 64) l.fp8_mult = fp8_multiplier(*l.plan, dict);
    return true;
}
// A buffer lent for scratch of `numel` fp16 values on the device of x.
bool lent(const Tensor *buffer, int64_t numel, const Tensor &x)
{
    return buffer && buffer->is_cuda() && f16(*buffer) && buffer->is_contiguous() && buffer->numel() >= numel &&
           buffer->device() == x.device();
}

struct Options {
    const FusedLayerNorm *layernorm = nullptr;
    const Layer *next = nullptr;
    bool gelu = false, x_is_xhat = false;
    const Tensor *residual = nullptr;
};

// Whether `a`'s launch may end with the stage 1 of `b` (ARCQPackedLinearOnTheFly.can_quantize_for).
bool can_quantize(const Layer &la, const Layer &lb, int64_t rows)
{
    const Plan &a = *la.plan, &b = *lb.plan;
    if (la.fp8 || lb.fp8 || rows <= 0 || a.gs != 64 || b.gs != 64 || a.bits != b.bits || b.K != a.N || a.N % 64 != 0 || a.K % 64 != 0 ||
        la.out != at::kHalf)
        return false;
    if (rows < 512) return a.K <= 1536;
    if (!la.lends || rows * a.K * 2 >= (int64_t(1) << 32)) return false;
    return strncmp(arcq_linear_otf_ws_kernel(rows, a.N, a.K, 1), "otf_rows", 8) != 0;
}

// ---- prepared operands: stage 1 and the weights in one launch, then the product -----------------------------------------
struct Weights {                 // w_hat of one layer inside a scratch tensor
    void *ptr;
    bool row_major;
    bool fp8 = false;            // FP8 operands: rows of Kp = K rounded up to 128 bytes, times `mult`
    float mult = 1.0f;
};
int64_t operand_row_bytes(int64_t K, bool fp8) { return fp8 ? (K + 127) / 128 * 128 : 2 * K; }
// Fields of arcq_prepare_args for a layer's own tensors.
void set_weights(arcq_prepare_weights &w, const Plan &p, const Weights &out)
{
    w.packed = static_cast<const uint8_t *>(p.p[W_PACKED]);
    w.codebook = static_cast<const float *>(p.p[W_CB]), w.center = static_cast<const float *>(p.p[W_CENTER]);
    w.scale = static_cast<const float *>(p.p[W_SCALE]), w.code_sum = static_cast<const float *>(p.p[W_SUM]);
    w.w_hat = out.ptr, w.N = p.N, w.K = p.K, w.row_major = out.row_major ? 1 : 0;
    w.w_mult = out.mult;
}
void run_prepare(const Tensor &x, int64_t rows, const Plan &first, const FusedLayerNorm *ln, void *x_hat, const Weights &w_first,
                 const Plan *second, const Weights *w_second, void *stream)
{
    arcq_prepare_args a = {};
    a.x_dtype = code_of(x);
    a.bits = static_cast<int32_t>(first.bits);
    a.fp8 = w_first.fp8 ? 1 : 0;
    a.rows = rows, a.K = first.K;
    a.x = x.const_data_ptr();
    if (ln) a.ln_weight = ln->weight, a.ln_bias = ln->bias, a.ln_eps = ln->eps;
    a.thresholds = static_cast<const float *>(first.p[A_THR]), a.codebook = static_cast<const float *>(first.p[A_CB]);
    a.x_hat = x_hat;
    if (w_first.ptr) set_weights(a.weights[0], first, w_first);
    if (second) set_weights(a.weights[1], *second, *w_second);
    check(arcq_prepare(&a, stream));
}
void run_product(const Plan &p, int64_t rows, const void *x_hat, const Weights &w, const Tensor *residual, bool gelu, const Plan *next,
                 void *y, int y_dtype, void *stream)
{
    arcq_linear_prepared_args a = {};
    a.y_dtype = y_dtype;
    a.activation = gelu ? ARCQ_ACT_GELU : ARCQ_ACT_NONE;
    a.w_row_major = w.row_major ? 1 : 0;
    a.M = rows, a.N = p.N, a.K = p.K;
    a.x_hat = x_hat, a.w_hat = w.ptr;
    a.bias = static_cast<const float *>(p.p[W_BIAS]);
    if (residual) a.residual = residual->const_data_ptr();
    if (next) {
        a.next_thresholds = static_cast<const float *>(next->p[A_THR]), a.next_codebook = static_cast<const float *>(next->p[A_CB]);
        a.next_bits = static_cast<int32_t>(next->bits);
    }
    a.y = y;
    a.fp8 = w.fp8 ? 1 : 0, a.w_mult = w.mult;
    check(arcq_linear_prepared(&a, stream));
}
// (packed codes that are not 16-byte aligned are left to the kernels and entry points that take them, or say why not)
bool can_prepare(const Plan &p, int64_t rows)
{
    return aligned16(p.p[W_PACKED]) && p.gs == 64 && p.K % 64 == 0 && (p.N % 32 == 0 || rows >= 512) &&
           rows * p.K < (int64_t(1) << 31) && p.N * p.K < (int64_t(1) << 31) && rows < (int64_t(1) << 26);
}
// Whether one layer call runs as prepare + product.  Below 512 rows from K = 768 on (up to 512 inputs the one-launch kernel
// is 1 us faster: 7.7 against 9.6 us at 197 x 384 x 384; 12.9 against 11.1 at 2 304 x 768, 43 against 16.5 with a LayerNorm
// at 3 072 x 1 024); above wherever no one-launch kernel would run (1 000 rows: 384 -> 1 152 13.1 -> 12.0 us, 1 024 -> 3 072
// 32 -> 19, 4 096 -> 1 024 51 -> 32).
bool prepare_pays(const Plan &p, const Tensor &x, int64_t rows, bool has_ws, bool layernorm)
{
    if (!can_prepare(p, rows) || !aligned16(x) || (layernorm && p.K > 2048)) return false;
    if (rows < 512) return p.K >= 768;
    return !(f16(x) && has_ws && strncmp(arcq_linear_otf_ws_kernel(rows, p.N, p.K, 1), "otf_rows", 8) == 0);
}

bool takes(const Layer &l, const Tensor &x)
{
    return here(x) && x.device().index() == l.plan->device && x.is_contiguous() && (f16(x) || f32(x)) && x.dim() >= 1 &&
           x.size(-1) == l.plan->K && x.numel() != 0;
}

// One layer's launches; nullopt before the first where the call is not the plain case.  No Python object is touched.
std::optional<Tensor> run_layer(const Layer &l, const Tensor &x, const Options &o)
{
    if (!takes(l, x) || !l.out) return std::nullopt;
    const Plan *plan = l.plan.get();
    const int64_t K = plan->K, N = plan->N, m = x.numel() / K;
    const at::ScalarType out_type = *l.out;
    const bool extras = o.layernorm || o.gelu || o.residual || o.next || o.x_is_xhat;
    if (extras) {
        if (l.fp8 || plan->gs != 64 || K % 64 != 0) return std::nullopt;
        if (o.layernorm && K > 1024 && (K > 1536 || m >= 512)) return std::nullopt;
        if (o.x_is_xhat && (!f16(x) || o.layernorm)) return std::nullopt;
        if (o.residual && (o.residual->scalar_type() != out_type || o.residual->device() != x.device() ||
                           !o.residual->is_contiguous() || o.residual->numel() != m * N || o.residual->size(-1) != N))
            return std::nullopt;
    }
    if (o.next && (o.next->plan->device != plan->device || !can_quantize(l, *o.next, m))) return std::nullopt;
    at::DimVector sizes(x.sizes());
    sizes.back() = N;
    void *stream = stream_of(x);
    const auto *p = plan->p;
    auto fp = [&](int i) { return static_cast<const float *>(p[i]); };
    if (l.fp8) {
        if (plan->gs != 64) return std::nullopt;
        const int64_t kp = (K + 127) / 128 * 128;
        Tensor x8 = empty({m * kp}, at::kByte, x.device()), w8 = empty({N * kp}, at::kByte, x.device());
        Tensor y = empty(sizes, out_type, x.device());
        check(arcq_linear_otf_fp8(x.const_data_ptr(), code_of(x), fp(A_THR), fp(A_CB), static_cast<const uint8_t *>(p[W_PACKED]),
                                  fp(W_CB), fp(W_CENTER), fp(W_SCALE), fp(W_SUM), fp(W_BIAS), l.fp8_mult,
                                  x8.mutable_data_ptr(), w8.mutable_data_ptr(), y.mutable_data_ptr(), code_of(y), m, N, K,
                                  static_cast<int>(plan->bits), stream));
        return y;
    }
    if (l.lends && !lent(l.weight_buffer, N * K, x)) return std::nullopt;
    const Tensor *w_ws = l.lends ? l.weight_buffer : nullptr;
    if (!o.next && !o.x_is_xhat && prepare_pays(*plan, x, m, w_ws != nullptr, o.layernorm != nullptr)) {
        // (x_hat and w_hat in one scratch tensor; w_hat first: 512-byte runs stay aligned)
        const bool use_ws = w_ws != nullptr && aligned16(*w_ws);
        Tensor scratch = empty({(use_ws ? 0 : N * K) + m * K}, at::kHalf, x.device());
        char *base = static_cast<char *>(scratch.mutable_data_ptr());
        const Weights w{use_ws ? w_ws->mutable_data_ptr() : base, arcq_prepared_row_major(m, N, K) != 0};
        void *x_hat = use_ws ? base : base + N * K * 2;
        Tensor y = empty(sizes, out_type, x.device());
        run_prepare(x, m, *plan, o.layernorm, x_hat, w, nullptr, nullptr, stream);
        run_product(*plan, m, x_hat, w, o.residual, o.gelu, nullptr, y.mutable_data_ptr(), code_of(y), stream);
        return y;
    }
    Tensor own_ws;
    const Tensor *ws = l.x_hat_buffer;
    if (!lent(ws, x.numel(), x)) {
        own_ws = empty({x.numel()}, at::kHalf, x.device());
        ws = &own_ws;
    }
    Tensor y = empty(sizes, out_type, x.device());
    if (!extras) {
        check(arcq_linear_otf_ws(x.const_data_ptr(), code_of(x), fp(A_THR), fp(A_CB), static_cast<const uint8_t *>(p[W_PACKED]),
                                 fp(W_CB), fp(W_CENTER), fp(W_SCALE), fp(W_SUM), fp(W_BIAS), ws->mutable_data_ptr(),
                                 w_ws ? w_ws->mutable_data_ptr() : nullptr, y.mutable_data_ptr(), code_of(y), m, N, K,
                                 static_cast<int>(plan->bits), static_cast<int>(plan->gs), stream));
        return y;
    }
    arcq_linear_ex_args a = {};
    a.struct_size = sizeof(a);
    a.x_dtype = code_of(x);
    a.y_dtype = code_of(y);
    a.bits = static_cast<int>(plan->bits);
    a.group_size = static_cast<int>(plan->gs);
    a.M = m, a.N = N, a.K = K;
    a.x = x.const_data_ptr();
    if (o.layernorm) {
        a.producer = ARCQ_PRODUCER_LAYERNORM;
        a.ln_weight = o.layernorm->weight, a.ln_bias = o.layernorm->bias, a.ln_eps = o.layernorm->eps;
    }
    if (o.x_is_xhat) a.producer = ARCQ_PRODUCER_XHAT;
    a.activation = o.gelu ? ARCQ_ACT_GELU : ARCQ_ACT_NONE;
    a.a_thresholds = fp(A_THR), a.a_codebook = fp(A_CB), a.packed_w = static_cast<const uint8_t *>(p[W_PACKED]);
    a.w_codebook = fp(W_CB), a.w_center = fp(W_CENTER), a.w_scale = fp(W_SCALE), a.w_code_sum = fp(W_SUM), a.bias = fp(W_BIAS);
    if (o.residual) a.residual = o.residual->const_data_ptr();
    if (o.next) {
        a.next_a_thresholds = static_cast<const float *>(o.next->plan->p[A_THR]);
        a.next_a_codebook = static_cast<const float *>(o.next->plan->p[A_CB]);
    }
    a.x_hat_ws = ws->mutable_data_ptr();
    a.w_hat_ws = w_ws ? w_ws->mutable_data_ptr() : nullptr;
    a.y = y.mutable_data_ptr();
    check(arcq_linear_otf_ex(&a, stream));
    return y;
}

// ---- whole block ----------------------------------------------------------------------------------------------------
bool no_hooks(PyObject *dict)      // calling the module would run its class's forward and nothing else
{
    if (!dict || get(dict, S.forward)) return false;
    for (PyObject *n : {S._forward_hooks, S._forward_pre_hooks, S._backward_hooks, S._backward_pre_hooks}) {
        PyObject *h = get(dict, n);
        if (!h || !PyDict_Check(h) || PyDict_Size(h) != 0) return false;
    }
    return true;
}
bool no_global_hooks()
{
    PyObject *d = PyModule_GetDict(g_torch_module);
    for (PyObject *n : {S._global_forward_hooks, S._global_forward_pre_hooks, S._global_backward_hooks, S._global_backward_pre_hooks}) {
        PyObject *h = get(d, n);
        if (!h || !PyDict_Check(h) || PyDict_Size(h) != 0) return false;
    }
    return true;
}
inline bool is_type(PyObject *o, PyObject *type) { return o && reinterpret_cast<PyObject *>(Py_TYPE(o)) == type; }

std::optional<Tensor> attention_call(const Tensor &qkv, int64_t heads, float scale)
{
    if (!here(qkv) || !f16(qkv) || qkv.dim() != 3 || !qkv.is_contiguous()) return std::nullopt;
    const int64_t b = qkv.size(0), n = qkv.size(1), c = qkv.size(2) / 3;
    if (qkv.size(2) != 3 * c || c != 64 * heads) return std::nullopt;
    Tensor out = empty({b, n, c}, at::kHalf, qkv.device());
    check(arcq_attention_fwd(qkv.const_data_ptr(), out.mutable_data_ptr(), b, n, heads, 64, scale, stream_of(qkv)));
    return out;
}

Tensor mix(const Tensor &qkv, int64_t heads, bool own)      // Attention.mix
{
    const int64_t b = qkv.size(0), n = qkv.size(1), c = qkv.size(2) / 3;
    if (own && c == 64 * heads && n <= 256) {
        auto y = attention_call(qkv, heads, 0.125f);
        if (y) return *y;
    }
    const auto t = qkv.reshape({b, n, 3, heads, c / heads}).permute({2, 0, 3, 1, 4});
    return at::scaled_dot_product_attention(t.select(0, 0), t.select(0, 1), t.select(0, 2)).transpose(1, 2).reshape({b, n, c});
}

struct LayerNorm {               // an nn.LayerNorm as torch runs it
    std::optional<Tensor> weight, bias;
    int64_t n = 0;
    double eps = 0;
    Tensor operator()(const Tensor &x) const { return at::layer_norm(x, {n}, weight, bias, eps); }
};
bool read_layernorm(PyObject *d, LayerNorm &out)
{
    PyObject *params = get(d, S._parameters), *e = get(d, S.eps), *shape = get(d, S.normalized_shape);
    PyObject *wo = get(params, S.weight), *bo = get(params, S.bias);
    if (!e || !PyFloat_Check(e) || !shape || !PyTuple_Check(shape) || PyTuple_GET_SIZE(shape) != 1 || !wo || !bo) return false;
    const Tensor *w = as_tensor(wo), *b = as_tensor(bo);
    if ((!w && wo != Py_None) || (!b && bo != Py_None)) return false;
    if (w) out.weight = *w;
    if (b) out.bias = *b;
    out.n = PyLong_AsLongLong(PyTuple_GET_ITEM(shape, 0));
    out.eps = PyFloat_AS_DOUBLE(e);
    return true;
}

// A block on prepared operands: [LayerNorm + stage 1, weights of qkv and proj] -> qkv -> attention ending with proj's stage 1
// -> proj + skip -> [LayerNorm + stage 1, weights of fc1 and fc2] -> fc1 + GELU + fc2's stage 1 -> fc2 + skip: seven launches.
//   fused == false: the LayerNorms are torch's (own launches); everything else that is folded into the products (skips, GELU,
//                   fc2's stage 1) gives the bits of the separate kernels anyway
//   fp8:            FP8 operands.  LayerNorms as torch runs them: that is what the layers do one by one, and a network of
//                   quantizers does not forgive another order of summation (one changed bit is 10 % of the logits 12 blocks on)
//   attention that the library's kernel does not run (or is not to): torch's, then stage 1 of proj as a launch of its own
struct BlockParts {
    int64_t heads;
    bool own;                    // attention on the library's kernel where it serves the shape
    bool fused, fp8;
    Layer qkv, proj, fc1, fc2;
    LayerNorm norm1, norm2;                  // as torch runs them: not fused, or FP8 operands
    FusedLayerNorm fused1, fused2;           // inside qkv's and fc1's launches
};
std::optional<Tensor> block_prepared(const BlockParts &k, const Tensor &x, int64_t rows)
{
    const Plan &pq = *k.qkv.plan, &pp = *k.proj.plan, &pf1 = *k.fc1.plan, &pf2 = *k.fc2.plan;
    const int64_t b = x.size(0), n = x.size(1), C = x.size(2);
    const bool fp8 = k.fp8, fuse_ln = k.fused && !fp8;
    const bool own_attention = k.own && n <= 256 && C == 64 * k.heads;
    if ((fuse_ln && C > 2048) || pf1.N % 64 != 0 || !aligned16(x)) return std::nullopt;      // (x is also proj's residual)
    for (const Plan *p : {&pq, &pp, &pf1, &pf2})
        if (!can_prepare(*p, rows) || p->bits != pq.bits) return std::nullopt;
    // Not where the one-launch kernels are at their best (one 64-row tile on most compute units, short rows).  With the LayerNorms
    // inside, hidden rows of four times the width and lent weight buffers, the block is three launches there, the last of them proj and
    // the whole MLP.  Forwards of twelve blocks against the seven launches, us: K = 192 6 501 rows 709 / 693, 6 698 706 / 716, 7 092
    // 714 / 739; K = 256 6 698 837 / 827, 7 092 837 / 836, 7 486 846 / 854, 8 668 857 / 1 019; K = 384 8 668 1 299 / 1 300, 8 865
    // 1 306 / 1 317, 10 244 1 341 / 1 429; K = 768 10 047 3 168 / 3 096, 10 244 3 179 / 3 181, 10 638 3 198 / 3 255, 10 835 3 205 / 3 569;
    // with more row tiles than compute units the seven win (a block of DeiT-Tiny at 19 700 rows 99 against 112).  Hidden rows of another
    // width, five launches: 9 000 rows (DeiT-S as five launches at 12 608 rows 1 625 us a forward against 1 939, at 6 304 1 353 -> 1 262).
    // Without lent buffers every layer call would be two launches; the seven are faster at every width (12 608 rows, six blocks: K = 192
    // 498 us against 577, 256 600 / 682, 384 889 / 970, 768 1 974 / 2 298).
    // With torch's LayerNorms and GELU those kernels run only on lent weight buffers, and win later and only beside torch's
    // attention: 10 638 rows DeiT-S 2 311 us against 2 264 here, DeiT-B 4 498 / 4 406, 11 032 rows 2 318 / 2 439 and 4 607 / 4 879,
    // 12 608 rows 2 399 / 2 564 and 4 892 / 5 147; without lent buffers (two launches a layer) 2 667 / 2 590 and 5 207 / 5 178, with
    // the library's attention, which takes proj's stage 1 along, 2 285 / 2 263 and 4 740 / 4 679, with more than one tile on a
    // compute unit (DeiT-Tiny, 17 730 rows) 2 287 / 2 201.
    if (!fp8 && strncmp(arcq_linear_otf_ws_kernel(rows, pq.N, C, 1), "otf_rows", 8) == 0) {
        const bool lends = k.qkv.lends && k.proj.lends && k.fc1.lends && k.fc2.lends;
        const bool alone = lends && (pf1.N == 4 * C ? arcq_mlp_otf_pays(rows, C, pf1.N) != 0 : rows > 9000);
        if (fuse_ln ? alone : lends && !own_attention && rows > 10800 && rows <= 16384) return std::nullopt;
    }
    Tensor t = fuse_ln ? x : k.norm1(x);
    void *stream = stream_of(x);
    auto layout = [&](const Plan &p) { return arcq_prepared_row_major(rows, p.N, p.K) != 0; };
    auto weight_bytes = [&](const Plan &p) { return p.N * operand_row_bytes(p.K, fp8); };
    const int64_t wq = weight_bytes(pq), wp = weight_bytes(pp), w1 = weight_bytes(pf1), w2 = weight_bytes(pf2);
    // Scratch from the layers' lent buffers where they have room, else from the allocator.  Two weights are in use at a time, and
    // fc1 reads its x_hat while it writes fc2's: of a pair that shares a buffer one lies elsewhere (fc1's x_hat where qkv was).
    auto scratch = [&](const Tensor *buffer, int64_t bytes) {
        return lent(buffer, (bytes + 1) / 2, x) && aligned16(*buffer) ? *buffer : empty({bytes}, at::kByte, x.device());
    };
    auto at_byte = [](const Tensor &t, int64_t i) { return static_cast<char *>(t.mutable_data_ptr()) + i; };
    const Tensor w_attn = scratch(k.qkv.weight_buffer, wq + wp), xh = scratch(k.qkv.x_hat_buffer, rows * operand_row_bytes(C, fp8));
    const Tensor wide = scratch(k.fc2.x_hat_buffer, rows * operand_row_bytes(pf2.K, fp8));         // fc1's quantized output
    const Tensor w_fc1 = scratch(k.fc1.weight_buffer, w1), w_fc2 = empty({w2}, at::kByte, x.device());
    Tensor qkv = empty({b, n, pq.N}, at::kHalf, x.device());
    Tensor x1 = empty(x.sizes(), at::kHalf, x.device()), y = empty(x.sizes(), at::kHalf, x.device());
    const Weights hq{at_byte(w_attn, 0), layout(pq), fp8, k.qkv.fp8_mult}, hp{at_byte(w_attn, wq), layout(pp), fp8, k.proj.fp8_mult},
                  h1{at_byte(w_fc1, 0), arcq_prepared_quant_row_major(rows, pf1.N, pf1.K, fp8 ? 1 : 0) != 0, fp8, k.fc1.fp8_mult}, h2{at_byte(w_fc2, 0), layout(pf2), fp8, k.fc2.fp8_mult};
    run_prepare(t, rows, pq, fuse_ln ? &k.fused1 : nullptr, xh.mutable_data_ptr(), hq, &pp, &hp, stream);
    run_product(pq, rows, xh.const_data_ptr(), hq, nullptr, false, nullptr, qkv.mutable_data_ptr(), ARCQ_F16, stream);
    if (own_attention) {
        check((fp8 ? arcq_attention_quant_fp8_fwd : arcq_attention_quant_fwd)(qkv.const_data_ptr(), static_cast<const float *>(pp.p[A_THR]),
            static_cast<const float *>(pp.p[A_CB]), static_cast<int>(pp.bits), xh.mutable_data_ptr(), b, n, k.heads, 64, 0.125f, stream));
    } else {
        const Tensor a = as_operand(mix(qkv, k.heads, false));        // (bf16 under autocast to that type)
        run_prepare(a, rows, pp, nullptr, xh.mutable_data_ptr(), Weights{nullptr, false, fp8}, nullptr, nullptr, stream);
    }
    run_product(pp, rows, xh.const_data_ptr(), hp, &x, false, nullptr, x1.mutable_data_ptr(), ARCQ_F16, stream);
    t = fuse_ln ? x1 : k.norm2(x1);
    run_prepare(t, rows, pf1, fuse_ln ? &k.fused2 : nullptr, qkv.mutable_data_ptr(), h1, &pf2, &h2, stream);
    run_product(pf1, rows, qkv.const_data_ptr(), h1, nullptr, true, &pf2, wide.mutable_data_ptr(), ARCQ_F16, stream);
    run_product(pf2, rows, wide.const_data_ptr(), h2, &x1, false, nullptr, y.mutable_data_ptr(), ARCQ_F16, stream);
    return y;
}

// The block's second half, x + fc2(GELU(fc1(LayerNorm(x)))), in one launch; nullopt before it where that does not serve or pay.
// With `attn`, attention's output, x + proj(attn) takes the place of x, in the same launch.
std::optional<Tensor> run_mlp(const Layer &fc1, const Layer &fc2, const FusedLayerNorm &ln, const Tensor &x, const Layer *proj = nullptr,
                              const Tensor *attn = nullptr)
{
    const Plan &p1 = *fc1.plan, &p2 = *fc2.plan;
    const int64_t rows = x.numel() / p1.K;
    if (!arcq_mlp_otf_pays(rows, p1.K, p1.N) || !lent(fc1.weight_buffer, p1.N * p1.K, x)) return std::nullopt;
    if (!takes(fc1, x) || !f16(x) || p2.K != p1.N || p2.N != p1.K || !aligned16(x) || !aligned16(ln.weight) || !aligned16(ln.bias))
        return std::nullopt;
    if (attn && (!takes(*proj, *attn) || !f16(*attn) || attn->numel() != x.numel() || proj->plan->K != p1.K || proj->plan->N != p1.K ||
                 !aligned16(*attn)))
        return std::nullopt;
    const Layer *const layers[3] = {&fc1, &fc2, proj};
    const int count = attn ? 3 : 2;
    for (int i = 0; i < count; ++i) {
        const Layer &l = *layers[i];
        if (!l.lends || l.fp8 || l.out != at::kHalf || l.plan->gs != 64 || l.plan->bits != p1.bits || l.plan->device != p1.device) return std::nullopt;
    }
    const Tensor others = empty({p2.N * p2.K + (attn ? p1.K * p1.K : 0)}, at::kHalf, x.device());      // (layers may share the buffer they lend)
    char *const w2 = static_cast<char *>(others.mutable_data_ptr());
    void *const ws[3] = {fc1.weight_buffer->mutable_data_ptr(), w2, w2 + 2 * p2.N * p2.K};
    arcq_mlp_args a = {};
    a.bits = static_cast<int32_t>(p1.bits);
    a.eps = 1.0e-6f, a.ln_eps = ln.eps;
    a.M = rows, a.K = p1.K, a.H = p1.N;
    a.x = x.const_data_ptr();
    a.attn = attn ? attn->const_data_ptr() : nullptr;
    a.ln_weight = ln.weight, a.ln_bias = ln.bias;
    arcq_mlp_layer *const l[3] = {&a.fc1, &a.fc2, &a.proj};
    for (int i = 0; i < count; ++i) {
        const auto *p = layers[i]->plan->p;
        auto fp = [&](int j) { return static_cast<const float *>(p[j]); };
        if (reinterpret_cast<uintptr_t>(p[W_PACKED]) % 4 != 0 || reinterpret_cast<uintptr_t>(ws[i]) % 128 != 0) return std::nullopt;
        *l[i] = arcq_mlp_layer{fp(A_THR), fp(A_CB), static_cast<const uint8_t *>(p[W_PACKED]), fp(W_CB), fp(W_CENTER), fp(W_SCALE), fp(W_SUM),
                               fp(W_BIAS), ws[i]};
    }
    Tensor y = empty(x.sizes(), at::kHalf, x.device());
    a.y = y.mutable_data_ptr();
    const int rc = arcq_mlp_otf(&a, stream_of(x));
    if (rc == ARCQ_ERR_UNSUPPORTED) return std::nullopt;      // (nothing launched: no counter left, or a device that holds fewer workgroups)
    check(rc);
    return y;
}

// One transformer block (vit.Block.forward), both of its forms.  No Python object is touched.
std::optional<Tensor> run_block(const BlockParts &k, const Tensor &x, bool chain)
{
    const int64_t rows = x.size(0) * x.size(1);
    if (k.fused) {
        if (chain) {
            auto whole = block_prepared(k, x, rows);
            if (whole) return whole;
        }
        if (k.fp8) return std::nullopt;
        Options o1;
        o1.layernorm = &k.fused1;
        auto t = run_layer(k.qkv, x, o1);
        if (!t) return std::nullopt;
        const Tensor a = as_operand(mix(*t, k.heads, k.own));
        if (chain) {
            auto y = run_mlp(k.fc1, k.fc2, k.fused2, x, &k.proj, &a);
            if (y) return y;
        }
        Options o2;
        o2.residual = &x;
        auto x1 = run_layer(k.proj, a, o2);
        if (!x1) return std::nullopt;
        if (chain) {
            auto y = run_mlp(k.fc1, k.fc2, k.fused2, *x1);
            if (y) return y;
        }
        Options o3, o4;
        o3.layernorm = &k.fused2;
        o3.gelu = true;
        if (chain && can_quantize(k.fc1, k.fc2, rows)) {
            o3.next = &k.fc2;
            o4.x_is_xhat = true;
        }
        auto h = run_layer(k.fc1, *x1, o3);
        if (!h) return std::nullopt;
        o4.residual = &*x1;
        return run_layer(k.fc2, *h, o4);
    }
    bool plain = f16(x) && x.size(2) % 64 == 0 && k.fc2.plan->K % 64 == 0;
    for (const Layer *l : {&k.qkv, &k.proj, &k.fc1, &k.fc2}) plain = plain && !l->fp8 && l->out == at::kHalf;
    // The skip connections of a default block carry gradients and tangents, torch's additions below record them.  (The packed layers
    // pass none, and a fused block never did.)
    plain = plain && !(c10::GradMode::is_enabled() && x.requires_grad()) && !x._fw_grad(0).defined();
    if (plain) {
        auto whole = block_prepared(k, x, rows);
        if (whole) return whole;
    }
    auto q = run_layer(k.qkv, as_operand(k.norm1(x)), Options{});
    if (!q) return std::nullopt;
    auto a = run_layer(k.proj, as_operand(mix(*q, k.heads, k.own)), Options{});
    if (!a) return std::nullopt;
    const Tensor x1 = at::add(x, *a);
    auto h = run_layer(k.fc1, as_operand(k.norm2(x1)), Options{});
    if (!h) return std::nullopt;
    auto y = run_layer(k.fc2, at::gelu(*h), Options{});
    if (!y) return std::nullopt;
    return at::add(x1, *y);
}

// nullopt before anything has been launched where a module is not the plain case
std::optional<Tensor> block_call(PyObject *block, const Tensor &x)
{
    PyObject *d = dict_of(block);
    PyObject *mods = get(d, S._modules);
    if (!mods || x.dim() != 3 || !here(x) || !x.is_contiguous() || x.numel() == 0 || !no_global_hooks()) return std::nullopt;
    PyObject *attn = get(mods, S.attn), *mlp = get(mods, S.mlp), *n1 = get(mods, S.norm1), *n2 = get(mods, S.norm2);
    if (!is_type(attn, g_attention_type) || !is_type(mlp, g_mlp_type) || !is_type(n1, g_layernorm_type) || !is_type(n2, g_layernorm_type))
        return std::nullopt;
    PyObject *ad = dict_of(attn), *md = dict_of(mlp), *d1 = dict_of(n1), *d2 = dict_of(n2);
    PyObject *am = get(ad, S._modules), *mm = get(md, S._modules);
    PyObject *qkv = get(am, S.qkv), *proj = get(am, S.proj), *fc1 = get(mm, S.fc1), *fc2 = get(mm, S.fc2), *act = get(mm, S.act);
    for (PyObject *l : {qkv, proj, fc1, fc2})
        if (!is_type(l, g_layer_type) || !no_hooks(dict_of(l))) return std::nullopt;
    if (!is_type(act, g_gelu_type) || get(ad, S.mix)) return std::nullopt;
    PyObject *approx = get(dict_of(act), S.approximate);
    if (!approx || !PyUnicode_Check(approx) || PyUnicode_Compare(approx, S.none) != 0) return std::nullopt;
    Refs refs;                   // (reading flags and FP8 metadata may run Python code)
    for (PyObject *o : {attn, mlp, n1, n2, qkv, proj, fc1, fc2, act}) refs.add(o);
    BlockParts k;
    if (!get_int(ad, S.num_heads, k.heads) || k.heads <= 0) return std::nullopt;
    k.own = is_true(get(ad, S.own_kernel));
    k.fused = is_true(get(d, S.fuse_elementwise));
    const bool chain = k.fused && is_true(get(d, S.chain_mlp));
    if (!k.fused)
        for (PyObject *dd : {ad, md, d1, d2, dict_of(act)})
            if (!no_hooks(dd)) return std::nullopt;
    if (!read_layer(qkv, refs, k.qkv) || !read_layer(proj, refs, k.proj) || !read_layer(fc1, refs, k.fc1) || !read_layer(fc2, refs, k.fc2))
        return std::nullopt;
    const Plan &pq = *k.qkv.plan, &pp = *k.proj.plan, &pf1 = *k.fc1.plan, &pf2 = *k.fc2.plan;
    const int64_t c = x.size(2), rows = x.size(0) * x.size(1);
    if (pq.K != c || pq.N != 3 * c || pp.K != c || pp.N != c || pf1.K != c || pf2.K != pf1.N || pf2.N != c || c % k.heads != 0)
        return std::nullopt;
    k.fp8 = k.fused && k.qkv.fp8;
    if (k.fused) {
        for (const Layer *l : {&k.qkv, &k.proj, &k.fc1, &k.fc2})
            if (l->fp8 != k.fp8 || l->out != at::kHalf || l->plan->gs != 64) return std::nullopt;
        if (!f16(x) || c > (rows >= 512 ? 1024 : 1536) || c % 64 != 0 || pf2.K % 64 != 0) return std::nullopt;
    }
    if (k.fused && !k.fp8) {
        if (!read_fused_layernorm(*k.qkv.plan, n1, refs, k.fused1) || !read_fused_layernorm(*k.fc1.plan, n2, refs, k.fused2))
            return std::nullopt;
    } else if (!read_layernorm(d1, k.norm1) || !read_layernorm(d2, k.norm2)) {
        return std::nullopt;
    }
    NoGil released;
    return run_block(k, x, chain);
}

// ---- Python entry points ----------------------------------------------------------------------------------------------
template <typename F>
PyObject *guarded(F &&f)
{
    try {
        return f();
    } catch (const Failure &) {
        return nullptr;
    } catch (const std::exception &) {
        torch::translate_exception_to_python(std::current_exception());       // OutOfMemoryError and its like keep their types
        return nullptr;
    }
}
PyObject *none() { Py_RETURN_NONE; }
PyObject *wrap(std::optional<Tensor> &&t)
{
    if (!t) return none();
    return THPVariable_Wrap(std::move(*t));
}

// layer_forward(module, x, layernorm, gelu, residual, next, x_is_xhat)
PyObject *py_layer_forward(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        const Tensor *x = n == 7 ? as_tensor(args[1]) : nullptr;
        if (!x) return none();
        Refs refs;
        Layer layer, next;
        FusedLayerNorm ln;
        Options o;
        o.gelu = is_true(args[3]);
        o.x_is_xhat = is_true(args[6]);
        if (args[4] != Py_None && !(o.residual = as_tensor(args[4]))) return none();
        if (!read_layer(args[0], refs, layer) || !takes(layer, *x)) return none();
        if (args[2] != Py_None) {
            if (!is_type(args[2], g_layernorm_type) || !read_fused_layernorm(*layer.plan, args[2], refs, ln)) return none();
            o.layernorm = &ln;
        }
        if (args[5] != Py_None) {
            if (!PyObject_TypeCheck(args[5], reinterpret_cast<PyTypeObject *>(g_layer_type)) || !read_layer(args[5], refs, next)) return none();
            o.next = &next;
        }
        std::optional<Tensor> y;
        {
            NoGil released;
            y = run_layer(layer, *x, o);
        }
        return wrap(std::move(y));
    });
}

PyObject *py_block_forward(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        const Tensor *x = n == 2 ? as_tensor(args[1]) : nullptr;
        return x ? wrap(block_call(args[0], *x)) : none();
    });
}

// attention(qkv, heads, scale)
PyObject *py_attention(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        const Tensor *q = n == 3 ? as_tensor(args[0]) : nullptr;
        if (!q || !PyLong_CheckExact(args[1]) || !PyFloat_CheckExact(args[2])) return none();
        const int64_t heads = PyLong_AsLongLong(args[1]);
        const float scale = static_cast<float>(PyFloat_AS_DOUBLE(args[2]));
        std::optional<Tensor> y;
        {
            NoGil released;
            y = attention_call(*q, heads, scale);
        }
        return wrap(std::move(y));
    });
}

// patch_embed(img, weight, bias or None, cls, pos)
PyObject *py_patch_embed(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        if (n != 5) return none();
        const Tensor *t[5];
        for (int i = 0; i < 5; ++i) {
            t[i] = as_tensor(args[i]);
            if (!t[i] && (i != 2 || args[i] != Py_None)) return none();
            if (t[i] && (!here(*t[i]) || !f16(*t[i]) || !t[i]->is_contiguous())) return none();
        }
        const Tensor &img = *t[0], &w = *t[1];
        if (img.dim() != 4 || img.size(1) != 3 || w.dim() != 4 || w.size(1) != 3 || w.size(2) != 16 || w.size(3) != 16) return none();
        const int64_t b = img.size(0), h = img.size(2), wd = img.size(3), N = w.size(0), tokens = 1 + (h / 16) * (wd / 16);
        if (b == 0 || N % 32 != 0 || h % 16 != 0 || wd % 16 != 0 || t[3]->numel() != N || t[4]->numel() != tokens * N ||
            (t[2] && t[2]->numel() != N))
            return none();
        Tensor out;
        {
            NoGil released;
            out = empty({b, tokens, N}, at::kHalf, img.device());
            check(arcq_patch_embed_fwd(img.const_data_ptr(), w.const_data_ptr(), t[2] ? t[2]->const_data_ptr() : nullptr,
                                       t[3]->const_data_ptr(), t[4]->const_data_ptr(), out.mutable_data_ptr(), b, h, wd, 16, N,
                                       stream_of(img)));
        }
        return THPVariable_Wrap(std::move(out));
    });
}

struct Quantized { Tensor codes, center, scale, sum; };
bool quantize_args_ok(const Tensor &x, const Tensor &thr, const Tensor &cb, int64_t bits, int64_t gs)
{
    return (bits == 2 || bits == 3 || bits == 4) && gs > 0 && here(x) && x.dim() == 2 && f32(x) && x.is_contiguous() &&
           x.size(1) % gs == 0 && thr.device() == x.device() && cb.device() == x.device() && f32(thr) && f32(cb) &&
           thr.is_contiguous() && cb.is_contiguous() && cb.numel() == (int64_t(1) << bits) && thr.numel() == cb.numel() - 1;
}
Quantized quantize(const Tensor &x, const float *thr, const float *cb, int64_t bits, int64_t gs, bool bytes)
{
    const int64_t rows = x.size(0), cols = x.size(1), groups = cols / gs;
    Quantized q;
    q.codes = empty({rows, bytes ? cols : (cols * bits + 7) / 8}, at::kByte, x.device());
    q.center = empty({rows, groups}, at::kFloat, x.device());
    q.scale = empty({rows, groups}, at::kFloat, x.device());
    q.sum = empty({rows, groups}, at::kFloat, x.device());
    uint8_t *codes = static_cast<uint8_t *>(q.codes.mutable_data_ptr());
    check(arcq_act_quant(x.const_data_ptr(), ARCQ_F32, thr, cb, bytes ? nullptr : codes, bytes ? codes : nullptr,
                         static_cast<float *>(q.center.mutable_data_ptr()), static_cast<float *>(q.scale.mutable_data_ptr()),
                         static_cast<float *>(q.sum.mutable_data_ptr()), nullptr, ARCQ_F32, rows, cols, static_cast<int>(bits),
                         static_cast<int>(gs), 1.0e-6f, stream_of(x)));
    return q;
}

// quantize(x, thresholds, codebook, bits, group_size, bytes) -> [codes, center, scale, code_sum]
PyObject *py_quantize(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        if (n != 6 || !PyLong_CheckExact(args[3]) || !PyLong_CheckExact(args[4])) return none();
        const Tensor *x = as_tensor(args[0]), *thr = as_tensor(args[1]), *cb = as_tensor(args[2]);
        const int64_t bits = PyLong_AsLongLong(args[3]), gs = PyLong_AsLongLong(args[4]);
        if (!x || !thr || !cb || !quantize_args_ok(*x, *thr, *cb, bits, gs)) return none();
        const bool bytes = is_true(args[5]);
        Quantized q;
        {
            NoGil released;
            q = quantize(*x, fptr(*thr), fptr(*cb), bits, gs, bytes);
        }
        PyObject *list = PyList_New(4);
        if (!list) return nullptr;
        PyList_SET_ITEM(list, 0, THPVariable_Wrap(std::move(q.codes)));
        PyList_SET_ITEM(list, 1, THPVariable_Wrap(std::move(q.center)));
        PyList_SET_ITEM(list, 2, THPVariable_Wrap(std::move(q.scale)));
        PyList_SET_ITEM(list, 3, THPVariable_Wrap(std::move(q.sum)));
        return list;
    });
}

enum class Format { Fused, DequantGemm, Packed, Bytes };
// ARCQPackedLinear's launches in one of its runtime formats; nullopt before the first where the call is not the plain case.
std::optional<Tensor> run_packed(const Plan &plan, Format fmt, const Tensor &x)
{
    const int64_t K = plan.K, N = plan.N, m = x.numel() / K;
    const int bits = static_cast<int>(plan.bits), gs = static_cast<int>(plan.gs);
    const auto *p = plan.p;
    auto fp = [&](int i) { return static_cast<const float *>(p[i]); };
    auto up = [&](int i) { return static_cast<const uint8_t *>(p[i]); };
    at::DimVector sizes(x.sizes());
    sizes.back() = N;
    void *stream = stream_of(x);
    if (fmt == Format::Fused) {
        if (gs != 64 || !aligned16(x)) return std::nullopt;             // (the general path's stage 1 takes any alignment)
        Tensor y = empty(sizes, at::kFloat, x.device());
        if (prepare_pays(plan, x, m, false, false)) {
            Tensor scratch = empty({N * K + m * K}, at::kHalf, x.device());
            char *base = static_cast<char *>(scratch.mutable_data_ptr());
            const Weights w{base, arcq_prepared_row_major(m, N, K) != 0};
            run_prepare(x, m, plan, nullptr, base + N * K * 2, w, nullptr, nullptr, stream);
            run_product(plan, m, base + N * K * 2, w, nullptr, false, nullptr, y.mutable_data_ptr(), ARCQ_F32, stream);
            return y;
        }
        Tensor x_hat = empty({m * K}, at::kHalf, x.device());
        check(arcq_linear_otf_ws(x.const_data_ptr(), ARCQ_F32, fp(A_THR), fp(A_CB), up(W_PACKED), fp(W_CB), fp(W_CENTER), fp(W_SCALE),
                                 fp(W_SUM), fp(W_BIAS), x_hat.mutable_data_ptr(), nullptr, y.mutable_data_ptr(), ARCQ_F32, m, N, K, bits,
                                 64, stream));
        return y;
    }
    if (fmt == Format::DequantGemm) {
        const Slot &dense = plan.slot[P_DENSE];
        if (gs != 64 || dense.type != at::kHalf || dense.numel() != N * K) return std::nullopt;
        Tensor x_hat = empty({m * K}, at::kHalf, x.device()), y = empty(sizes, at::kFloat, x.device());
        check(arcq_act_quant_blocked(x.const_data_ptr(), ARCQ_F32, fp(A_THR), fp(A_CB), x_hat.mutable_data_ptr(), m, K, bits, 1.0e-6f, stream));
        check(arcq_linear_fused_blocked(x_hat.const_data_ptr(), up(W_PACKED), fp(W_CB), fp(W_CENTER), fp(W_SCALE), fp(W_SUM), fp(W_BIAS),
                                        const_cast<void *>(dense.ptr()), 1, y.mutable_data_ptr(), ARCQ_F32, m, N, K, bits, 64, stream));
        return y;
    }
    const bool bytes = fmt == Format::Bytes;
    const Slot &table = plan.slot[P_TABLE];
    if (table.sizes.size() != 2 || table.sizes[0] != table.sizes[1]) return std::nullopt;
    if (plan.slot[A_CB].numel() != table.sizes[0] || plan.slot[W_CB].numel() != table.sizes[0]) return std::nullopt;
    if (bytes && (!p[P_CODES] || plan.slot[P_CODES].numel() != N * K || plan.slot[P_CODES].type != at::kByte)) return std::nullopt;
    const Tensor x2 = x.dim() == 2 ? x : x.view({m, K});
    Quantized q = quantize(x2, fp(A_THR), fp(A_CB), bits, gs, bytes);
    Tensor y = empty(sizes, at::kFloat, x.device());
    arcq_linear_index_args a = {};
    a.x_codes = bptr(q.codes), a.x_center = fptr(q.center), a.x_scale = fptr(q.scale), a.x_code_sum = fptr(q.sum);
    a.w_codes = up(bytes ? P_CODES : W_PACKED), a.w_center = fp(W_CENTER), a.w_scale = fp(W_SCALE), a.w_code_sum = fp(W_SUM);
    a.product_table = fp(P_TABLE), a.a_codebook = fp(A_CB), a.w_codebook = fp(W_CB), a.bias = fp(W_BIAS);
    a.y = static_cast<float *>(y.mutable_data_ptr());
    a.rows = m, a.out_features = N, a.in_features = K;
    a.bits = bytes ? 0 : bits, a.group_size = gs, a.levels = static_cast<int>(table.sizes[0]);
    check(arcq_linear_index(&a, stream));
    return y;
}

// packed_forward(module, x): ARCQPackedLinear in its four runtime formats, group size 64 or (index-space formats) any
PyObject *py_packed_forward(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        const Tensor *x = n == 2 ? as_tensor(args[1]) : nullptr;
        if (!x) return none();
        Refs refs;
        PyObject *dict;
        const auto plan = plan_of(args[0], Kind::Packed, refs, dict);
        if (!plan || !here(*x) || x->device().index() != plan->device || !f32(*x) || !x->is_contiguous() || x->dim() < 1 ||
            x->size(-1) != plan->K || x->numel() == 0)
            return none();
        PyObject *fo = get(dict, S.runtime_code_format);
        const char *name = fo && PyUnicode_Check(fo) ? PyUnicode_AsUTF8(fo) : nullptr;
        if (!name) return none();
        Format fmt;
        if (strcmp(name, "hip_fused") == 0) fmt = Format::Fused;
        else if (strcmp(name, "dequant_gemm") == 0) fmt = Format::DequantGemm;
        else if (strcmp(name, "packed") == 0) fmt = Format::Packed;
        else if (strcmp(name, "u8") == 0) fmt = Format::Bytes;
        else return none();
        std::optional<Tensor> y;
        {
            NoGil released;
            y = run_packed(*plan, fmt, *x);
        }
        return wrap(std::move(y));
    });
}

Tensor run_patches(const Plan &plan, const Tensor &x)
{
    const int64_t b = x.size(0), hp = x.size(2) / 16, wp = x.size(3) / 16, m = b * hp * wp, N = plan.N, K = 768;
    const int bits = static_cast<int>(plan.bits);
    auto fp = [&](int i) { return static_cast<const float *>(plan.p[i]); };
    void *stream = stream_of(x);
    Tensor y = empty({b, hp, wp, N}, x.scalar_type(), x.device());
    if (can_prepare(plan, m)) {
        Tensor scratch = empty({N * K + m * K}, at::kHalf, x.device());
        char *base = static_cast<char *>(scratch.mutable_data_ptr());
        const Weights w{base, arcq_prepared_row_major(m, N, K) != 0};
        void *x_hat = base + N * K * 2;
        arcq_prepare_weights pwt = {};
        set_weights(pwt, plan, w);
        check(arcq_prepare_patches(x.const_data_ptr(), code_of(x), fp(A_THR), fp(A_CB), x_hat, b, 3, x.size(2), x.size(3), 16, bits, 1.0e-6f,
                                   &pwt, stream));
        run_product(plan, m, x_hat, w, nullptr, false, nullptr, y.mutable_data_ptr(), code_of(y), stream);
        return y.permute({0, 3, 1, 2});
    }
    Tensor rows = empty({m * K}, at::kHalf, x.device());
    check(arcq_act_quant_patches(x.const_data_ptr(), code_of(x), fp(A_THR), fp(A_CB), rows.mutable_data_ptr(), b, 3, x.size(2), x.size(3), 16,
                                 bits, 1.0e-6f, 0, stream));
    check(arcq_linear_fused(rows.const_data_ptr(), static_cast<const uint8_t *>(plan.p[W_PACKED]), fp(W_CB), fp(W_CENTER), fp(W_SCALE),
                            fp(W_SUM), fp(W_BIAS), y.mutable_data_ptr(), code_of(y), m, N, K, bits, 64, stream));
    return y.permute({0, 3, 1, 2});
}

// patch_conv_forward(module, img): ARCQPackedPatchConv with 16 x 16 patches of three channels, group sizes 3 and 64
PyObject *py_patch_conv_forward(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    return guarded([&]() -> PyObject * {
        const Tensor *xp = n == 2 ? as_tensor(args[1]) : nullptr;
        if (!xp) return none();
        const Tensor &x = *xp;
        Refs refs;
        PyObject *dict;
        const auto plan = plan_of(args[0], Kind::Conv, refs, dict);
        int64_t ags, c;
        PyObject *ks = get(dict, S.kernel_size);
        if (!plan || plan->gs != 64 || !get_int(dict, S.act_group_size, ags) || ags != 3 || !get_int(dict, S.in_channels, c) || c != 3 ||
            !ks || !PyTuple_Check(ks) || PyTuple_GET_SIZE(ks) != 2 || PyLong_AsLong(PyTuple_GET_ITEM(ks, 0)) != 16 ||
            PyLong_AsLong(PyTuple_GET_ITEM(ks, 1)) != 16)
            return none();
        if (!here(x) || x.device().index() != plan->device || (!f16(x) && !f32(x)) || !x.is_contiguous() || x.dim() != 4 ||
            x.size(1) != 3 || x.size(2) % 16 != 0 || x.size(3) % 16 != 0 || x.numel() == 0)
            return none();
        Tensor y;
        {
            NoGil released;
            y = run_patches(*plan, x);
        }
        return THPVariable_Wrap(std::move(y));
    });
}

// register_types(layer, attention, mlp, gelu, layernorm, torch.nn.modules.module, fp8_weight_multiplier); None leaves an entry as it is
PyObject *py_register_types(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    PyObject **const to[7] = {&g_layer_type, &g_attention_type, &g_mlp_type, &g_gelu_type, &g_layernorm_type, &g_torch_module,
                              &g_fp8_multiplier};
    for (Py_ssize_t i = 0; i < n && i < 7; ++i) {
        if (args[i] == Py_None) continue;
        Py_INCREF(args[i]);
        Py_XDECREF(*to[i]);
        *to[i] = args[i];
    }
    g_half = reinterpret_cast<PyObject *>(torch::getTHPDtype(at::kHalf));       // (they live as long as torch)
    g_float = reinterpret_cast<PyObject *>(torch::getTHPDtype(at::kFloat));
    Py_RETURN_NONE;
}

#define FASTCALL(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f))
PyMethodDef methods[] = {
    {"layer_forward", FASTCALL(py_layer_forward), METH_FASTCALL, "one ARCQPackedLinearOnTheFly call, or None"},
    {"block_forward", FASTCALL(py_block_forward), METH_FASTCALL, "one transformer block, or None"},
    {"attention", FASTCALL(py_attention), METH_FASTCALL, "arcq_attention_fwd, or None"},
    {"patch_embed", FASTCALL(py_patch_embed), METH_FASTCALL, "arcq_patch_embed_fwd, or None"},
    {"quantize", FASTCALL(py_quantize), METH_FASTCALL, "arcq_act_quant to codes and metadata, or None"},
    {"packed_forward", FASTCALL(py_packed_forward), METH_FASTCALL, "one ARCQPackedLinear call, or None"},
    {"patch_conv_forward", FASTCALL(py_patch_conv_forward), METH_FASTCALL, "one ARCQPackedPatchConv call, or None"},
    {"register_types", FASTCALL(py_register_types), METH_FASTCALL, "classes whose instances are recognised"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_arcq_host", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__arcq_host(void)
{
#define X(n) S.n = PyUnicode_InternFromString(#n);
    ARCQ_NAMES(X)
#undef X
    PlanType.tp_name = "arcq_vit_amd._arcq_host.Plan";
    PlanType.tp_basicsize = sizeof(PlanObject);
    PlanType.tp_flags = Py_TPFLAGS_DEFAULT;
    PlanType.tp_new = plan_new;
    PlanType.tp_dealloc = plan_dealloc;
    PlanType.tp_methods = plan_methods;
    if (PyType_Ready(&PlanType) < 0) return nullptr;
    PyObject *m = PyModule_Create(&module_def);
    if (!m) return nullptr;
    Py_INCREF(&PlanType);
    if (PyModule_AddObject(m, "Plan", reinterpret_cast<PyObject *>(&PlanType)) < 0) return nullptr;
    return m;
}
