// ternainfer_amd._native: the host path of one library call as one native function -- checks, output tensors, current
// stream, launch(es).  In Python (ctypes) that path costs 13 - 16 us a call, several times what a decode-sized launch
// takes on the device; here 2 - 3 us.  PyTorch stays what it is elsewhere in the package: the owner of device memory
// and streams.  The library is the one _lib.py loads; init() binds its entry points by name.
//
// Every function checks shapes and element counts before anything is enqueued (the C ABI takes pointers on trust) and
// raises ValueError, or TypeError where an argument is no tensor; the tensors' types and devices are the caller's business
// where linear.py does not state otherwise.  What follows the checks -- allocations, copies, launches, which may wait for the
// device -- runs without the interpreter's lock, as the same calls do from Python.
#include <dlfcn.h>

#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ops/empty.h>
#include <ATen/EmptyTensor.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <cstdarg>
#include <vector>

#include "../../include/ternaspmm.h"

namespace {

#define TERNA_ENTRY_POINTS(X)                                                                                          \
    X(bitlinear_TernaSpMM)                                                                                             \
    X(bitlinear_TernaSpMM_bf16)                                                                                        \
    X(bitlinear_TernaSpMM_bf16_decode)                                                                                 \
    X(bitlinear_TernaSpMM_bf16_prefill)                                                                                \
    X(bitlinear_TernaSpMM_packed_ws)                                                                                   \
    X(bitlinear_TernaSpMM_bf16_packed_ws)                                                                              \
    X(bitlinear_TernaSpMM_quant)                                                                                       \
    X(bitlinear_TernaSpMM_quant_packed)                                                                                \
    X(ternaspmm_quant_rows_linear)                                                                                     \
    X(ternaspmm_quant_rows_linear_packed)                                                                              \
    X(ternaspmm_qkv_rope_linear)                                                                                       \
    X(ternaspmm_prefill_attention_rows)                                                                                \
    X(ternaspmm_gate_linear)                                                                                           \
    X(ternaspmm_residual_linear)                                                                                       \
    X(ternaspmm_quant_input)                                                                                           \
    X(ternaspmm_rmsnorm_quant)                                                                                         \
    X(ternaspmm_rmsnorm_quant_ahead)                                                                                   \
    X(ternaspmm_relu2_mul_rmsnorm_quant)                                                                               \
    X(ternaspmm_relu2_mul_rmsnorm_quant_ahead)                                                                         \
    X(ternaspmm_fused_linear)                                                                                          \
    X(ternaspmm_quant_from_stats)                                                                                      \
    X(ternaspmm_rope_kv_store)                                                                                         \
    X(ternaspmm_prefill_attention)                                                                                     \
    X(ternaspmm_rope_decode_attention)                                                                                 \
    X(ternaspmm_rope_decode_attention_stats)                                                                           \
    X(ternaspmm_step_attention)                                                                                        \
    X(ternaspmm_step_attention_merge)                                                                                  \
    X(ternaspmm_attention_partial_bytes)                                                                               \
    X(ternaspmm_attention_workspace_bytes)                                                                             \
    X(ternaspmm_attention_merge)                                                                                       \
    X(ternaspmm_attention_merge_rmsnorm_quant)                                                                         \
    X(ternaspmm_row_stats_count)                                                                                       \
    X(ternaspmm_step_inputs)                                                                                           \
    X(ternaspmm_prompt_inputs)                                                                                         \
    X(ternaspmm_decode_step_bytes)                                                                                     \
    X(ternaspmm_decode_step)
struct Library {
#define X(name) decltype(&::name) name = nullptr;
    TERNA_ENTRY_POINTS(X)
#undef X
} lib;

struct Refused : std::exception {};            // a Python error is set

// From its construction to end() other Python threads run: no Python object is touched and nothing refused in between.
class Unlocked {
    PyThreadState* state = PyEval_SaveThread();

public:
    Unlocked() = default;
    Unlocked(const Unlocked&) = delete;
    ~Unlocked() { end(); }
    void end()
    {
        if (state != nullptr) PyEval_RestoreThread(state);
        state = nullptr;
    }
};

// an argument that is a tensor
const at::Tensor& tensor(PyObject* o)
{
    if (!THPVariable_CheckExact(o) && !THPVariable_Check(o)) {
        PyErr_Format(PyExc_TypeError, "expected a torch.Tensor, got %s", Py_TYPE(o)->tp_name);
        throw Refused();
    }
    return THPVariable_Unpack(o);
}
// ... or None
const at::Tensor* optional(PyObject* o) { return o == Py_None ? nullptr : &tensor(o); }

[[noreturn]] void refuse(const char* format, ...)
{
    va_list args;
    va_start(args, format);
    PyErr_FormatV(PyExc_ValueError, format, args);
    va_end(args);
    throw Refused();
}

long long integer(PyObject* o)
{
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw Refused();
    return v;
}
int integer32(PyObject* o)
{
    const long long v = integer(o);
    if (v < INT32_MIN || v > INT32_MAX) refuse("integer argument %lld out of range", v);
    return static_cast<int>(v);
}
float real(PyObject* o)
{
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw Refused();
    return static_cast<float>(v);
}

template <typename T = void>
T* data(const at::Tensor* t) { return t == nullptr ? nullptr : static_cast<T*>(t->data_ptr()); }

void check_matrix(const char* who, const at::Tensor& x)
{
    if (x.dim() != 2) refuse("%s: expected a [M, K] tensor, got %d dimensions", who, static_cast<int>(x.dim()));
    if (x.size(0) > INT32_MAX || x.size(1) > INT32_MAX) refuse("%s: tensor too large", who);
}
void check_numel(const char* who, const char* name, const at::Tensor* t, int64_t want)
{
    if (t != nullptr && t->numel() != want)
        refuse("%s: %s has %lld elements, expected %lld", who, name, static_cast<long long>(t->numel()), static_cast<long long>(want));
}
void check_weight(const char* who, const at::Tensor& packed, const at::Tensor& ws, int ws_num, int64_t n, int64_t k)
{
    if (static_cast<int64_t>(packed.numel() * packed.element_size()) < n * k / 4 || ws.numel() < ws_num)
        refuse("%s: packed weight or weight scales too small for this shape", who);
}

// The caching allocator under the device name that torch's Python side uses.
c10::Allocator* device_allocator() { return c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get(); }

// A device tensor straight from the caching allocator: torch's dispatcher costs more than the allocation (1.2 against 0.6 us).
at::Tensor make(at::IntArrayRef shape, at::ScalarType type, const at::Tensor& like)
{
    if (like.is_cuda() && like.device().index() == c10::hip::current_device())
        return at::Tensor(at::detail::empty_generic(shape, device_allocator(), c10::DispatchKeySet(c10::DispatchKey::CUDA), type, std::nullopt));
    return at::empty(shape, at::TensorOptions(type).device(like.device()));
}
terna_stream stream() { return c10::hip::getCurrentHIPStream().stream(); }

// int8 rows and their bf16 scales, for the length of one call: (rows [m][k], scales [m]) on the current device
struct QuantRows {
    c10::DataPtr held;
    int8_t* q;
    terna_bf16* s;
};
QuantRows make_quant_rows(int64_t m, int64_t k)
{
    QuantRows r{device_allocator()->allocate(m * k + 2 * m), nullptr, nullptr};     // k is even: the scales are aligned
    r.q = static_cast<int8_t*>(r.held.get());
    r.s = reinterpret_cast<terna_bf16*>(r.q + m * k);
    return r;
}

// Results: the end of an unlocked stretch.
PyObject* none(Unlocked& unlocked)
{
    unlocked.end();
    Py_RETURN_NONE;
}
PyObject* wrap(at::Tensor t, Unlocked& unlocked)
{
    unlocked.end();
    return THPVariable_Wrap(std::move(t));
}
PyObject* wrap_or_none(at::Tensor t) { return t.defined() ? THPVariable_Wrap(std::move(t)) : Py_NewRef(Py_None); }
template <typename... Ts>
PyObject* pack(Unlocked& unlocked, Ts&&... items)
{
    unlocked.end();
    PyObject* tuple = PyTuple_New(sizeof...(items));
    Py_ssize_t i = 0;
    (PyTuple_SET_ITEM(tuple, i++, wrap_or_none(std::forward<Ts>(items))), ...);
    return tuple;
}

// A module's activations: bf16 rows on the current device.  False: something the native path does not take (another type, an
// empty batch ...), linear.py goes on.
bool bf16_rows(const at::Tensor& x, int64_t* m, int64_t* k)
{
    if (!x.is_cuda() || x.scalar_type() != at::kBFloat16 || x.dim() < 1) return false;
    *k = x.size(-1);
    if (*k < 64 || x.numel() == 0 || x.device().index() != c10::hip::current_device()) return false;
    *m = x.numel() / *k;
    return *m <= INT32_MAX && *k <= INT32_MAX;
}
at::Tensor make_output(const at::Tensor& x, int64_t n)
{
    at::DimVector shape(x.sizes());
    shape.back() = n;
    return make(shape, at::kBFloat16, x);
}
void check_format(const char* who, const at::Tensor& bitmap, int64_t n, int64_t k)
{
    if (bitmap.numel() * 64 != n * k)
        refuse("%s: the weight's bitmap does not belong to a [%lld, %lld] matrix", who, static_cast<long long>(n), static_cast<long long>(k));
}

#define TERNA_FUNCTION(name, count)                                                                                    \
    PyObject* name##_body(PyObject* const* a);                                                                         \
    PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n)                                                        \
    {                                                                                                                  \
        HANDLE_TH_ERRORS                                                                                               \
        if (n != (count)) {                                                                                            \
            PyErr_Format(PyExc_TypeError, #name ": %d arguments expected", (count));                                   \
            return nullptr;                                                                                            \
        }                                                                                                              \
        try {                                                                                                          \
            return name##_body(a);                                                                                     \
        } catch (const Refused&) {                                                                                     \
            return nullptr;                                                                                            \
        }                                                                                                              \
        END_HANDLE_TH_ERRORS                                                                                           \
    }                                                                                                                  \
    PyObject* name##_body(PyObject* const* a)

// (x, packed | None, bitmap, tile offsets, median offsets, signs, ws, ws_num, out_features, workspace | None): SpBitLinear -- quantise
// the rows, then the int8 linear on the repacked weight or on the reference format.  None: x is not for this path.
TERNA_FUNCTION(bit_linear, 10)
{
    const at::Tensor &x = tensor(a[0]), &bitmap = tensor(a[2]), &offsets = tensor(a[3]), &median = tensor(a[4]), &signs = tensor(a[5]), &ws = tensor(a[6]);
    const at::Tensor *packed = optional(a[1]), *workspace = optional(a[9]);
    const int ws_num = integer32(a[7]);
    const int64_t n = integer32(a[8]);
    int64_t m, k;
    if (!bf16_rows(x, &m, &k) || k > 8192) Py_RETURN_NONE;
    if (packed != nullptr) check_weight("SpBitLinear", *packed, ws, ws_num, n, k);
    else check_format("SpBitLinear", bitmap, n, k);
    Unlocked unlocked;
    const at::Tensor rows = x.contiguous();
    at::Tensor out = make_output(x, n);
    const terna_stream st = stream();
    if (m <= 8) {                       // a few rows: both steps in one launch
        const int done = packed != nullptr ? lib.bitlinear_TernaSpMM_quant_packed(data<terna_bf16>(&rows), data(packed), data<terna_bf16>(&out),
                                                                                  data<terna_bf16>(&ws), ws_num, m, n, k, st)
                                           : lib.bitlinear_TernaSpMM_quant(data<terna_bf16>(&rows), data<uint64_t>(&bitmap), data<int>(&offsets),
                                                                           data<uint16_t>(&median), data<uint32_t>(&signs), data<terna_bf16>(&out),
                                                                           data<terna_bf16>(&ws), ws_num, m, n, k, st);
        if (done) return wrap(std::move(out), unlocked);
    }
    {                                   // ... or of more rows, where one round of workgroups covers the matrix
        const int done = packed != nullptr ? lib.ternaspmm_quant_rows_linear_packed(data<terna_bf16>(&rows), data(packed), data<terna_bf16>(&out),
                                                                                    data<terna_bf16>(&ws), ws_num, m, n, k, st)
                                           : lib.ternaspmm_quant_rows_linear(data<terna_bf16>(&rows), data<uint64_t>(&bitmap), data<int>(&offsets),
                                                                             data<uint16_t>(&median), data<uint32_t>(&signs), data<terna_bf16>(&out),
                                                                             data<terna_bf16>(&ws), ws_num, m, n, k, st);
        if (done) return wrap(std::move(out), unlocked);
    }
    QuantRows q = make_quant_rows(m, k);
    if (lib.ternaspmm_quant_input(data<terna_bf16>(&rows), q.q, q.s, m, k, st) != 0) return none(unlocked);
    if (packed != nullptr)
        lib.bitlinear_TernaSpMM_packed_ws(q.q, data(packed), data<terna_bf16>(&out), q.s, data<terna_bf16>(&ws), ws_num, m, n, k, 0,
                                          data(workspace), workspace != nullptr ? workspace->numel() : 0, st);
    else
        lib.bitlinear_TernaSpMM(q.q, data<uint64_t>(&bitmap), data<int>(&offsets), data<uint16_t>(&median), data<uint32_t>(&signs),
                                data<terna_bf16>(&out), q.s, data<terna_bf16>(&ws), ws_num, m, n, k, 7, data<int32_t>(workspace), st);
    return wrap(std::move(out), unlocked);
}

// (x, bitmap, tile offsets, median offsets, signs, scale, ws_num, out_features, route 0 auto / 1 decode / 2 prefill)
TERNA_FUNCTION(bit_linear_bf16, 9)
{
    const at::Tensor &x = tensor(a[0]), &bitmap = tensor(a[1]), &offsets = tensor(a[2]), &median = tensor(a[3]), &signs = tensor(a[4]), &scale = tensor(a[5]);
    const int ws_num = integer32(a[6]), route = integer32(a[8]);
    const int64_t n = integer32(a[7]);
    int64_t m, k;
    if (!bf16_rows(x, &m, &k)) Py_RETURN_NONE;
    check_format("TernaInfer_linear_bf16", bitmap, n, k);
    Unlocked unlocked;
    const at::Tensor rows = x.contiguous();
    at::Tensor out = make_output(x, n);
    const auto fn = route == 1 ? lib.bitlinear_TernaSpMM_bf16_decode : route == 2 ? lib.bitlinear_TernaSpMM_bf16_prefill : lib.bitlinear_TernaSpMM_bf16;
    fn(data<terna_bf16>(&rows), data<uint64_t>(&bitmap), data<int>(&offsets), data<uint16_t>(&median), data<uint32_t>(&signs),
       data<terna_bf16>(&out), data<float>(&scale), ws_num, m, n, k, 1, nullptr, stream());
    return wrap(std::move(out), unlocked);
}

// (x bf16 [..., K]) -> (int8 [..., K], bf16 [..., 1]), or None
TERNA_FUNCTION(quant_input, 1)
{
    const at::Tensor& x = tensor(a[0]);
    int64_t m, k;
    if (!bf16_rows(x, &m, &k)) Py_RETURN_NONE;
    Unlocked unlocked;
    const at::Tensor rows = x.contiguous();
    at::DimVector shape(x.sizes());
    at::Tensor q = make(shape, at::kChar, x);
    shape.back() = 1;
    at::Tensor s = make(shape, at::kBFloat16, x);
    if (lib.ternaspmm_quant_input(data<terna_bf16>(&rows), data<int8_t>(&q), data<terna_bf16>(&s), m, k, stream()) != 0) return none(unlocked);
    return pack(unlocked, std::move(q), std::move(s));
}

// (x int8 [M, K], s, packed, ws, ws_num, out_features, workspace | None)
TERNA_FUNCTION(linear_packed, 7)
{
    const char* who = "TernaInfer_linear_packed";
    const at::Tensor &x = tensor(a[0]), &s = tensor(a[1]), &packed = tensor(a[2]), &ws = tensor(a[3]);
    const at::Tensor* workspace = optional(a[6]);
    const int ws_num = integer32(a[4]);
    const int64_t n = integer32(a[5]);
    check_matrix(who, x);
    const int64_t m = x.size(0), k = x.size(1);
    check_numel(who, "s", &s, m);
    check_weight(who, packed, ws, ws_num, n, k);
    Unlocked unlocked;
    const at::Tensor rows = x.contiguous(), scales = s.contiguous();
    at::Tensor out = make({m, n}, at::kBFloat16, x);
    lib.bitlinear_TernaSpMM_packed_ws(data<int8_t>(&rows), data(&packed), data<terna_bf16>(&out), data<terna_bf16>(&scales), data<terna_bf16>(&ws),
                                      ws_num, m, n, k, 0, data(workspace), workspace != nullptr ? workspace->numel() : 0, stream());
    return wrap(std::move(out), unlocked);
}

// (x bf16 [M, K], packed, scale fp32, ws_num, out_features, workspace | None)
TERNA_FUNCTION(linear_bf16_packed, 6)
{
    const char* who = "bf16 linear on a packed weight";
    const at::Tensor &x = tensor(a[0]), &packed = tensor(a[1]), &scale = tensor(a[2]);
    const at::Tensor* workspace = optional(a[5]);
    const int ws_num = integer32(a[3]);
    const int64_t n = integer32(a[4]);
    check_matrix(who, x);
    const int64_t m = x.size(0), k = x.size(1);
    check_weight(who, packed, scale, ws_num, n, k);
    Unlocked unlocked;
    const at::Tensor rows = x.contiguous();
    at::Tensor out = make({m, n}, at::kBFloat16, x);
    lib.bitlinear_TernaSpMM_bf16_packed_ws(data<terna_bf16>(&rows), data(&packed), data<terna_bf16>(&out), data<float>(&scale), ws_num, m, n, k, 0,
                                           data(workspace), workspace != nullptr ? workspace->numel() : 0, stream());
    return wrap(std::move(out), unlocked);
}

// (x, weight, eps, residual | None, quant) -> (xq, s, h) or (y, None, h)
TERNA_FUNCTION(rmsnorm_quant, 5)
{
    const char* who = "rmsnorm_quant";
    const at::Tensor &x = tensor(a[0]), &weight = tensor(a[1]);
    const at::Tensor* residual = optional(a[3]);
    const float eps = real(a[2]);
    check_matrix(who, x);
    const int64_t m = x.size(0), k = x.size(1);
    check_numel(who, "residual", residual, m * k);
    check_numel(who, "weight", &weight, k);
    const bool quant = PyObject_IsTrue(a[4]);
    Unlocked unlocked;
    const at::Tensor rows = x.contiguous();
    at::Tensor added, h = rows, q, s;
    if (residual != nullptr) {
        added = residual->contiguous();
        h = make({m, k}, at::kBFloat16, x);
    }
    q = make({m, k}, quant ? at::kChar : at::kBFloat16, x);
    if (quant) s = make({m}, at::kBFloat16, x);
    lib.ternaspmm_rmsnorm_quant(data<terna_bf16>(&rows), residual != nullptr ? data<terna_bf16>(&added) : nullptr,
                                residual != nullptr ? data<terna_bf16>(&h) : nullptr, data<terna_bf16>(&weight), eps,
                                quant ? nullptr : data<terna_bf16>(&q), quant ? data<int8_t>(&q) : nullptr, quant ? data<terna_bf16>(&s) : nullptr, m, k,
                                stream());
    return pack(unlocked, std::move(q), std::move(s), std::move(h));             // (x itself where it is neither added to nor copied)
}

// (x13, weight, eps, quant) -> (xq, s) or (y, None)
TERNA_FUNCTION(relu2_mul_rmsnorm_quant, 4)
{
    const char* who = "relu2_mul_rmsnorm_quant";
    const at::Tensor &x = tensor(a[0]), &weight = tensor(a[1]);
    const float eps = real(a[2]);
    check_matrix(who, x);
    const int64_t m = x.size(0), f = x.size(1) / 2;
    check_numel(who, "weight", &weight, f);
    const bool quant = PyObject_IsTrue(a[3]);
    Unlocked unlocked;
    const at::Tensor rows = x.contiguous();
    at::Tensor q = make({m, f}, quant ? at::kChar : at::kBFloat16, x), s;
    if (quant) s = make({m}, at::kBFloat16, x);
    lib.ternaspmm_relu2_mul_rmsnorm_quant(data<terna_bf16>(&rows), data<terna_bf16>(&weight), eps, quant ? nullptr : data<terna_bf16>(&q),
                                          quant ? data<int8_t>(&q) : nullptr, quant ? data<terna_bf16>(&s) : nullptr, m, f, stream());
    return pack(unlocked, std::move(q), std::move(s));
}

void check_stats(const char* who, const at::Tensor& stats, int64_t m)
{
    if (stats.scalar_type() != at::kFloat || stats.dim() != 3 || stats.size(0) != m || stats.size(2) != 2 || !stats.is_contiguous())
        refuse("%s: stats must be a contiguous fp32 [M, count, 2] tensor", who);
}

// (h, stats, norm_weight, eps) -> (xq, s)
TERNA_FUNCTION(quant_from_stats, 4)
{
    const char* who = "quant_from_stats";
    const at::Tensor &h = tensor(a[0]), &stats = tensor(a[1]), &weight = tensor(a[2]);
    const float eps = real(a[3]);
    check_matrix(who, h);
    const int64_t m = h.size(0), k = h.size(1);
    check_numel(who, "norm_weight", &weight, k);
    check_stats(who, stats, m);
    Unlocked unlocked;
    const at::Tensor rows = h.contiguous();
    at::Tensor q = make({m, k}, at::kChar, h), s = make({m}, at::kBFloat16, h);
    const int rc = lib.ternaspmm_quant_from_stats(data<terna_bf16>(&rows), data<float>(&stats), stats.size(1), data<terna_bf16>(&weight), eps,
                                                  data<int8_t>(&q), data<terna_bf16>(&s), m, k, stream());
    unlocked.end();
    if (rc != 0) refuse("%s: unsupported shape M=%d K=%d", who, static_cast<int>(m), static_cast<int>(k));
    return pack(unlocked, std::move(q), std::move(s));
}

// (x, norm_weight | None, eps, packed, ws, ws_num, out_features, in_features, stats | None, attention splits (0: none), head_dim,
//  quantised | None, epilogue, residual | None, next_norm_weight | None, want_raw, publish) -> the five tensors of
// linear.fused_linear, or None where the library does not take the combination
PyObject* chained_linear(const char* who, bool own_stats, PyObject* const* a)
{
    const at::Tensor &x = tensor(a[0]), &packed = tensor(a[3]), &ws = tensor(a[4]);
    const at::Tensor *weight = optional(a[1]), *stats = optional(a[8]), *quantised = optional(a[11]), *residual = optional(a[13]), *next_weight = optional(a[14]);
    const int64_t n = integer32(a[6]), k = integer32(a[7]);
    ternaspmm_fused_linear_desc d{};
    d.eps = real(a[2]);
    d.ws_num = integer32(a[5]);
    d.attention_splits = integer32(a[9]);
    d.head_dim = integer32(a[10]);
    d.epilogue = integer32(a[12]);
    at::Tensor rows = x, scales, stream_in, out, stats_out, raw, xq, s;
    int64_t m = 1;
    if (d.attention_splits > 0) {
        d.prologue = TERNASPMM_PROLOGUE_ATTENTION;
    } else {
        check_matrix(who, x);
        m = x.size(0);
        if (x.size(1) != k) refuse("%s: expected a [M, %lld] tensor", who, static_cast<long long>(k));
        if (quantised != nullptr) {
            d.prologue = TERNASPMM_PROLOGUE_QUANTISED;
            check_numel(who, "s", quantised, m);
            if (x.scalar_type() != at::kChar || quantised->scalar_type() != at::kBFloat16)
                refuse("%s: quantised activations are int8 with bf16 scales", who);
        } else {
            d.prologue = stats == nullptr ? TERNASPMM_PROLOGUE_NORM : own_stats ? TERNASPMM_PROLOGUE_OWN_STATS : TERNASPMM_PROLOGUE_STATS;
            check_numel(who, "norm_weight", weight, k);
        }
    }
    check_weight(who, packed, ws, d.ws_num, n, k);
    d.M = m, d.N = n, d.K = k;
    d.packed = data(&packed), d.ws = data<terna_bf16>(&ws), d.norm_weight = data<terna_bf16>(weight);
    if (stats != nullptr) {
        check_stats(who, *stats, m);
        d.stats_in = data<float>(stats), d.stats_count = stats->size(1);
    }
    const int64_t columns = d.epilogue == TERNASPMM_EPILOGUE_GATE ? n / 2 : n;
    if (d.epilogue != TERNASPMM_EPILOGUE_STORE && (next_weight == nullptr || next_weight->numel() != columns))
        refuse("%s: a producing epilogue needs the next norm's weights", who);
    if (d.epilogue == TERNASPMM_EPILOGUE_RESIDUAL) {
        if (residual == nullptr || residual->numel() != m * n || residual->scalar_type() != at::kBFloat16)
            refuse("%s: the residual epilogue needs a bf16 [M, N] stream", who);
    }
    const bool want_raw = d.epilogue == TERNASPMM_EPILOGUE_RESIDUAL && PyObject_IsTrue(a[15]), publish = PyObject_IsTrue(a[16]);

    Unlocked unlocked;
    if (d.attention_splits <= 0) rows = x.contiguous();
    d.x = data(&rows);
    if (d.prologue == TERNASPMM_PROLOGUE_QUANTISED) {
        scales = quantised->contiguous();
        d.s_in = data<terna_bf16>(&scales);
    }
    if (d.epilogue == TERNASPMM_EPILOGUE_RESIDUAL) {
        stream_in = residual->contiguous();
        d.residual = data<terna_bf16>(&stream_in);
    }
    if (want_raw) {
        raw = make({m, n}, at::kBFloat16, packed);
        d.raw_out = data<terna_bf16>(&raw);
    }
    out = make({m, columns}, at::kBFloat16, packed);
    d.out = data<terna_bf16>(&out);
    if (d.epilogue != TERNASPMM_EPILOGUE_STORE) {
        stats_out = make({m, columns / 16, 2}, at::kFloat, packed);
        d.next_norm_weight = data<terna_bf16>(next_weight), d.stats_out = data<float>(&stats_out);
    }
    if (publish) {
        xq = make({m, k}, at::kChar, packed), s = make({m}, at::kBFloat16, packed);
        d.xq_out = data<int8_t>(&xq), d.s_out = data<terna_bf16>(&s);
    }
    if (lib.ternaspmm_fused_linear(&d, stream()) < 0) return none(unlocked);
    return pack(unlocked, std::move(out), std::move(stats_out), std::move(raw), std::move(xq), std::move(s));
}

TERNA_FUNCTION(fused_linear, 17) { return chained_linear("fused_linear", false, a); }
// The same where `stats` are the rows' own (TERNASPMM_PROLOGUE_OWN_STATS).
TERNA_FUNCTION(fused_linear_own_stats, 17) { return chained_linear("fused_linear_own_stats", true, a); }

// What the attention entry points read beside a block's new rows, checked against these and each other.
struct AttentionArgs {
    const at::Tensor &cos, &sin, &pos, &ck, &cv;
    int64_t heads, head_dim, batch, kv, slots, t;
    float scale;
    int adjacent;
    bool each;                     // every sequence has its own positions

    // a: cos, sin, pos, cache_k, cache_v, heads, head_dim, scale, adjacent; qkv is [new_rows = B * T, columns = (H + 2 KV) D]
    AttentionArgs(const char* who, PyObject* const* a, int64_t new_rows, int64_t columns)
        : cos(tensor(a[0])), sin(tensor(a[1])), pos(tensor(a[2])), ck(tensor(a[3])), cv(tensor(a[4])), heads(integer32(a[5])),
          head_dim(integer32(a[6])), scale(real(a[7])), adjacent(integer32(a[8]))
    {
        if (ck.dim() != 4 || ck.sizes() != cv.sizes() || ck.size(0) < 1 || ck.size(3) != head_dim || !ck.is_contiguous() || !cv.is_contiguous())
            refuse("%s: the caches are contiguous [B, KV, S, D] tensors of one shape", who);
        batch = ck.size(0), kv = ck.size(1), slots = ck.size(2), t = new_rows / batch;
        if (t < 1 || new_rows != batch * t || columns != (heads + 2 * kv) * head_dim)
            refuse("%s: qkv does not have the shape of its caches", who);
        each = pos.dim() == 2;
        const int64_t rows = each ? batch * t : t;
        if (pos.scalar_type() != at::kLong || pos.numel() != rows || !pos.is_contiguous())
            refuse("%s: positions are a contiguous int64 [T] or [B, T] tensor", who);
        if (cos.numel() < rows * (head_dim / 2) || sin.numel() != cos.numel() || cos.scalar_type() != at::kFloat || sin.scalar_type() != at::kFloat ||
            !cos.is_contiguous() || !sin.is_contiguous())
            refuse("%s: cos / sin are contiguous fp32 rows of D / 2, one per position", who);
    }
};
// the leading arguments of those entry points
#define TERNA_ATTENTION_INPUTS(qkv, g)                                                                                 \
    qkv, data<float>(&(g).cos), data<float>(&(g).sin), data<long long>(&(g).pos), (g).each

// the new rows of an attention call
const at::Tensor& new_rows(const char* who, PyObject* o)
{
    const at::Tensor& qkv = tensor(o);
    check_matrix(who, qkv);
    if (!qkv.is_contiguous()) refuse("%s: qkv is a contiguous tensor", who);
    return qkv;
}

// (qkv, the nine of AttentionArgs, attention): RoPE and cache write of T new tokens per sequence, and with `attention` the multi-token
// attention -> bf16 [B * T, H D]; without it the rotated q [B, H, T, D]
TERNA_FUNCTION(prompt_attention, 11)
{
    const char* who = "prompt_attention";
    const at::Tensor& qkv = new_rows(who, a[0]);
    const AttentionArgs g(who, a + 1, qkv.size(0), qkv.size(1));
    const bool attention = PyObject_IsTrue(a[10]);
    Unlocked unlocked;
    at::Tensor q = make({g.batch, g.heads, g.t, g.head_dim}, at::kBFloat16, qkv);
    const terna_stream st = stream();
    lib.ternaspmm_rope_kv_store(TERNA_ATTENTION_INPUTS(data<terna_bf16>(&qkv), g), data<terna_bf16>(&q), data<terna_bf16>(&g.ck), data<terna_bf16>(&g.cv), g.batch, g.t, g.heads,
                                g.kv, g.head_dim, g.slots, g.adjacent, st);
    if (!attention) return wrap(std::move(q), unlocked);
    at::Tensor o = make({g.batch * g.t, g.heads * g.head_dim}, at::kBFloat16, qkv);
    lib.ternaspmm_prefill_attention(data<terna_bf16>(&q), data<terna_bf16>(&g.ck), data<terna_bf16>(&g.cv), data<long long>(&g.pos), g.each,
                                    data<terna_bf16>(&o), g.batch, g.t, g.heads, g.kv, g.head_dim, g.slots, g.scale, st);
    return wrap(std::move(o), unlocked);
}

// (qkv, the nine of AttentionArgs, workspace | None, norm_weight | None, partial | None, splits): RoPE, cache write and attention of one new
// token per sequence -> (out bf16 [B, H D], None); with the norm's weights (out, its partial statistics [B, H, 2]); with a
// buffer for partial results these are all that is written -> None
TERNA_FUNCTION(decode_attention, 14)
{
    const char* who = "decode_attention";
    const at::Tensor& qkv = new_rows(who, a[0]);
    const AttentionArgs g(who, a + 1, qkv.size(0), qkv.size(1));
    const at::Tensor *workspace = optional(a[10]), *weight = optional(a[11]), *partial = optional(a[12]);
    if (g.t != 1) refuse("%s: one new token per sequence", who);
    const terna_stream st = stream();
    terna_bf16 *ck = data<terna_bf16>(&g.ck), *cv = data<terna_bf16>(&g.cv);
    if (partial != nullptr) {
        const long long need = lib.ternaspmm_attention_partial_bytes(g.batch, g.heads, g.head_dim);
        if (need < 0 || static_cast<long long>(partial->numel() * partial->element_size()) < need) refuse("%s: the partial buffer is too small", who);
        const int splits = integer32(a[13]);
        Unlocked unlocked;
        const int left = lib.ternaspmm_step_attention(TERNA_ATTENTION_INPUTS(data<terna_bf16>(&qkv), g), ck, cv, data<float>(partial), splits, g.batch, g.heads, g.kv,
                                                      g.head_dim, g.slots, g.scale, g.adjacent, nullptr, nullptr, nullptr, 0, st);
        if (left != 0) {
            unlocked.end();
            refuse("%s: one to eight splits, 65536 of all heads", who);
        }
        return none(unlocked);
    }
    check_numel(who, "norm_weight", weight, g.heads * g.head_dim);
    if (weight == nullptr && workspace != nullptr &&
        static_cast<long long>(workspace->numel() * workspace->element_size()) < lib.ternaspmm_attention_workspace_bytes(g.batch, g.heads, g.head_dim))
        refuse("%s: the workspace is too small", who);
    Unlocked unlocked;
    at::Tensor o = make({g.batch, g.heads * g.head_dim}, at::kBFloat16, qkv), stats;
    if (weight != nullptr) {
        stats = make({g.batch, g.heads, 2}, at::kFloat, qkv);
        const int left = lib.ternaspmm_rope_decode_attention_stats(TERNA_ATTENTION_INPUTS(data<terna_bf16>(&qkv), g), ck, cv, data<terna_bf16>(&o), g.batch, g.heads, g.kv,
                                                                   g.head_dim, g.slots, g.scale, g.adjacent, data<terna_bf16>(weight), data<float>(&stats), st);
        unlocked.end();
        if (left != g.heads) refuse("%s: ternaspmm_rope_decode_attention_stats refused the launch", who);
    } else {
        lib.ternaspmm_rope_decode_attention(TERNA_ATTENTION_INPUTS(data<terna_bf16>(&qkv), g), ck, cv, data<terna_bf16>(&o), g.batch, g.heads, g.kv, g.head_dim, g.slots, g.scale,
                                            g.adjacent, data(workspace), st);
    }
    return pack(unlocked, std::move(o), std::move(stats));
}

// A ternary matrix of a block as four arguments: packed, ws, ws_num, out_features.
struct BlockLinear {
    const at::Tensor &packed, &ws;
    int ws_num;
    int64_t n;
    BlockLinear(const char* who, PyObject* const* a, int64_t k) : packed(tensor(a[0])), ws(tensor(a[1])), ws_num(integer32(a[2])), n(integer32(a[3]))
    {
        check_weight(who, packed, ws, ws_num, n, k);
    }
};

// (x, pending | None, cos, sin, pos, cache_k, cache_v, heads, head_dim, scale, adjacent, eps, attention workspace | (partial results, splits) | None, linear workspace | None,
//  attention_norm, attn_sub_norm, ffn_norm, ffn_sub_norm, wqkv [4], wo [4], w13 [4], w2 [4], interleaved w13 | None) -> (stream, pending; None where the stream has it): a whole block on int8
// activations with its norms as launches of their own (prompt pass, decode steps of many sequences): the nine launches and nothing
// else.  Called one by one from Python they cost 53 us of host time, more than they take on the device up to a hundred tokens.
TERNA_FUNCTION(block, 35)
{
    const char* who = "block";
    const at::Tensor& x = tensor(a[0]);
    const at::Tensor *pending = optional(a[1]), *attn_work = nullptr, *partial = nullptr, *work = optional(a[13]), *interleaved = optional(a[34]);
    int splits = 1;
    if (PyTuple_Check(a[12])) {
        if (PyTuple_GET_SIZE(a[12]) != 2) refuse("%s: (partial results, splits)", who);
        partial = &tensor(PyTuple_GET_ITEM(a[12], 0));
        splits = integer32(PyTuple_GET_ITEM(a[12], 1));
    } else {
        attn_work = optional(a[12]);
    }
    const at::Tensor *norm[4] = {&tensor(a[14]), &tensor(a[15]), &tensor(a[16]), &tensor(a[17])};
    const int64_t heads = integer32(a[7]), head_dim = integer32(a[8]);
    const float eps = real(a[11]);
    check_matrix(who, x);
    const int64_t m = x.size(0), dim = x.size(1), wide = heads * head_dim;
    const BlockLinear qkv_w(who, a + 18, dim), o_w(who, a + 22, wide), gate_w(who, a + 26, dim), down_w(who, a + 30, gate_w.n / 2);
    const int64_t ffn = gate_w.n / 2;
    if (interleaved != nullptr) check_weight(who, *interleaved, gate_w.ws, gate_w.ws_num, gate_w.n, dim);
    check_numel(who, "pending", pending, m * dim);
    check_numel(who, "attention_norm", norm[0], dim);
    check_numel(who, "attn_sub_norm", norm[1], wide);
    check_numel(who, "ffn_norm", norm[2], dim);
    check_numel(who, "ffn_sub_norm", norm[3], ffn);
    if (!x.is_contiguous() || (pending != nullptr && !pending->is_contiguous()) || x.scalar_type() != at::kBFloat16 || o_w.n != dim || down_w.n != dim)
        refuse("%s: the stream is a contiguous bf16 [M, dim] tensor, and the O and down projections return to it", who);

    const AttentionArgs g(who, a + 2, m, qkv_w.n);
    if (g.t == 1 && attn_work != nullptr && static_cast<long long>(attn_work->numel() * attn_work->element_size()) <
                                                lib.ternaspmm_attention_workspace_bytes(g.batch, heads, head_dim))
        refuse("%s: the attention workspace is too small", who);
    if (partial != nullptr && (g.t != 1 || splits < 1 || splits > 8 || g.batch * heads * splits > 65536 ||
                               static_cast<long long>(partial->numel() * partial->element_size()) < lib.ternaspmm_attention_partial_bytes(g.batch, heads, head_dim)))
        refuse("%s: split attention takes one new token, one to eight splits and a buffer that holds their results", who);

    Unlocked unlocked;
    // scratch of this call, in one piece: int8 rows and scales; then qkv, rotated queries, attention output and its projection,
    // in whose place the gate and up outputs go
    auto up = [](int64_t bytes) { return (bytes + 255) & ~int64_t{255}; };
    const int64_t q_bytes = up(m * std::max(std::max(dim, wide), ffn)), s_bytes = up(2 * m), qkv_bytes = up(2 * m * qkv_w.n), wide_bytes = up(2 * m * wide);
    const int64_t attn_bytes = qkv_bytes + 2 * wide_bytes + up(2 * m * dim);
    const c10::DataPtr held = device_allocator()->allocate(q_bytes + s_bytes + std::max(attn_bytes, up(2 * m * gate_w.n)));
    char* at_byte = static_cast<char*>(held.get());
    int8_t* xq = reinterpret_cast<int8_t*>(at_byte);
    terna_bf16* s = reinterpret_cast<terna_bf16*>(at_byte + q_bytes);
    auto rows = [&](int64_t offset) { return reinterpret_cast<terna_bf16*>(at_byte + q_bytes + s_bytes + offset); };
    terna_bf16 *qkv = rows(0), *q = rows(qkv_bytes), *o = rows(qkv_bytes + wide_bytes), *attn = rows(qkv_bytes + 2 * wide_bytes), *x13 = rows(0);

    at::Tensor mid = make({m, dim}, at::kBFloat16, x), out = make({m, dim}, at::kBFloat16, x), first;
    if (pending != nullptr) first = make({m, dim}, at::kBFloat16, x);
    const auto next = [](const BlockLinear& w, int64_t k) { return ternaspmm_next_linear{data(&w.packed), static_cast<int>(w.n), static_cast<int>(k), 0}; };
    const ternaspmm_next_linear next_qkv = next(qkv_w, dim), next_o = next(o_w, wide), next_down = next(down_w, ffn);
    ternaspmm_next_linear next_gate = next(gate_w, dim);
    if (interleaved != nullptr) next_gate.packed = data(interleaved), next_gate.gate = 1;
    const terna_bf16* in = data<terna_bf16>(&x);
    const terna_stream st = stream();
    terna_bf16 *ck = data<terna_bf16>(&g.ck), *cv = data<terna_bf16>(&g.cv);
    auto linear = [&](const BlockLinear& w, int64_t k, terna_bf16* to) {
        lib.bitlinear_TernaSpMM_packed_ws(xq, data(&w.packed), to, s, data<terna_bf16>(&w.ws), w.ws_num, m, w.n, k, 0, data(work),
                                          work != nullptr ? work->numel() : 0, st);
    };
    lib.ternaspmm_rmsnorm_quant_ahead(in, data<terna_bf16>(pending), pending != nullptr ? data<terna_bf16>(&first) : nullptr, data<terna_bf16>(norm[0]), eps, nullptr,
                                      xq, s, m, dim, &next_qkv, st);
    if (pending != nullptr) in = data<terna_bf16>(&first);
    // RoPE and the cache write in the projection's epilogue, for the attention that reads its rows
    const bool rows_in_place =
        g.t > 1 && g.adjacent && head_dim == 128 && heads == 4 * g.kv &&
        lib.ternaspmm_qkv_rope_linear(xq, data(&qkv_w.packed), qkv, s, data<terna_bf16>(&qkv_w.ws), qkv_w.ws_num, m, qkv_w.n, dim, data<float>(&g.cos),
                                      data<float>(&g.sin), data<long long>(&g.pos), g.each, ck, cv, g.t, heads, g.kv, head_dim, g.slots, st);
    if (!rows_in_place) linear(qkv_w, dim, qkv);
    if (rows_in_place) {
        if (!lib.ternaspmm_prefill_attention_rows(qkv, qkv_w.n, ck, cv, data<long long>(&g.pos), g.each, o, g.batch, g.t, heads, g.kv, head_dim, g.slots,
                                                  g.scale, st)) {
            unlocked.end();
            refuse("%s: the attention over the projection's rows refused the launch", who);
        }
    } else if (g.t > 1) {
        lib.ternaspmm_rope_kv_store(TERNA_ATTENTION_INPUTS(qkv, g), q, ck, cv, g.batch, g.t, heads, g.kv, head_dim, g.slots, g.adjacent, st);
        lib.ternaspmm_prefill_attention(q, ck, cv, data<long long>(&g.pos), g.each, o, g.batch, g.t, heads, g.kv, head_dim, g.slots, g.scale, st);
    } else if (partial != nullptr) {
        lib.ternaspmm_step_attention(TERNA_ATTENTION_INPUTS(qkv, g), ck, cv, data<float>(partial), splits, g.batch, heads, g.kv, head_dim, g.slots, g.scale, g.adjacent,
                                     nullptr, nullptr, nullptr, 0, st);
    } else {
        lib.ternaspmm_rope_decode_attention(TERNA_ATTENTION_INPUTS(qkv, g), ck, cv, o, g.batch, heads, g.kv, head_dim, g.slots, g.scale, g.adjacent,
                                            data(attn_work), st);
    }
    // the stream's sums in the epilogues of the projections that return to it, where these have one (elsewhere in the norm that follows)
    auto add_linear = [&](const BlockLinear& w, int64_t k, const terna_bf16* stream_in, terna_bf16* to) {
        return lib.ternaspmm_residual_linear(xq, data(&w.packed), to, s, data<terna_bf16>(&w.ws), w.ws_num, stream_in, m, w.n, k, data(work),
                                             work != nullptr ? work->numel() : 0, st) == 1;
    };
    if (partial == nullptr || lib.ternaspmm_step_attention_merge(data<float>(partial), splits, data<terna_bf16>(norm[1]), eps, nullptr, xq, s, g.batch, heads,
                                                                 head_dim, &next_o, st) != 0) {
        if (partial != nullptr) lib.ternaspmm_attention_merge(data<float>(partial), splits, o, g.batch, heads, head_dim, st);
        lib.ternaspmm_rmsnorm_quant_ahead(o, nullptr, nullptr, data<terna_bf16>(norm[1]), eps, nullptr, xq, s, m, wide, &next_o, st);
    }
    if (add_linear(o_w, wide, in, data<terna_bf16>(&mid))) {
        lib.ternaspmm_rmsnorm_quant_ahead(data<terna_bf16>(&mid), nullptr, nullptr, data<terna_bf16>(norm[2]), eps, nullptr, xq, s, m, dim, &next_gate, st);
    } else {
        linear(o_w, wide, attn);
        lib.ternaspmm_rmsnorm_quant_ahead(in, attn, data<terna_bf16>(&mid), data<terna_bf16>(norm[2]), eps, nullptr, xq, s, m, dim, &next_gate, st);
    }
    if (interleaved != nullptr && lib.ternaspmm_gate_linear(xq, data(interleaved), x13, s, data<terna_bf16>(&gate_w.ws), gate_w.ws_num, m, gate_w.n, dim, st)) {
        lib.ternaspmm_rmsnorm_quant_ahead(x13, nullptr, nullptr, data<terna_bf16>(norm[3]), eps, nullptr, xq, s, m, ffn, &next_down, st);
    } else {
        linear(gate_w, dim, x13);
        lib.ternaspmm_relu2_mul_rmsnorm_quant_ahead(x13, data<terna_bf16>(norm[3]), eps, nullptr, xq, s, m, ffn, &next_down, st);
    }
    if (add_linear(down_w, ffn, data<terna_bf16>(&mid), data<terna_bf16>(&out))) return pack(unlocked, std::move(out), at::Tensor());
    linear(down_w, ffn, data<terna_bf16>(&out));
    return pack(unlocked, std::move(mid), std::move(out));
}

// (packed, out_features, in_features, gate) | None: the linear behind a launch
ternaspmm_next_linear next_linear(const char* who, PyObject* o)
{
    if (o == Py_None) return ternaspmm_next_linear{};
    if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != 4) refuse("%s: the next linear is (packed, out_features, in_features, gate)", who);
    const at::Tensor& packed = tensor(PyTuple_GET_ITEM(o, 0));
    const int n = integer32(PyTuple_GET_ITEM(o, 1)), k = integer32(PyTuple_GET_ITEM(o, 2));
    if (n < 1 || k < 1 || static_cast<int64_t>(packed.numel() * packed.element_size()) < static_cast<int64_t>(n) * k / 4)
        refuse("%s: the next linear's weight is too small", who);
    return ternaspmm_next_linear{data(&packed), n, k, PyObject_IsTrue(PyTuple_GET_ITEM(o, 3))};
}

PyObject* merge_norm_quant(const char* who, bool any_splits, const ternaspmm_next_linear& next, PyObject* const* a)
{
    const at::Tensor &partial = tensor(a[0]), &weight = tensor(a[4]);
    const int splits = integer32(a[1]), heads = integer32(a[2]), head_dim = integer32(a[3]), sequences = integer32(a[6]);
    const float eps = real(a[5]);
    const int64_t k = static_cast<int64_t>(heads) * head_dim;
    const long long held = partial.numel() * partial.element_size(), need = lib.ternaspmm_attention_partial_bytes(sequences, heads, head_dim);
    if (sequences < 1 || need < 0 || held < need) refuse("partial buffer of %lld bytes does not hold %d sequences", held, sequences);
    if (weight.numel() != k || weight.scalar_type() != at::kBFloat16) refuse("%s: the norm weight is a bf16 vector of heads * head_dim elements", who);
    const bool want_output = PyObject_IsTrue(a[7]);
    Unlocked unlocked;
    at::Tensor q = make({sequences, k}, at::kChar, partial), s = make({sequences}, at::kBFloat16, partial), o;
    if (want_output) o = make({sequences, k}, at::kBFloat16, partial);
    terna_bf16* const o_out = o.defined() ? data<terna_bf16>(&o) : nullptr;
    if ((any_splits ? lib.ternaspmm_step_attention_merge(data<float>(&partial), splits, data<terna_bf16>(&weight), eps, o_out, data<int8_t>(&q), data<terna_bf16>(&s),
                                                         sequences, heads, head_dim, &next, stream())
                    : lib.ternaspmm_attention_merge_rmsnorm_quant(data<float>(&partial), splits, data<terna_bf16>(&weight), eps, o_out, data<int8_t>(&q),
                                                                  data<terna_bf16>(&s), sequences, heads, head_dim, stream())) != 0)
        return none(unlocked);
    return pack(unlocked, std::move(q), std::move(s), std::move(o));
}

// (partial, splits, heads, head_dim, norm_weight, eps, sequences, want_output) -> (xq, s, o | None), or None
TERNA_FUNCTION(attention_merge_rmsnorm_quant, 8) { return merge_norm_quant("attention_merge_rmsnorm_quant", false, ternaspmm_next_linear{}, a); }
// (..., next linear | None): the same for any split count up to eight
TERNA_FUNCTION(step_attention_merge, 9) { return merge_norm_quant("step_attention_merge", true, next_linear("step_attention_merge", a[8]), a); }

// (tokens, pos, embedding, rope_table, norm_weight) -> (x, stats, rope [2, B, half]); tokens / pos contiguous int64 vectors
TERNA_FUNCTION(step_inputs, 5)
{
    const char* who = "step_inputs";
    const at::Tensor &tokens = tensor(a[0]), &pos = tensor(a[1]), &embedding = tensor(a[2]), &table = tensor(a[3]), &weight = tensor(a[4]);
    check_matrix(who, embedding);
    const int64_t b = tokens.numel(), v = embedding.size(0), k = embedding.size(1);
    if (table.dim() != 3 || table.size(1) != 2 || tokens.scalar_type() != at::kLong || pos.scalar_type() != at::kLong || (pos.numel() != 1 && pos.numel() != b) ||
        table.scalar_type() != at::kFloat || embedding.scalar_type() != at::kBFloat16 || !embedding.is_contiguous() || !table.is_contiguous())
        refuse("%s: tokens / pos int64, embedding bf16 [V, K] and rope_table fp32 [S, 2, half] contiguous", who);
    check_numel(who, "norm_weight", &weight, k);
    const int count = lib.ternaspmm_row_stats_count(k);
    if (count < 1) refuse("%s: unsupported K=%d", who, static_cast<int>(k));
    Unlocked unlocked;
    const at::Tensor ids = tokens.contiguous(), at_slot = pos.contiguous();         // (copies only where a caller passed a strided view)
    const int64_t slots = table.size(0), half = table.size(2);
    at::Tensor x = make({b, k}, at::kBFloat16, embedding), stats = make({b, count, 2}, at::kFloat, embedding), rope = make({2, b, half}, at::kFloat, embedding);
    const int left = lib.ternaspmm_step_inputs(data<long long>(&ids), data<long long>(&at_slot), pos.numel() == b && b > 1, data<terna_bf16>(&embedding), v, k,
                                               data<float>(&table), slots, half, data<terna_bf16>(&weight), data<terna_bf16>(&x), data<float>(&stats),
                                               data<float>(&rope), b, stream());
    unlocked.end();
    if (left != count)
        refuse("%s: the library refused the launch (B=%d V=%d K=%d S=%d half=%d)", who, static_cast<int>(b), static_cast<int>(v), static_cast<int>(k),
               static_cast<int>(slots), static_cast<int>(half));
    return pack(unlocked, std::move(x), std::move(stats), std::move(rope));
}

// (tokens, pos, embedding, rope_table) -> (x, rope [2, positions, half]): int64 tokens [B, T] and positions of T or B T elements
TERNA_FUNCTION(prompt_inputs, 4)
{
    const char* who = "prompt_inputs";
    const at::Tensor &tokens = tensor(a[0]), &pos = tensor(a[1]), &embedding = tensor(a[2]), &table = tensor(a[3]);
    check_matrix(who, embedding);
    const int64_t m = tokens.numel(), v = embedding.size(0), k = embedding.size(1), rows = pos.numel();
    if (tokens.dim() != 2 || m < 1 || m > INT32_MAX || (rows != m && rows != tokens.size(1)))
        refuse("%s: tokens [B, T] and positions of T or B * T elements", who);
    if (table.dim() != 3 || table.size(1) != 2 || tokens.scalar_type() != at::kLong || pos.scalar_type() != at::kLong || table.scalar_type() != at::kFloat ||
        embedding.scalar_type() != at::kBFloat16 || !embedding.is_contiguous() || !table.is_contiguous())
        refuse("%s: tokens / pos int64, embedding bf16 [V, K] and rope_table fp32 [S, 2, half] contiguous", who);
    Unlocked unlocked;
    const at::Tensor ids = tokens.contiguous(), at_slot = pos.contiguous();
    const int64_t slots = table.size(0), half = table.size(2);
    at::Tensor x = make({m, k}, at::kBFloat16, embedding), rope = make({2, rows, half}, at::kFloat, embedding);
    const int rc = lib.ternaspmm_prompt_inputs(data<long long>(&ids), data<long long>(&at_slot), rows, data<terna_bf16>(&embedding), v, k, data<float>(&table), slots,
                                               half, data<terna_bf16>(&x), data<float>(&rope), m, stream());
    unlocked.end();
    if (rc != 0)
        refuse("%s: the library refused the launch (M=%d V=%d K=%d S=%d half=%d)", who, static_cast<int>(m), static_cast<int>(v), static_cast<int>(k),
               static_cast<int>(slots), static_cast<int>(half));
    return pack(unlocked, std::move(x), std::move(rope));
}

// (tokens, pos, embedding, rope_table, heads, head_dim, scale, eps, splits, blocks) -> the residual stream behind the last block, bf16 [B, dim],
// or None where the step is not one for this launch (the launches it stands for have the checks that raise).  blocks: a sequence of tuples (wqkv, ws, ws_num, out_features, wo [4], interleaved
// w13 [4], w2 [4], attention_norm, attn_sub_norm, ffn_norm, ffn_sub_norm, cache_k, cache_v).
TERNA_FUNCTION(decode_step, 10)
{
    const char* who = "decode_step";
    const at::Tensor &tokens = tensor(a[0]), &pos = tensor(a[1]), &embedding = tensor(a[2]), &table = tensor(a[3]);
    check_matrix(who, embedding);
    const int64_t b = tokens.numel(), v = embedding.size(0), dim = embedding.size(1);
    const int64_t heads = integer32(a[4]), head_dim = integer32(a[5]), wide = heads * head_dim;
    if (table.dim() != 3 || table.size(1) != 2 || 2 * table.size(2) != head_dim || tokens.scalar_type() != at::kLong || pos.scalar_type() != at::kLong ||
        (pos.numel() != 1 && pos.numel() != b) || table.scalar_type() != at::kFloat || embedding.scalar_type() != at::kBFloat16 || !embedding.is_contiguous() ||
        !table.is_contiguous() || !embedding.is_cuda())
        Py_RETURN_NONE;
    if (!PyTuple_Check(a[9]) && !PyList_Check(a[9])) refuse("%s: blocks is a list", who);
    const Py_ssize_t layers = PySequence_Fast_GET_SIZE(a[9]);
    if (b < 1 || b > 64 || layers < 1 || layers > 1024) Py_RETURN_NONE;
    ternaspmm_step_desc d{};
    d.layers = layers, d.M = b, d.dim = dim, d.heads = heads, d.head_dim = head_dim, d.slots = table.size(0);
    d.splits = integer32(a[8]), d.per_sequence = pos.numel() == b && b > 1, d.vocab = v;
    d.scale = real(a[6]), d.eps = real(a[7]);
    std::vector<ternaspmm_step_block> blocks(layers);
    for (Py_ssize_t n = 0; n < layers; ++n) {
        PyObject* item = PySequence_Fast_GET_ITEM(a[9], n);
        if (!PyTuple_Check(item) || PyTuple_GET_SIZE(item) != 22) refuse("%s: a block is a tuple of 22", who);
        PyObject* const* p = reinterpret_cast<PyTupleObject*>(item)->ob_item;
        const int64_t qkv_n = integer32(p[3]), gate_n = integer32(p[11]), ffn = gate_n / 2;
        const BlockLinear qkv_w(who, p, dim), o_w(who, p + 4, wide), gate_w(who, p + 8, dim), down_w(who, p + 12, ffn);
        const at::Tensor* norm[4] = {&tensor(p[16]), &tensor(p[17]), &tensor(p[18]), &tensor(p[19])};
        const int64_t want[4] = {dim, wide, dim, ffn};
        for (int i = 0; i < 4; ++i)
            if (norm[i]->numel() != want[i] || norm[i]->scalar_type() != at::kBFloat16 || !norm[i]->is_contiguous()) Py_RETURN_NONE;
        const at::Tensor &ck = tensor(p[20]), &cv = tensor(p[21]);
        if (ck.dim() != 4 || ck.sizes() != cv.sizes() || ck.size(0) != b || ck.size(2) != d.slots || ck.size(3) != head_dim || !ck.is_contiguous() ||
            !cv.is_contiguous() || ck.scalar_type() != at::kBFloat16 || cv.scalar_type() != at::kBFloat16)
            Py_RETURN_NONE;
        const int kv = ck.size(1);
        if (o_w.n != dim || down_w.n != dim || qkv_n != (heads + 2 * kv) * head_dim) Py_RETURN_NONE;
        if (n == 0) {
            d.kv_heads = kv, d.ffn = ffn, d.ws_num_qkv = qkv_w.ws_num, d.ws_num_o = o_w.ws_num, d.ws_num_down = down_w.ws_num;
        } else if (d.kv_heads != kv || d.ffn != ffn || d.ws_num_qkv != qkv_w.ws_num || d.ws_num_o != o_w.ws_num || d.ws_num_down != down_w.ws_num) {
            Py_RETURN_NONE;                      // blocks of different shapes
        }
        if (gate_w.ws_num != 2 || ffn * 2 != gate_n) Py_RETURN_NONE;
        blocks[n] = ternaspmm_step_block{data(&qkv_w.packed), data(&o_w.packed), data(&gate_w.packed), data(&down_w.packed),
                                         data<terna_bf16>(&qkv_w.ws), data<terna_bf16>(&o_w.ws), data<terna_bf16>(&gate_w.ws), data<terna_bf16>(&down_w.ws),
                                         data<terna_bf16>(norm[0]), data<terna_bf16>(norm[1]), data<terna_bf16>(norm[2]), data<terna_bf16>(norm[3]),
                                         data<terna_bf16>(&ck), data<terna_bf16>(&cv)};
    }
    const long long bytes = lib.ternaspmm_decode_step_bytes(&d);
    if (bytes < 0) Py_RETURN_NONE;
    Unlocked unlocked;
    const at::Tensor ids = tokens.contiguous(), at_slot = pos.contiguous();
    at::Tensor x = make({b, dim}, at::kBFloat16, embedding);
    const c10::DataPtr scratch = device_allocator()->allocate(bytes);
    if (lib.ternaspmm_decode_step(&d, blocks.data(), data<long long>(&ids), data<long long>(&at_slot), data<terna_bf16>(&embedding), data<float>(&table), scratch.get(),
                                  data<terna_bf16>(&x), stream()) != 0)
        return none(unlocked);
    return wrap(std::move(x), unlocked);
}

// (path of libternaspmm.so)
TERNA_FUNCTION(init, 1)
{
    const char* path = PyUnicode_AsUTF8(a[0]);
    if (path == nullptr) throw Refused();
    void* handle = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    if (handle == nullptr) {
        PyErr_SetString(PyExc_ImportError, dlerror());
        throw Refused();
    }
#define X(name)                                                                                                        \
    if ((lib.name = reinterpret_cast<decltype(&::name)>(dlsym(handle, #name))) == nullptr) {                             \
        PyErr_SetString(PyExc_ImportError, "libternaspmm.so does not export " #name);                                  \
        throw Refused();                                                                                               \
    }
    TERNA_ENTRY_POINTS(X)
#undef X
    Py_RETURN_NONE;
}

#define METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(init), METHOD(bit_linear), METHOD(bit_linear_bf16), METHOD(quant_input), METHOD(linear_packed),
                         METHOD(linear_bf16_packed), METHOD(rmsnorm_quant), METHOD(relu2_mul_rmsnorm_quant), METHOD(quant_from_stats),
                         METHOD(fused_linear), METHOD(fused_linear_own_stats), METHOD(prompt_attention), METHOD(decode_attention), METHOD(block),
                         METHOD(attention_merge_rmsnorm_quant), METHOD(step_attention_merge), METHOD(step_inputs), METHOD(prompt_inputs), METHOD(decode_step), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module); }
