// The hot operators' host path as one native call each: CPython module `_calls`, bound to the kernel library that _lib
// has loaded.  A call checks its operands, allocates the result and enqueues the kernels on the current stream; whatever it
// does not take as it lies (other layouts, dtypes or devices, subclasses, an active mode or transform, empty sizes, an error
// status) returns None, and the Python form of the operator in ops.py, which has every check and conversion, runs instead.  So
// nothing is accepted, refused or routed here that the Python form would not do the same way.
//
// What it answers: a decode step calls these at 5 to 10 us of kernel time, and the same steps in Python took 20 us (int4
// product) to 30 us (row quantizer + int8 product) of host time a call, so the card waited.
// Measured (us a pass with the modules' own Python, host time, before / with this): int8 dynamic linear 30.6 / 10.0, int4 at one
// row 21.2 / 6.6, int4 with bias at 48 rows 27.5 / 12.4, 2-bit linear 20.2 / 6.3, ternary MLP (two linears and a relu) 59.9 / 21.7,
// affine quantize + dequantize 28.3 / 9.4.  Above 32 rows only the routes that the library picks itself are taken here: from there
// on the kernels are longer than either form.
#include <Python.h>

#include <dlfcn.h>

#include <cstdint>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <ATen/core/LegacyTypeDispatch.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <c10/util/Exception.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "tpq.h"

namespace {

// the entry points of the bound library
struct Library {
#define TPQ_ENTRY(NAME) decltype(&::NAME) NAME = nullptr;
#define TPQ_ENTRIES                                                                                                       \
    TPQ_ENTRY(tpq_quantize_rowwise) TPQ_ENTRY(tpq_int8_mm_workspace_bytes) TPQ_ENTRY(tpq_int8_mm_dequant_ws)                \
    TPQ_ENTRY(tpq_ternary_mm_workspace_bytes) TPQ_ENTRY(tpq_ternary_linear_workspace_bytes) TPQ_ENTRY(tpq_ternary_linear_row) TPQ_ENTRY(tpq_ternary_linear)                \
    TPQ_ENTRY(tpq_int4_mm_ws)                                                                                             \
    TPQ_ENTRY(tpq_int4_mm_rows_workspace_bytes) TPQ_ENTRY(tpq_packed_rows_call_workspace_bytes) TPQ_ENTRY(tpq_int4_mm_rows_bias) \
    TPQ_ENTRY(tpq_int4_mm_rows_takes) TPQ_ENTRY(tpq_lowbit_mm_rows) TPQ_ENTRY(tpq_lowbit_mm_rows_takes)                     \
    TPQ_ENTRY(tpq_lowbit_mm) TPQ_ENTRY(tpq_quantize_affine) TPQ_ENTRY(tpq_dequantize_affine) \
    TPQ_ENTRY(tpq_f32_linear_grads_workspace_bytes) TPQ_ENTRY(tpq_f32_linear_grads) \
    TPQ_ENTRY(tpq_f32_linear_grads_takes) TPQ_ENTRY(tpq_quantize_beside_takes) \
    TPQ_ENTRY(tpq_int8_linear_few_pays) TPQ_ENTRY(tpq_ternary_linear_few_pays) TPQ_ENTRY(tpq_int8_linear_few_takes) TPQ_ENTRY(tpq_int8_linear_few) TPQ_ENTRY(tpq_ternary_linear_few_takes) TPQ_ENTRY(tpq_ternary_linear_few) \
    TPQ_ENTRY(tpq_quantize_both_rowwise) TPQ_ENTRY(tpq_quantize_rowwise_pad)
    TPQ_ENTRIES
#undef TPQ_ENTRY
};
Library lib;

constexpr int64_t kAlign = 256;  // parts of one scratch allocation
int64_t padded(int64_t bytes) { return (bytes + kAlign - 1) / kAlign * kAlign; }

int float_tag(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return TPQ_DTYPE_F32;
        case at::kHalf: return TPQ_DTYPE_F16;
        case at::kBFloat16: return TPQ_DTYPE_BF16;
        default: return -1;
    }
}

// Something is watching or rewriting tensor operations: those see the Python form.
bool observed() {
    return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set() ||
           c10::impl::tls_local_dispatch_key_set().included_.has(c10::DispatchKey::Tracer);
}

// An ordinary dense GPU tensor (no subclass, no transform's wrapper, no lazy conjugate or negative), contiguous.
const at::Tensor* plain(PyObject* o) {
    static const uint64_t ordinary =
        c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA}).raw_repr();
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || (t.key_set().raw_repr() & ~ordinary) != 0 || t.layout() != at::kStrided || !t.is_contiguous()) return nullptr;
    return &t;
}

bool same_device(const at::Tensor& a, const at::Tensor& b) { return a.device() == b.device(); }

// An operand that may be None: false if it is there and not a plain tensor of that type and size on x's device
bool optional_vector(PyObject* o, at::ScalarType type, int64_t numel, const at::Tensor& x, const at::Tensor** out) {
    *out = nullptr;
    if (o == Py_None) return true;
    const at::Tensor* t = plain(o);
    if (!t || t->scalar_type() != type || t->numel() != numel || !same_device(*t, x)) return false;
    *out = t;
    return true;
}

bool as_int(PyObject* o, int64_t* v) {
    if (!PyLong_CheckExact(o)) return false;
    *v = PyLong_AsLongLong(o);
    if (*v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

bool as_float(PyObject* o, double* v) {
    if (!PyFloat_CheckExact(o)) return false;
    *v = PyFloat_AS_DOUBLE(o);
    return true;
}

// The GIL off while the allocator and the launches run, the operand's device current.
struct GilOff {
    PyThreadState* state = PyEval_SaveThread();
    GilOff() = default;
    ~GilOff() { PyEval_RestoreThread(state); }
    GilOff(const GilOff&) = delete;
    GilOff& operator=(const GilOff&) = delete;
};
struct Enqueue {
    GilOff gil;
    c10::DeviceGuard guard;
    void* stream;
    explicit Enqueue(const at::Tensor& x) : guard(x.device()), stream(c10::hip::getCurrentHIPStream(x.device().index()).stream()) {}
};

at::Tensor allocate(at::IntArrayRef sizes, at::ScalarType type, const at::Tensor& like) {
    return at::empty(sizes, at::TensorOptions().dtype(type).device(like.device()));
}

// x [..., K] -> the sizes of a product with N channels; rows in *M
c10::SmallVector<int64_t, 4> product_sizes(const at::Tensor& x, int64_t N, int64_t* M) {
    c10::SmallVector<int64_t, 4> sizes(x.sizes().begin(), x.sizes().end());
    *M = 1;
    for (size_t i = 0; i + 1 < sizes.size(); ++i) *M *= sizes[i];
    sizes.back() = N;
    return sizes;
}

// Codes and row scales of M activation rows and a product's scratch.  Small ones share one allocation; from 1 MB of codes on they
// are tensors of their own, as the separate operators ask for them, which leaves the allocator blocks of sizes that others ask for too.
// Where the codes lie does not matter to the kernels (2048 rows of 4096 -> 4096, four processes in turn: 39.0 / 39.3 and 39.0 / 38.8 us a
// pass own / 39.2 / 39.3 and 39.3 / 39.4 one block).
struct Quantized {
    at::Tensor first, second, third;
    int8_t* codes;
    float* scales;
    void* scratch;
    int64_t scratch_bytes;
};
constexpr int64_t kOwnTensors = int64_t{1} << 20;

template <class T>
const T* ptr(const at::Tensor* t) { return t ? static_cast<const T*>(t->const_data_ptr()) : nullptr; }
template <class T>
T* out_ptr(const at::Tensor& t) { return static_cast<T*>(t.data_ptr()); }

Quantized room_for_codes(const at::Tensor& x, int64_t M, int64_t K, int64_t scratch_bytes) {
    Quantized q;
    q.scratch_bytes = scratch_bytes;
    if (M * K >= kOwnTensors) {
        q.first = allocate({M, K}, at::kChar, x);
        q.second = allocate({M}, at::kFloat, x);
        if (scratch_bytes) q.third = allocate({scratch_bytes}, at::kByte, x);
        q.codes = out_ptr<int8_t>(q.first);
        q.scales = out_ptr<float>(q.second);
        q.scratch = scratch_bytes ? q.third.data_ptr() : nullptr;
        return q;
    }
    const int64_t scales_at = padded(M * K), scratch_at = scales_at + padded(4 * M);
    q.first = allocate({scratch_at + scratch_bytes}, at::kByte, x);
    char* const base = out_ptr<char>(q.first);
    q.codes = reinterpret_cast<int8_t*>(base);
    q.scales = reinterpret_cast<float*>(base + scales_at);
    q.scratch = scratch_bytes ? base + scratch_at : nullptr;
    return q;
}

// a tuple of two references, which it takes over; null (an error is set) where one of them is
PyObject* pair_of(PyObject* first, PyObject* second) {
    PyObject* pair = first && second ? PyTuple_New(2) : nullptr;
    if (!pair) {
        Py_XDECREF(first);
        Py_XDECREF(second);
        return nullptr;
    }
    PyTuple_SET_ITEM(pair, 0, first);
    PyTuple_SET_ITEM(pair, 1, second);
    return pair;
}

#define TPQ_CALL(NAME, COUNT)                                              \
    PyObject* NAME(PyObject*, PyObject* const* args, Py_ssize_t count) {   \
        HANDLE_TH_ERRORS                                                   \
        if (count != COUNT) {                                              \
            PyErr_SetString(PyExc_TypeError, #NAME ": " #COUNT " arguments expected"); \
            return nullptr;                                                \
        }                                                                  \
        if (lib.tpq_quantize_rowwise == nullptr || observed()) Py_RETURN_NONE; \
        try {
// Too little memory: the Python form has routes with less (a ternary weight that is not written out, gradients without slices), or
// fails as it did.
#define TPQ_CALL_END   \
        } catch (const c10::OutOfMemoryError&) { \
            Py_RETURN_NONE;                      \
        }                                        \
        END_HANDLE_TH_ERRORS \
    }

// quantize_rowwise(x [M, K], eps, divisor, qmin, qmax, sign_mode) -> (codes, scales)
TPQ_CALL(quantize_rowwise, 6)
    const at::Tensor* x = plain(args[0]);
    double eps, divisor;
    int64_t qmin, qmax, sign_mode;
    if (!x || x->dim() != 2 || x->numel() == 0 || float_tag(x->scalar_type()) < 0 || !as_float(args[1], &eps) || !as_float(args[2], &divisor) ||
        !as_int(args[3], &qmin) || !as_int(args[4], &qmax) || !as_int(args[5], &sign_mode))
        Py_RETURN_NONE;
    const int64_t M = x->size(0), K = x->size(1);
    at::Tensor codes, scales;
    int status;
    {
        Enqueue q(*x);
        codes = allocate({M, K}, at::kChar, *x);
        scales = allocate({M}, at::kFloat, *x);
        status = lib.tpq_quantize_rowwise(x->const_data_ptr(), float_tag(x->scalar_type()), M, K, static_cast<float>(eps), static_cast<float>(divisor),
                                          static_cast<int>(qmin), static_cast<int>(qmax), static_cast<int>(sign_mode), out_ptr<int8_t>(codes), out_ptr<float>(scales), q.stream);
    }
    if (status != TPQ_OK) Py_RETURN_NONE;
    PyObject* first = THPVariable_Wrap(std::move(codes));
    return pair_of(first, first ? THPVariable_Wrap(std::move(scales)) : nullptr);
TPQ_CALL_END

// int8_mm_dequant(a int8 [M, K], w int8 [N, K], row_scale, col_scale, bias or None, out_dtype, ragged_rows)
TPQ_CALL(int8_mm_dequant, 7)
    const at::Tensor *a = plain(args[0]), *w = plain(args[1]), *rs = plain(args[2]), *cs = plain(args[3]), *bias;
    int64_t ragged_rows;
    if (!a || !w || !rs || !cs || a->dim() != 2 || w->dim() != 2 || a->scalar_type() != at::kChar || w->scalar_type() != at::kChar ||
        a->size(1) != w->size(1) || rs->scalar_type() != at::kFloat || cs->scalar_type() != at::kFloat || !same_device(*a, *w) || !same_device(*a, *rs) ||
        !same_device(*a, *cs) || !THPDtype_Check(args[5]) || !as_int(args[6], &ragged_rows))
        Py_RETURN_NONE;
    const int64_t M = a->size(0), K = a->size(1), N = w->size(0);
    const at::ScalarType type = reinterpret_cast<THPDtype*>(args[5])->scalar_type;
    if (M == 0 || N == 0 || K == 0 || rs->numel() != M || cs->numel() != N || float_tag(type) < 0 || (K % 16 && M > ragged_rows) ||
        !optional_vector(args[4], at::kFloat, N, *a, &bias))
        Py_RETURN_NONE;
    at::Tensor out;
    int status;
    {
        Enqueue q(*a);
        out = allocate({M, N}, type, *a);
        const int64_t scratch_bytes = lib.tpq_int8_mm_workspace_bytes(M, N, K);
        const at::Tensor scratch = scratch_bytes ? allocate({scratch_bytes}, at::kByte, *a) : at::Tensor();
        status = lib.tpq_int8_mm_dequant_ws(ptr<int8_t>(a), ptr<int8_t>(w), ptr<float>(rs), ptr<float>(cs), ptr<float>(bias), out.data_ptr(), float_tag(type), M, N, K,
                                            scratch_bytes ? scratch.data_ptr() : nullptr, scratch_bytes, q.stream);
    }
    if (status != TPQ_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
TPQ_CALL_END

// Rows of codes that a product of more than ragged_rows rows reads: the next multiple of 128 where K is none of 16
int64_t code_pitch(int64_t K) { return K % 16 ? (K + 127) / 128 * 128 : K; }

// A launch saved that makes the device's part longer (the library's answer 1) is saved in eager calls only; the bits are the same either way.
bool pays_here(int pays, const at::Tensor& x) {
    if (pays != 1) return pays != 0;
    hipStreamCaptureStatus capture = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(c10::hip::getCurrentHIPStream(x.device().index()).stream(), &capture) == hipSuccess) return capture == hipStreamCaptureStatusNone;
    (void)hipGetLastError();  // the default stream beside a capture that waits for it: not captured itself
    return true;
}

// int8_linear(x [..., K] float, w int8 [N, K], col_scale, bias or None, eps, out_dtype, ragged_rows): quantize + product.  Above ragged_rows
// rows with K % 16 != 0 the quantizer's launch copies the weight to padded rows as well.
TPQ_CALL(int8_linear, 7)
    const at::Tensor *x = plain(args[0]), *w = plain(args[1]), *cs = plain(args[2]), *bias;
    double eps;
    int64_t ragged_rows;
    if (!x || !w || !cs || x->dim() < 1 || x->numel() == 0 || float_tag(x->scalar_type()) < 0 || w->dim() != 2 || w->scalar_type() != at::kChar ||
        x->size(-1) != w->size(1) || cs->scalar_type() != at::kFloat || cs->numel() != w->size(0) || w->size(0) == 0 || !same_device(*x, *w) ||
        !same_device(*x, *cs) || !as_float(args[4], &eps) || !THPDtype_Check(args[5]) || !as_int(args[6], &ragged_rows))
        Py_RETURN_NONE;
    const int64_t K = w->size(1), N = w->size(0);
    int64_t M;
    const auto sizes = product_sizes(*x, N, &M);
    const at::ScalarType type = reinterpret_cast<THPDtype*>(args[5])->scalar_type;
    const bool pad = K % 16 != 0 && M > ragged_rows;
    const int64_t pitch = pad ? code_pitch(K) : K;
    if (float_tag(type) < 0 || !optional_vector(args[3], at::kFloat, N, *x, &bias) ||
        (pad && !lib.tpq_quantize_beside_takes(x->const_data_ptr(), nullptr, M, N, K, pitch)))
        Py_RETURN_NONE;
    at::Tensor out;
    int status;
    if (lib.tpq_int8_linear_few_takes(x->const_data_ptr(), ptr<int8_t>(w), M, N, K) && pays_here(lib.tpq_int8_linear_few_pays(M, N, K), *x)) {
        {
            Enqueue q(*x);
            out = allocate(sizes, type, *x);
            status = lib.tpq_int8_linear_few(x->const_data_ptr(), float_tag(x->scalar_type()), ptr<int8_t>(w), ptr<float>(cs), ptr<float>(bias), M, N, K,
                                             static_cast<float>(eps), out.data_ptr(), float_tag(type), q.stream);
        }
        if (status != TPQ_OK) Py_RETURN_NONE;
        return THPVariable_Wrap(std::move(out));
    }
    {
        Enqueue q(*x);
        const Quantized room = room_for_codes(*x, M, pitch, lib.tpq_int8_mm_workspace_bytes(M, N, pitch));
        const at::Tensor padded_w = pad ? allocate({N, pitch}, at::kChar, *x) : at::Tensor();
        out = allocate(sizes, type, *x);
        if (pad)
            status = lib.tpq_quantize_rowwise_pad(x->const_data_ptr(), float_tag(x->scalar_type()), M, K, static_cast<float>(eps), ptr<int8_t>(w), N, pitch, room.codes,
                                                  room.scales, out_ptr<int8_t>(padded_w), q.stream);
        else
            status = lib.tpq_quantize_rowwise(x->const_data_ptr(), float_tag(x->scalar_type()), M, K, static_cast<float>(eps), 127.0f, -127, 127, 0, room.codes, room.scales,
                                              q.stream);
        if (status == TPQ_OK)
            status = lib.tpq_int8_mm_dequant_ws(room.codes, pad ? out_ptr<int8_t>(padded_w) : ptr<int8_t>(w), room.scales, ptr<float>(cs), ptr<float>(bias), out.data_ptr(),
                                                float_tag(type), M, N, pitch, room.scratch, room.scratch_bytes, q.stream);
    }
    if (status != TPQ_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
TPQ_CALL_END

// lowbit_linear(x [..., K] float, w [N, K] of the same type, x_eps, w_eps, divisor, qmin, qmax, sign_mode) -> float32: rows of both
// quantized in one launch (x to 8 bits, w by the parameters given) + product
TPQ_CALL(lowbit_linear, 8)
    const at::Tensor *x = plain(args[0]), *w = plain(args[1]);
    double x_eps, w_eps, divisor;
    int64_t qmin, qmax, sign_mode;
    if (!x || !w || !as_float(args[2], &x_eps) || !as_float(args[3], &w_eps) || !as_float(args[4], &divisor) || !as_int(args[5], &qmin) || !as_int(args[6], &qmax) ||
        !as_int(args[7], &sign_mode) || x->dim() < 1 || x->numel() == 0 || float_tag(x->scalar_type()) < 0 || w->scalar_type() != x->scalar_type() || w->dim() != 2 ||
        w->numel() == 0 || x->size(-1) != w->size(1) || !same_device(*x, *w))
        Py_RETURN_NONE;
    const int64_t K = w->size(1), N = w->size(0), pitch = code_pitch(K);
    int64_t M;
    const auto sizes = product_sizes(*x, N, &M);
    if (!lib.tpq_quantize_beside_takes(x->const_data_ptr(), w->const_data_ptr(), M, N, K, pitch)) Py_RETURN_NONE;
    at::Tensor out;
    int status;
    {
        Enqueue q(*x);
        const Quantized room = room_for_codes(*x, M, pitch, lib.tpq_int8_mm_workspace_bytes(M, N, pitch));
        const Quantized weight = room_for_codes(*x, N, pitch, 0);
        out = allocate(sizes, at::kFloat, *x);
        status = lib.tpq_quantize_both_rowwise(x->const_data_ptr(), w->const_data_ptr(), float_tag(x->scalar_type()), M, N, K, pitch, static_cast<float>(x_eps),
                                               static_cast<float>(w_eps), static_cast<float>(divisor), static_cast<int>(qmin), static_cast<int>(qmax),
                                               static_cast<int>(sign_mode), room.codes, room.scales, weight.codes, weight.scales, q.stream);
        if (status == TPQ_OK)
            status = lib.tpq_int8_mm_dequant_ws(room.codes, weight.codes, room.scales, weight.scales, nullptr, out.data_ptr(), TPQ_DTYPE_F32, M, N, pitch, room.scratch,
                                                room.scratch_bytes, q.stream);
    }
    if (status != TPQ_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
TPQ_CALL_END

// One row of a weight of up to this many codes: the row kernel quantizes the row itself.  Each of its workgroups reads and quantizes
// the whole row, so beyond, the kernel of few rows, one workgroup per compute unit, or the quantizer's launch and codes in memory are the cheaper way.  Measured (us, weights from HBM,
// float16, one launch / two): 2560 -> 6912 5.49 / 6.06, 4096 x 4096 5.34 / 6.02, 2560 -> 9216 5.67 / 5.91, 4096 -> 6144 6.01 / 5.98,
// 5120 x 5120 6.23 / 6.41 (float32 7.30 / 6.62), 2560 -> 10240 6.39 / 6.16, 4096 -> 8192 7.23 / 6.75, 4096 -> 14336 10.2 / 7.6,
// 8192 -> 28672 35.7 / 17.3.
constexpr int64_t kRowQuantizedInProduct = int64_t{3} << 23;

// ternary_linear(x [..., K] float, packed uint8 [N, ceil(K / 4)], w_scale, K, bias or None, eps) -> float32
TPQ_CALL(ternary_linear, 6)
    const at::Tensor *x = plain(args[0]), *packed = plain(args[1]), *bias;
    double w_scale, eps;
    int64_t K;
    if (!x || !packed || !as_float(args[2], &w_scale) || !as_int(args[3], &K) || !as_float(args[5], &eps) || x->dim() < 1 || x->numel() == 0 ||
        float_tag(x->scalar_type()) < 0 || x->size(-1) != K || packed->dim() != 2 || packed->scalar_type() != at::kByte || packed->size(0) == 0 ||
        packed->size(1) != (K + 3) / 4 || !same_device(*x, *packed))
        Py_RETURN_NONE;
    const int64_t N = packed->size(0);
    int64_t M;
    const auto sizes = product_sizes(*x, N, &M);
    if (!optional_vector(args[4], at::kFloat, N, *x, &bias)) Py_RETURN_NONE;
    at::Tensor out;
    int status = TPQ_ERR_UNSUPPORTED;
    {
        Enqueue q(*x);
        const bool row = M == 1 && N * K <= kRowQuantizedInProduct;
        const bool one_launch = row || (lib.tpq_ternary_linear_few_takes(x->const_data_ptr(), ptr<uint8_t>(packed), M, N, K) && pays_here(lib.tpq_ternary_linear_few_pays(M, N, K), *x));
        if (one_launch) out = allocate(sizes, at::kFloat, *x);
        if (one_launch && !row)
            status = lib.tpq_ternary_linear_few(x->const_data_ptr(), float_tag(x->scalar_type()), ptr<uint8_t>(packed), static_cast<float>(w_scale), ptr<float>(bias), M, N, K,
                                                static_cast<float>(eps), out_ptr<float>(out), q.stream);
        if (row) {
            status = lib.tpq_ternary_linear_row(x->const_data_ptr(), float_tag(x->scalar_type()), ptr<uint8_t>(packed), static_cast<float>(w_scale), ptr<float>(bias), N, K,
                                                static_cast<float>(eps), out_ptr<float>(out), q.stream);
        }
        if (!one_launch || status != TPQ_OK) {
            // rows off 16 bytes are quantized by themselves: the product behind them is that of the codes
            const auto workspace_bytes = reinterpret_cast<uintptr_t>(x->const_data_ptr()) % 16 ? lib.tpq_ternary_mm_workspace_bytes : lib.tpq_ternary_linear_workspace_bytes;
            const Quantized room = room_for_codes(*x, M, K, workspace_bytes(M, N, K));
            if (!one_launch) out = allocate(sizes, at::kFloat, *x);
            status = lib.tpq_ternary_linear(x->const_data_ptr(), float_tag(x->scalar_type()), ptr<uint8_t>(packed), static_cast<float>(w_scale), ptr<float>(bias), M, N, K,
                                            static_cast<float>(eps), room.codes, room.scales, out_ptr<float>(out), room.scratch, room.scratch_bytes, q.stream);
        }
    }
    if (status != TPQ_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
TPQ_CALL_END

// int4_mm(x [..., K], packed int32 [N / 8, K / 32, 32, 1], group, scales_and_zeros [K / group, N, 2] of x's type, bias or None,
// workspaces): the rows kernel, which adds the bias as a separate add would, and, up to 32 rows, the decode kernels and an add.  workspaces: {(device, stream): zero-filled buffer} of
// ops._int4_workspace; a stream that has none yet, or too small a one, gets it in the Python form.
TPQ_CALL(int4_mm, 6)
    const at::Tensor *x = plain(args[0]), *packed = plain(args[1]), *sz = plain(args[3]), *bias;
    int64_t group;
    if (!x || !packed || !sz || !as_int(args[2], &group) || !PyDict_CheckExact(args[5]) || (group != 32 && group != 64 && group != 128) || x->dim() < 1 ||
        x->numel() == 0 || packed->dim() != 4 || packed->scalar_type() != at::kInt || packed->size(0) == 0 || packed->size(2) != 32 || packed->size(3) != 1 ||
        sz->dim() != 3 || sz->scalar_type() != x->scalar_type() || !same_device(*x, *packed) || !same_device(*x, *sz))
        Py_RETURN_NONE;
    const int tag = float_tag(x->scalar_type());
    const int64_t K = x->size(-1), N = packed->size(0) * 8;
    if (tag < 0 || packed->size(1) != (K + 31) / 32 || sz->size(0) != (K + group - 1) / group || sz->size(1) != N || sz->size(2) != 2) Py_RETURN_NONE;
    // a bias that something differentiates is added where that is seen
    if (!optional_vector(args[4], x->scalar_type(), N, *x, &bias) || (bias && (bias->dim() != 1 || bias->requires_grad() || bias->_fw_grad(0).defined()))) Py_RETURN_NONE;
    int64_t M;
    const auto sizes = product_sizes(*x, N, &M);
    const bool rows = lib.tpq_int4_mm_rows_takes(x->const_data_ptr(), tag, M, N, K, group, ptr<int32_t>(packed), sz->const_data_ptr()) != 0;
    if (!rows && M > (tag == TPQ_DTYPE_F32 ? 1 : 32)) Py_RETURN_NONE;
    // owned by this call: without the GIL, another thread may put a larger buffer in its place in the dict
    at::Tensor workspace;
    int64_t workspace_bytes = 0;
    if (rows) {
        workspace_bytes = lib.tpq_packed_rows_call_workspace_bytes(tag, M, N, K, 0, group);
    } else {
        const int64_t stream = static_cast<int64_t>(reinterpret_cast<intptr_t>(c10::hip::getCurrentHIPStream(x->device().index()).stream()));
        PyObject* key = Py_BuildValue("(iL)", static_cast<int>(x->device().index()), static_cast<long long>(stream));
        if (!key) return nullptr;
        PyObject* held = PyDict_GetItemWithError(args[5], key);
        Py_DECREF(key);
        if (!held) {
            if (PyErr_Occurred()) return nullptr;
            Py_RETURN_NONE;
        }
        const at::Tensor* const found = plain(held);
        if (!found || found->numel() < static_cast<int64_t>(lib.tpq_int4_mm_rows_workspace_bytes(M, N, K))) Py_RETURN_NONE;
        workspace = *found;
        workspace_bytes = workspace.numel();
    }
    at::Tensor out;
    int status;
    {
        Enqueue q(*x);
        out = allocate(sizes, x->scalar_type(), *x);
        if (rows) {
            const at::Tensor part = workspace_bytes ? allocate({workspace_bytes}, at::kByte, *x) : at::Tensor();
            status = lib.tpq_int4_mm_rows_bias(x->const_data_ptr(), tag, M, K, ptr<int32_t>(packed), N, group, sz->const_data_ptr(), ptr<void>(bias), out.data_ptr(),
                                          workspace_bytes ? part.data_ptr() : nullptr, workspace_bytes, q.stream);
        } else {
            status = lib.tpq_int4_mm_ws(x->const_data_ptr(), tag, M, K, ptr<int32_t>(packed), 2, N, group, sz->const_data_ptr(), out.data_ptr(), workspace.data_ptr(),
                                        static_cast<size_t>(workspace_bytes), q.stream);
            if (status == TPQ_OK && bias) {
                const at::AutoDispatchBelowADInplaceOrView raw;
                out.add_(*bias);
            }
        }
    }
    if (status != TPQ_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
TPQ_CALL_END

// lowbit_mm(x [..., K], packed uint8 [N, ceil(K / per_byte)], bits, K, scales_and_zeros float32 [groups, N, 2], bias or None, lsb_first):
// the rows kernel and, up to 32 rows, the decode kernels
TPQ_CALL(lowbit_mm, 7)
    const at::Tensor *x = plain(args[0]), *packed = plain(args[1]), *sz = plain(args[4]), *bias;
    int64_t bits, K;
    if (!x || !packed || !sz || !as_int(args[2], &bits) || !as_int(args[3], &K) || !PyBool_Check(args[6]) || bits < 1 || bits > 8 || x->dim() < 1 || x->numel() == 0 ||
        x->size(-1) != K || packed->dim() != 2 || packed->scalar_type() != at::kByte || packed->size(0) == 0 || sz->dim() != 3 || sz->scalar_type() != at::kFloat ||
        sz->size(0) < 1 || sz->size(1) != packed->size(0) || sz->size(2) != 2 || K % sz->size(0) != 0 || !same_device(*x, *packed) || !same_device(*x, *sz))
        Py_RETURN_NONE;
    const int tag = float_tag(x->scalar_type()), lsb_first = args[6] == Py_True;
    const int64_t N = packed->size(0), per_byte = 8 / bits, group = K / sz->size(0);
    int64_t M;
    const auto sizes = product_sizes(*x, N, &M);
    if (tag < 0 || packed->size(1) != (K + per_byte - 1) / per_byte || !optional_vector(args[5], at::kFloat, N, *x, &bias)) Py_RETURN_NONE;
    const bool rows = lib.tpq_lowbit_mm_rows_takes(x->const_data_ptr(), tag, M, N, K, static_cast<int>(bits), lsb_first, group, ptr<uint8_t>(packed), ptr<float>(sz)) != 0;
    if (!rows && M > 32) Py_RETURN_NONE;
    at::Tensor out;
    int status;
    {
        Enqueue q(*x);
        out = allocate(sizes, x->scalar_type(), *x);
        if (rows) {
            const int64_t bytes = lib.tpq_packed_rows_call_workspace_bytes(tag, M, N, K, static_cast<int>(bits), group);
            const at::Tensor part = bytes ? allocate({bytes}, at::kByte, *x) : at::Tensor();
            status = lib.tpq_lowbit_mm_rows(x->const_data_ptr(), tag, M, K, ptr<uint8_t>(packed), static_cast<int>(bits), lsb_first, N, group, ptr<float>(sz), ptr<float>(bias),
                                            out.data_ptr(), bytes ? part.data_ptr() : nullptr, bytes, q.stream);
        } else {
            status = lib.tpq_lowbit_mm(x->const_data_ptr(), tag, M, K, ptr<uint8_t>(packed), static_cast<int>(bits), lsb_first, N, group, ptr<float>(sz), ptr<float>(bias),
                                       out.data_ptr(), q.stream);
        }
    }
    if (status != TPQ_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
TPQ_CALL_END

constexpr int kMaxDims = 8;

// block sizes as a tuple or list of ints, one per dimension
bool as_blocks(PyObject* o, int64_t dims, int64_t* blocks) {
    if (dims > kMaxDims || !(PyTuple_CheckExact(o) || PyList_CheckExact(o)) || PySequence_Fast_GET_SIZE(o) != dims) return false;
    for (int64_t i = 0; i < dims; ++i)
        if (!as_int(PySequence_Fast_GET_ITEM(o, i), blocks + i)) return false;
    return true;
}

// a parameter of the affine codec: float32, never empty, any size (the library checks it against the blocks)
bool affine_parameters(PyObject* scales, PyObject* zeros, const at::Tensor& x, const at::Tensor** sc, const at::Tensor** zp) {
    *sc = plain(scales);
    *zp = zeros == Py_None ? nullptr : plain(zeros);
    if (!*sc || (zeros != Py_None && !*zp)) return false;
    for (const at::Tensor* t : {*sc, *zp})
        if (t && (t->scalar_type() != at::kFloat || t->numel() == 0 || !same_device(*t, x))) return false;
    return true;
}

// quantize_affine(x, block_size, scales, zero_points or None, storage, per_byte, code dtype, quant_min, quant_max)
TPQ_CALL(quantize_affine, 9)
    const at::Tensor *x = plain(args[0]), *sc, *zp;
    int64_t blocks[kMaxDims], storage, per_byte, qmin, qmax;
    if (!x || x->numel() == 0 || x->dim() < 1 || float_tag(x->scalar_type()) < 0 || !as_blocks(args[1], x->dim(), blocks) ||
        !affine_parameters(args[2], args[3], *x, &sc, &zp) || !as_int(args[4], &storage) || !as_int(args[5], &per_byte) || !THPDtype_Check(args[6]) ||
        !as_int(args[7], &qmin) || !as_int(args[8], &qmax) || per_byte < 1)
        Py_RETURN_NONE;
    at::Tensor out;
    int status;
    {
        Enqueue q(*x);
        const at::ScalarType type = reinterpret_cast<THPDtype*>(args[6])->scalar_type;
        out = per_byte == 1 ? allocate(x->sizes(), type, *x) : allocate({(x->numel() + per_byte - 1) / per_byte}, at::kByte, *x);
        status = lib.tpq_quantize_affine(x->const_data_ptr(), float_tag(x->scalar_type()), static_cast<int>(x->dim()), x->sizes().data(), blocks, ptr<float>(sc), sc->numel(),
                                         ptr<float>(zp), zp ? zp->numel() : 0, static_cast<int>(storage), qmin, qmax, out.data_ptr(), q.stream);
    }
    if (status != TPQ_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
TPQ_CALL_END

// dequantize_affine(codes, shape, block_size, scales, zero_points or None, storage) -> float32
TPQ_CALL(dequantize_affine, 6)
    const at::Tensor *codes = plain(args[0]), *sc, *zp;
    int64_t shape[kMaxDims], blocks[kMaxDims], storage;
    if (!codes || codes->numel() == 0 || !PyTuple_Check(args[1])) Py_RETURN_NONE;
    const int64_t dims = PyTuple_GET_SIZE(args[1]);
    if (dims < 1 || dims > kMaxDims) Py_RETURN_NONE;
    for (int64_t i = 0; i < dims; ++i)
        if (!as_int(PyTuple_GET_ITEM(args[1], i), shape + i) || shape[i] <= 0) Py_RETURN_NONE;
    if (!as_blocks(args[2], dims, blocks) || !affine_parameters(args[3], args[4], *codes, &sc, &zp) || !as_int(args[5], &storage)) Py_RETURN_NONE;
    at::Tensor out;
    int status;
    {
        Enqueue q(*codes);
        out = allocate({shape, static_cast<size_t>(dims)}, at::kFloat, *codes);
        status = lib.tpq_dequantize_affine(codes->const_data_ptr(), static_cast<int>(storage), static_cast<int>(dims), shape, blocks, ptr<float>(sc), sc->numel(),
                                           ptr<float>(zp), zp ? zp->numel() : 0, out_ptr<float>(out), q.stream);
    }
    if (status != TPQ_OK) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(out));
TPQ_CALL_END

// linear_grads(grad [..., N], x [..., K], w [N, K], want_x, want_w), float32 -> (grad_x like x or None, grad_w or None).  Not while
// gradients are recorded (a second derivative), an operand carries a tangent (a derivative of the gradient in forward mode) or products
// are cast: those need the products as torch operations.
TPQ_CALL(linear_grads, 5)
    const at::Tensor *g = plain(args[0]), *x = plain(args[1]), *w = plain(args[2]);
    if (!g || !x || !w || g->_fw_grad(0).defined() || x->_fw_grad(0).defined() || w->_fw_grad(0).defined() || c10::GradMode::is_enabled() || at::autocast::is_autocast_enabled(at::kCUDA) || g->scalar_type() != at::kFloat ||
        x->scalar_type() != at::kFloat || w->scalar_type() != at::kFloat || g->dim() < 1 || x->dim() < 1 || w->dim() != 2 || g->numel() == 0 ||
        x->numel() == 0 || g->size(-1) != w->size(0) || x->size(-1) != w->size(1) || g->numel() / w->size(0) != x->numel() / w->size(1) ||
        !same_device(*g, *x) || !same_device(*g, *w))
        Py_RETURN_NONE;
    const int64_t N = w->size(0), K = w->size(1), M = g->numel() / N;
    if (!lib.tpq_f32_linear_grads_takes(ptr<float>(g), ptr<float>(x), ptr<float>(w), M, K, N)) Py_RETURN_NONE;
    const bool want_x = args[3] == Py_True, want_w = args[4] == Py_True;
    at::Tensor grad_x, grad_w;
    int status;
    {
        Enqueue q(*g);
        const size_t bytes = lib.tpq_f32_linear_grads_workspace_bytes(M, K, N, want_x, want_w);
        const at::Tensor scratch = bytes ? allocate({static_cast<int64_t>(bytes)}, at::kByte, *g) : at::Tensor();
        if (want_x) grad_x = allocate(x->sizes(), at::kFloat, *g);
        if (want_w) grad_w = allocate({N, K}, at::kFloat, *g);
        status = lib.tpq_f32_linear_grads(ptr<float>(g), ptr<float>(x), ptr<float>(w), M, K, N, want_x ? out_ptr<float>(grad_x) : nullptr,
                                          want_w ? out_ptr<float>(grad_w) : nullptr, bytes ? scratch.data_ptr() : nullptr, bytes, q.stream);
    }
    if (status != TPQ_OK) Py_RETURN_NONE;
    PyObject* first = want_x ? THPVariable_Wrap(std::move(grad_x)) : Py_NewRef(Py_None);
    PyObject* second = !first ? nullptr : want_w ? THPVariable_Wrap(std::move(grad_w)) : Py_NewRef(Py_None);
    return pair_of(first, second);
TPQ_CALL_END

// bind(handle): the entry points of the loaded library (a dlopen handle)
PyObject* bind(PyObject*, PyObject* handle_obj) {
    void* handle = PyLong_AsVoidPtr(handle_obj);
    if (!handle && PyErr_Occurred()) return nullptr;
    Library found;
#define TPQ_ENTRY(NAME)                                                                       \
    found.NAME = reinterpret_cast<decltype(found.NAME)>(dlsym(handle, #NAME));                \
    if (!found.NAME) {                                                                        \
        PyErr_SetString(PyExc_RuntimeError, "the kernel library does not export " #NAME);     \
        return nullptr;                                                                       \
    }
    TPQ_ENTRIES
#undef TPQ_ENTRY
    lib = found;
    Py_RETURN_NONE;
}

#define TPQ_METHOD(NAME) {#NAME, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(NAME)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {TPQ_METHOD(quantize_rowwise), TPQ_METHOD(int8_mm_dequant),  TPQ_METHOD(int8_linear),       TPQ_METHOD(ternary_linear),
                         TPQ_METHOD(lowbit_linear),
                         TPQ_METHOD(int4_mm),          TPQ_METHOD(lowbit_mm),        TPQ_METHOD(quantize_affine),   TPQ_METHOD(dequantize_affine),
                         TPQ_METHOD(linear_grads),
                         {"bind", bind, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef definition = {PyModuleDef_HEAD_INIT, "_calls", "The hot operators' host path as native calls.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__calls() { return PyModule_Create(&definition); }
