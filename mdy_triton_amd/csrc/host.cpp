// Host side of the operators in native code: argument checks, output allocation, the current stream and the call
// into libmdyfp8.so, for the calls whose kernels take a few microseconds (one call of a Python wrapper cost 7.5 us of
// host time against 2.3-4 us of kernel at one token; a small layer's training step made 110 us of them, one of 32 small
// experts 1070 us).
//
// Every function takes the ordinary case - plain tensors on the current device, the layouts the operators document, sizes that
// all of its products take - and returns None for anything else, before anything is allocated or launched: the Python wrapper
// then goes its own way, which handles or rejects the rest with its own messages.  What only the library or the allocator can
// refuse (a grid beyond the launch limits, memory that is not there) also returns None and is met again there.
// Outputs come from torch's caching allocator on the current stream, as torch.empty gives them; nothing is kept between calls.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <algorithm>
#include <cstdlib>
#include <cstring>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DefaultDtype.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Device.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/variable.h>

#include "../../include/mdy_fp8.h"

namespace {

using at::ScalarType;
using at::Tensor;

constexpr ScalarType kE4m3 = ScalarType::Float8_e4m3fn;

// Tensors whose value is not simply what lies at their address: lazy ones, wrappers of the function transforms, subclasses.
const c10::DispatchKeySet kWrapped({c10::DispatchKey::Conjugate, c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor, c10::DispatchKey::Python,
                                    c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                    c10::DispatchKey::NestedTensor});
// Something watches the calls of this thread: a trace, a dispatch mode.
bool watched() {
    return c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::Tracer) || c10::impl::TorchDispatchModeTLS::any_modes_set();
}

// the tensor behind a Python object if it is a plain tensor on `device` (device < 0: on the current one, which is returned), without
// a forward-mode tangent and with nothing watching: what bypasses an autograd function must not bypass these
const Tensor* plain(PyObject* o, int& device) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.key_set().has_any(kWrapped) || t._fw_grad(0).defined()) return nullptr;
    if (device < 0 && watched()) return nullptr;      // every function looks at its first tensor with device < 0
    if (device < 0) device = (int)c10::hip::current_device();
    return t.get_device() == device ? &t : nullptr;
}

bool flag(PyObject* o) { return PyObject_IsTrue(o) == 1; }

// Runs f without the interpreter lock: allocations and launches can wait (for memory, for room in the queue), and other threads
// run meanwhile.
template <typename F>
auto unlocked(F f) {
    struct Lock {
        PyThreadState* state = PyEval_SaveThread();
        ~Lock() { PyEval_RestoreThread(state); }
    } lock;
    return f();
}

void* stream_of(int device) { return (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

Tensor make(at::IntArrayRef sizes, ScalarType dtype, const at::Device& dev) {
    return Tensor(at::detail::empty_cuda(sizes, dtype, dev, std::nullopt));
}
Tensor make_strided(at::IntArrayRef sizes, at::IntArrayRef strides, ScalarType dtype, const at::Device& dev) {
    return Tensor(at::detail::empty_strided_cuda(sizes, strides, dtype, dev));
}

// Memory on the current stream for what no caller sees, from the same allocator (0.2 us; a tensor around it takes another 0.25).  It may go as soon as the
// launches that use it are enqueued: the allocator hands it out again in stream order only.
struct Scratch {
    c10::DataPtr p;
    explicit Scratch(int64_t bytes) {
        if (bytes > 0) p = c10::hip::HIPCachingAllocator::get()->allocate((size_t)bytes);
    }
    uint8_t* at(int64_t offset) const { return p.get() == nullptr ? nullptr : static_cast<uint8_t*>(p.get()) + offset; }
};
int64_t round_up(int64_t v, int64_t m) { return (v + m - 1) / m * m; }

PyObject* tuple2(Tensor&& a, Tensor&& b) {
    PyObject* r = PyTuple_New(2);
    if (r == nullptr) return nullptr;
    PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(a)));
    PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(b)));
    return r;
}

int xt_code(ScalarType t) {
    return t == ScalarType::BFloat16 ? MDY_XT_BF16 : t == ScalarType::Half ? MDY_XT_F16 : t == ScalarType::Float ? MDY_XT_F32 : -1;
}
int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }
bool aligned16(const Tensor& t) { return ((uintptr_t)t.data_ptr() & 15) == 0; }

// A bias argument: None or a contiguous bf16 [N] tensor.  False: something else.
bool bias_arg(PyObject* o, int64_t N, int& device, const void*& p) {
    p = nullptr;
    if (o == Py_None) return true;
    const Tensor* b = plain(o, device);
    if (b == nullptr || b->scalar_type() != ScalarType::BFloat16 || b->numel() != N || !b->is_contiguous()) return false;
    p = b->data_ptr();
    return true;
}

// c[M, N] = a . b^T with block scales; false when the library rejects the call
bool gemm(const void* a, const float* a_s, int64_t rs, int64_t cs, const void* b, const float* b_s, void* c, const void* bias, int bias_mode,
          int64_t M, int64_t N, int64_t K, int fmt, int out_code, void* stream) {
    const int64_t bytes = mdy_fp8_gemm_workspace_bytes(M, N, K);
    const Scratch ws(bytes);
    return mdy_fp8_gemm_nt_ex(a, a_s, rs, cs, b, b_s, c, bias, bias_mode, M, N, K, fmt, out_code, ws.at(0), bytes > 0 ? bytes : 0, stream) == 0;
}
// What the MFMA kernels need of a GEMM (anything else may run the scalar kernel, about which the wrapper warns)
bool gemm_shape_ok(int64_t M, int64_t N, int64_t K, int64_t rs, int64_t cs) {
    return M > 0 && N > 0 && K > 0 && M <= (1 << 30) && N <= (1 << 30) && K % 128 == 0 && K <= 65536 && rs >= 0 && cs >= 0 &&
           ((M - 1) * rs + (K / 128 - 1) * cs + 1) * 4 < ((int64_t)1 << 31);
}
// the same for the GEMM with row scales on both operands
bool row_scaled_shape_ok(int64_t M, int64_t N, int64_t K, int64_t a_rs, int64_t a_cs, int64_t b_rs, int64_t b_cs) {
    const auto extent_ok = [&](int64_t rows, int64_t rs, int64_t cs) { return rs >= 0 && cs >= 0 && ((rows - 1) * rs + (K / 128 - 1) * cs + 1) * 4 < ((int64_t)1 << 31); };
    return M > 0 && N > 0 && K > 0 && M <= (1 << 30) && N <= (1 << 30) && K % 128 == 0 && K <= (1 << 20) && extent_ok(M, a_rs, a_cs) && extent_ok(N, b_rs, b_cs);
}

ScalarType fmt_type(int fmt) { return fmt == MDY_FMT_E4M3 ? kE4m3 : ScalarType::Float8_e5m2; }
int fmt_mode(int fmt) { return fmt == MDY_FMT_E4M3 ? MDY_QUANT_OFFICIAL : MDY_QUANT_OFFICIAL_E5M2; }

// act_quant(x, block_size, fmt) -> (y, s)
PyObject* act_quant(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 3 || !PyLong_CheckExact(args[1]) || !PyLong_CheckExact(args[2])) Py_RETURN_NONE;
    const int fmt = (int)PyLong_AsLong(args[2]);
    int device = -1;
    const Tensor* x = plain(args[0], device);
    const long bs = PyLong_AsLong(args[1]);
    if (x == nullptr || bs < 8 || bs > 512 || (bs & (bs - 1)) != 0 || x->dim() < 1 || x->numel() == 0 || !x->is_contiguous()) Py_RETURN_NONE;
    const int xt = xt_code(x->scalar_type());
    const int64_t K = x->size(-1), M = x->numel() / K;
    if (xt < 0 || K % bs != 0) Py_RETURN_NONE;
    Tensor y, s;
    const int rc = unlocked([&] {
        y = make(x->sizes(), fmt_type(fmt), x->device());
        auto sizes = x->sizes().vec();
        sizes.back() = K / bs;
        s = make(sizes, ScalarType::Float, x->device());
        return mdy_act_quant_typed(x->data_ptr(), xt, (int)bs, y.data_ptr(), (float*)s.data_ptr(), M, K, K, M, K, K / bs, 1, fmt_mode(fmt), stream_of(device));
    });
    if (rc != 0) Py_RETURN_NONE;
    return tuple2(std::move(y), std::move(s));
}

// fp8_gemm(a [.., K], a_s, b, b_s, out_dtype or None, bias or None, fmt) -> c [.., N]
PyObject* fp8_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 7 || !PyLong_CheckExact(args[6])) Py_RETURN_NONE;
    const int fmt = (int)PyLong_AsLong(args[6]);
    int device = -1;
    const Tensor *a = plain(args[0], device), *as = plain(args[1], device), *b = plain(args[2], device), *bs = plain(args[3], device);
    if (a == nullptr || as == nullptr || b == nullptr || bs == nullptr) Py_RETURN_NONE;
    if (args[4] != Py_None && !THPDtype_Check(args[4])) Py_RETURN_NONE;
    const ScalarType out = args[4] == Py_None ? c10::get_default_dtype_as_scalartype() : reinterpret_cast<THPDtype*>(args[4])->scalar_type;
    const int code = out == ScalarType::BFloat16 ? MDY_DT_BF16 : out == ScalarType::Float ? MDY_DT_F32 : -1;
    if (code < 0 || a->scalar_type() != fmt_type(fmt) || b->scalar_type() != fmt_type(fmt) || as->scalar_type() != ScalarType::Float ||
        bs->scalar_type() != ScalarType::Float || a->dim() < 1 || b->dim() != 2 || bs->dim() != 2 || a->numel() == 0 || !a->is_contiguous() ||
        !b->is_contiguous() || !as->is_contiguous() || !bs->is_contiguous())
        Py_RETURN_NONE;
    const int64_t K = a->size(-1), M = a->numel() / K, N = b->size(0), KB = K / 128;
    const void* bias;
    if (b->size(1) != K || !gemm_shape_ok(M, N, K, KB, 1) || as->numel() != M * KB || bs->size(0) != cdiv(N, 128) || bs->size(1) != KB ||
        !aligned16(*a) || !aligned16(*b) || !bias_arg(args[5], N, device, bias))
        Py_RETURN_NONE;
    Tensor c;
    const bool ok = unlocked([&] {
        auto sizes = a->sizes().vec();
        sizes.back() = N;
        c = make(sizes, out, a->device());
        return gemm(a->data_ptr(), (const float*)as->data_ptr(), KB, 1, b->data_ptr(), (const float*)bs->data_ptr(), c.data_ptr(), bias, MDY_BIAS_IN_SUM,
                    M, N, K, fmt, code, stream_of(device));
    });
    if (!ok) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(c));
}

// weight_dequant(x [N, K], s, block_size, out_dtype or None) -> y
PyObject* weight_dequant(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 4 || !PyLong_CheckExact(args[2]) || (args[3] != Py_None && !THPDtype_Check(args[3]))) Py_RETURN_NONE;
    int device = -1;
    const Tensor *x = plain(args[0], device), *s = plain(args[1], device);
    const int64_t bs = PyLong_AsLongLong(args[2]);
    const ScalarType out = args[3] == Py_None ? c10::get_default_dtype_as_scalartype() : reinterpret_cast<THPDtype*>(args[3])->scalar_type;
    const int code = out == ScalarType::BFloat16 ? MDY_DT_BF16 : out == ScalarType::Float ? MDY_DT_F32 : -1;
    if (x == nullptr || s == nullptr || code < 0 || bs < 8 || (bs & (bs - 1)) != 0 || x->scalar_type() != kE4m3 || s->scalar_type() != ScalarType::Float ||
        x->dim() != 2 || s->dim() != 2 || x->numel() == 0 || !x->is_contiguous() || !s->is_contiguous() || s->size(0) != cdiv(x->size(0), bs) ||
        s->size(1) != cdiv(x->size(1), bs) || bs > (1 << 20))
        Py_RETURN_NONE;
    Tensor y;
    const int rc = unlocked([&] {
        y = make(x->sizes(), out, x->device());
        return mdy_weight_dequant_block(x->data_ptr(), (const float*)s->data_ptr(), y.data_ptr(), x->size(0), x->size(1), (int)bs, code, stream_of(device));
    });
    if (rc != 0) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(y));
}

// matmul(qa [>= M, K], sa logical [>= M, K/128], qb [>= N, K], sb, bias or None, bias_mode, M, N) -> bf16 [M, N]: the first M and N
// rows of operands that the quantizers padded (M, N < 0: all of them)
PyObject* matmul(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 8 || !PyLong_CheckExact(args[5]) || !PyLong_CheckExact(args[6]) || !PyLong_CheckExact(args[7])) Py_RETURN_NONE;
    int device = -1;
    const Tensor *a = plain(args[0], device), *as = plain(args[1], device), *b = plain(args[2], device), *bs = plain(args[3], device);
    if (a == nullptr || as == nullptr || b == nullptr || bs == nullptr) Py_RETURN_NONE;
    if (a->scalar_type() != kE4m3 || b->scalar_type() != kE4m3 || as->scalar_type() != ScalarType::Float || bs->scalar_type() != ScalarType::Float ||
        a->dim() != 2 || b->dim() != 2 || as->dim() != 2 || bs->dim() != 2 || !a->is_contiguous() || !b->is_contiguous() || !bs->is_contiguous())
        Py_RETURN_NONE;
    const int64_t m = PyLong_AsLongLong(args[6]), nn = PyLong_AsLongLong(args[7]);
    const int64_t M = m < 0 ? a->size(0) : m, N = nn < 0 ? b->size(0) : nn;
    const int64_t K = a->size(1), KB = K / 128, rs = as->stride(0), cs = as->stride(1);
    const void* bias;
    if (b->size(1) != K || !gemm_shape_ok(M, N, K, rs, cs) || M > a->size(0) || N > b->size(0) || as->size(1) != KB || bs->size(1) != KB ||
        (m < 0 ? as->size(0) != M : as->size(0) < M) || (nn < 0 ? bs->size(0) != cdiv(N, 128) : bs->size(0) < cdiv(N, 128)) || !aligned16(*a) || !aligned16(*b) || !bias_arg(args[4], N, device, bias))
        Py_RETURN_NONE;
    const int mode = (int)PyLong_AsLong(args[5]);
    Tensor c;
    const bool ok = unlocked([&] {
        c = make({M, N}, ScalarType::BFloat16, a->device());
        return gemm(a->data_ptr(), (const float*)as->data_ptr(), rs, cs, b->data_ptr(), (const float*)bs->data_ptr(), c.data_ptr(), bias, mode, M, N, K,
                    MDY_FMT_E4M3, MDY_DT_BF16, stream_of(device));
    });
    if (!ok) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(c));
}

// a 2-D activation whose rows are contiguous, as the forward quantizer of the DeepLinear dialect takes it
struct Rows {
    const Tensor* t;
    int64_t M, K, stride;
    int xt;
};
bool rows_arg(PyObject* o, int& device, Rows& r) {
    r.t = plain(o, device);
    if (r.t == nullptr || r.t->dim() < 1 || r.t->numel() == 0) return false;
    r.xt = xt_code(r.t->scalar_type());
    r.K = r.t->size(-1);
    r.M = r.t->numel() / r.K;
    if (r.xt < 0) return false;
    if (r.t->is_contiguous()) {
        r.stride = r.K;
        return true;
    }
    if (r.t->dim() != 2 || r.t->stride(1) != 1) return false;
    r.stride = r.t->stride(0);
    return r.stride >= r.K;
}

// per-token quantization with padding: y [PM, PN] e4m3fn and s, logical [PM, PN/128] with strides (1, PM)
bool quantize_rows(const Rows& r, Tensor& y, Tensor& s, void* stream) {
    const int64_t PM = cdiv(r.M, 4) * 4, PN = cdiv(r.K, 256) * 256;
    y = make({PM, PN}, kE4m3, r.t->device());
    s = make_strided({PM, PN / 128}, {1, PM}, ScalarType::Float, r.t->device());
    return mdy_act_quant_typed(r.t->data_ptr(), r.xt, 128, y.data_ptr(), (float*)s.data_ptr(), r.M, r.K, r.stride, PM, PN, 1, PM, MDY_QUANT_DEEPLINEAR,
                               stream) == 0;
}

// quant_input(x 2-D) -> (y, s)
PyObject* quant_input(PyObject*, PyObject* const* args, Py_ssize_t n) {
    int device = -1;
    Rows r;
    if (n != 1 || !rows_arg(args[0], device, r) || r.t->dim() != 2) Py_RETURN_NONE;
    Tensor y, s;
    if (!unlocked([&] { return quantize_rows(r, y, s, stream_of(device)); })) Py_RETURN_NONE;
    return tuple2(std::move(y), std::move(s));
}

// deep_linear(x [..., K], qw [PN, PK], sw, N, bias or None, bias_mode) -> bf16 [..., N]: quant_input and the GEMM of a layer whose
// weight is quantized already, without gradients
PyObject* deep_linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 6 || !PyLong_CheckExact(args[3]) || !PyLong_CheckExact(args[5])) Py_RETURN_NONE;
    int device = -1;
    Rows r;
    if (!rows_arg(args[0], device, r)) Py_RETURN_NONE;
    const Tensor *b = plain(args[1], device), *bs = plain(args[2], device);
    const int64_t N = PyLong_AsLongLong(args[3]), PK = cdiv(r.K, 256) * 256, KB = PK / 128, PM = cdiv(r.M, 4) * 4;
    const void* bias;
    if (b == nullptr || bs == nullptr || b->scalar_type() != kE4m3 || bs->scalar_type() != ScalarType::Float || b->dim() != 2 || bs->dim() != 2 ||
        !b->is_contiguous() || !bs->is_contiguous() || b->size(0) < N || b->size(1) != PK || bs->size(0) < cdiv(N, 128) || bs->size(1) != KB ||
        !gemm_shape_ok(r.M, N, PK, 1, PM) || !aligned16(*b) || !bias_arg(args[4], N, device, bias))
        Py_RETURN_NONE;
    const int mode = (int)PyLong_AsLong(args[5]);
    Tensor c;
    const bool ok = unlocked([&] {
        void* stream = stream_of(device);
        // the quantized rows, their scales and the product's workspace
        const int64_t s_at = round_up(PM * PK, 512), ws_at = round_up(s_at + PM * KB * 4, 512), bytes = mdy_fp8_gemm_workspace_bytes(r.M, N, PK);
        const Scratch room(ws_at + std::max<int64_t>(bytes, 0));
        if (mdy_act_quant_typed(r.t->data_ptr(), r.xt, 128, room.at(0), (float*)room.at(s_at), r.M, r.K, r.stride, PM, PK, 1, PM, MDY_QUANT_DEEPLINEAR,
                                stream) != 0)
            return false;
        auto sizes = r.t->sizes().vec();
        sizes.back() = N;
        c = make(sizes, ScalarType::BFloat16, r.t->device());
        return mdy_fp8_gemm_nt_ex(room.at(0), (const float*)room.at(s_at), 1, PM, b->data_ptr(), (const float*)bs->data_ptr(), c.data_ptr(), bias, mode, r.M,
                                  N, PK, MDY_FMT_E4M3, MDY_DT_BF16, bytes > 0 ? room.at(ws_at) : nullptr, bytes > 0 ? bytes : 0, stream) == 0;
    });
    if (!ok) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(c));
}

// parameter(module, name, getattr) -> module.<name>.  What torch.nn.Module keeps under that name is taken without the failed lookup that comes in front of
// it (0.25 us), but only where nothing comes in front of it: not an attribute of the type (a subclass's property) or of the instance, not a lookup of the
// type's own; getattr is torch.nn.Module's.  The type is asked on each call (by the interpreter's own cache): a class may change.
PyObject* parameter(PyObject*, PyObject* const* args, Py_ssize_t n) {
    static PyObject *const lookup = PyUnicode_InternFromString("__getattribute__"), *const missing = PyUnicode_InternFromString("__getattr__"),
                    *const parameters = PyUnicode_InternFromString("_parameters");
    if (n != 3 || lookup == nullptr || missing == nullptr || parameters == nullptr) Py_RETURN_NONE;
    PyObject *module = args[0], *name = args[1];
    PyTypeObject* type = Py_TYPE(module);
    PyObject** dict = _PyObject_GetDictPtr(module);
    if (dict != nullptr && *dict != nullptr && PyUnicode_CheckExact(name) && _PyType_Lookup(type, name) == nullptr && _PyType_Lookup(type, missing) == args[2] &&
        _PyType_Lookup(type, lookup) == _PyType_Lookup(&PyBaseObject_Type, lookup) && PyDict_GetItemWithError(*dict, name) == nullptr) {
        PyObject* kept = PyDict_GetItemWithError(*dict, parameters);
        PyObject* found = kept != nullptr && PyDict_CheckExact(kept) ? PyDict_GetItemWithError(kept, name) : nullptr;
        if (found != nullptr) {
            Py_INCREF(found);
            return found;
        }
    }
    return PyErr_Occurred() ? nullptr : PyObject_GetAttr(module, name);
}

// cached_weight(weight, cache, with_transpose) -> the quantized copies (y, s, yt, st) that DeepLinear keeps, if they are the weight's: cache is
// ((data_ptr, version, shape, device), copies, fingerprint).  None where that has to be looked at more closely, and where
// MDY_FP8_CHECK_WEIGHT_CACHE asks for it.
PyObject* cached_weight(PyObject*, PyObject* const* args, Py_ssize_t n) {
    int device = -1;
    if (n != 3 || !PyTuple_CheckExact(args[1]) || PyTuple_GET_SIZE(args[1]) != 3) Py_RETURN_NONE;
    const Tensor* w = plain(args[0], device);
    PyObject *key = PyTuple_GET_ITEM(args[1], 0), *copies = PyTuple_GET_ITEM(args[1], 1);
    if (w == nullptr || w->is_inference() || !PyTuple_CheckExact(key) || PyTuple_GET_SIZE(key) != 4 || !PyTuple_CheckExact(copies) || PyTuple_GET_SIZE(copies) != 4)
        Py_RETURN_NONE;
    PyObject *ptr = PyTuple_GET_ITEM(key, 0), *version = PyTuple_GET_ITEM(key, 1), *shape = PyTuple_GET_ITEM(key, 2), *dev = PyTuple_GET_ITEM(key, 3);
    if (!PyLong_CheckExact(ptr) || !PyLong_CheckExact(version) || !PyTuple_Check(shape) || PyTuple_GET_SIZE(shape) != w->dim() || !THPDevice_Check(dev)) Py_RETURN_NONE;
    if (PyLong_AsUnsignedLongLong(ptr) != (unsigned long long)(uintptr_t)w->const_data_ptr() || PyLong_AsLongLong(version) != (long long)w->_version() ||
        reinterpret_cast<THPDevice*>(dev)->device != w->device())
        Py_RETURN_NONE;
    for (int64_t d = 0; d < w->dim(); ++d)
        if (!PyLong_CheckExact(PyTuple_GET_ITEM(shape, d)) || PyLong_AsLongLong(PyTuple_GET_ITEM(shape, d)) != w->size(d)) Py_RETURN_NONE;
    if (flag(args[2]) && PyTuple_GET_ITEM(copies, 2) == Py_None) Py_RETURN_NONE;
    const char* check = std::getenv("MDY_FP8_CHECK_WEIGHT_CACHE");
    if (check != nullptr && check[0] != 0 && std::strcmp(check, "0") != 0) Py_RETURN_NONE;
    Py_INCREF(copies);
    return copies;
}

// ---------------------------------------------------------------------------------------------------------------------------
// training
// ---------------------------------------------------------------------------------------------------------------------------

// Thrown when the library rejects a call in the middle of a composite one for what could not be told beforehand: the whole call
// returns None and is repeated by the wrapper, whose own checks say what is wrong.  (Launches already made wrote outputs that
// nobody has seen.)
struct Rejected {};
void done(int rc) {
    if (rc != 0) throw Rejected();
}

// a matrix: a 2-D tensor of any strides, or the flattened rows of a contiguous one
struct Mat {
    const Tensor* t = nullptr;
    int64_t M = 0, K = 0, rs = 0, cs = 1;
    int xt = -1;
    const void* data() const { return t->data_ptr(); }
    const at::Device dev() const { return t->device(); }
};
bool mat_arg(PyObject* o, int& device, Mat& m) {
    m.t = plain(o, device);
    if (m.t == nullptr || m.t->dim() < 1 || m.t->numel() == 0) return false;
    m.xt = xt_code(m.t->scalar_type());
    m.K = m.t->size(-1);
    m.M = m.t->numel() / m.K;
    if (m.t->dim() == 2) {
        m.rs = m.t->stride(0);
        m.cs = m.t->stride(1);
    } else {
        if (!m.t->is_contiguous()) return false;
        m.rs = m.K;
    }
    return m.xt >= 0;
}
float* f32(const Tensor& t) { return t.defined() ? (float*)t.data_ptr() : nullptr; }
void* raw(const Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

// row-wise copy y, s and transposed copy yt, st of one matrix (undefined: not asked for)
struct Copies {
    Tensor y, s, yt, st;
};

// DeepLinear dialect, padded to multiples of 256 (fp8.py:46-77, 122-161): s logical [PM, PK/128], strides (1, PM); t_mode 0: st
// logical [PK, PM/128], strides (1, PK); t_mode 1: st [PK/128, PM/128].  col_sum (t_mode 0): bf16 [K], the columns' sums.
Copies deep_copies(const Mat& x, int t_mode, const Tensor& col_sum, void* stream) {
    const int64_t PM = cdiv(x.M, 256) * 256, PK = cdiv(x.K, 256) * 256;
    Copies c;
    c.y = make({PM, PK}, kE4m3, x.dev());
    c.s = make_strided({PM, PK / 128}, {1, PM}, ScalarType::Float, x.dev());
    c.yt = make({PK, PM}, kE4m3, x.dev());
    c.st = t_mode == 0 ? make_strided({PK, PM / 128}, {1, PK}, ScalarType::Float, x.dev()) : make({PK / 128, PM / 128}, ScalarType::Float, x.dev());
    if (col_sum.defined()) {
        Tensor part = make({PM / 128, PK}, ScalarType::Float, x.dev());
        done(mdy_quant_transpose_colsum(x.data(), raw(c.y), f32(c.s), raw(c.yt), f32(c.st), x.M, x.K, x.rs, x.cs, PM, PK, PM, MDY_QUANT_DEEPLINEAR,
                                        f32(part), raw(col_sum), stream));
    } else {
        done(mdy_quant_transpose_typed(x.data(), x.xt, raw(c.y), f32(c.s), raw(c.yt), f32(c.st), x.M, x.K, x.rs, x.cs, PM, PK, PM, t_mode, stream));
    }
    return c;
}

// official dialect: y [PM, K], s [PM, K/128], yt [K, PM], st [K, PM/128], PM = M to a multiple of 128, K % 128 == 0
Copies official_copies(const Mat& x, bool rows, int fmt, const Tensor& col_sum, void* stream) {
    const int64_t PM = cdiv(x.M, 128) * 128;
    Copies c;
    if (rows) {
        c.y = make({PM, x.K}, fmt_type(fmt), x.dev());
        c.s = make({PM, x.K / 128}, ScalarType::Float, x.dev());
    }
    c.yt = make({x.K, PM}, fmt_type(fmt), x.dev());
    c.st = make({x.K, PM / 128}, ScalarType::Float, x.dev());
    if (col_sum.defined()) {
        Tensor part = make({PM / 128, x.K}, ScalarType::Float, x.dev());
        done(mdy_quant_transpose_colsum(x.data(), raw(c.y), f32(c.s), raw(c.yt), f32(c.st), x.M, x.K, x.rs, x.cs, PM, x.K, 0, fmt_mode(fmt), f32(part),
                                        raw(col_sum), stream));
    } else {
        done(mdy_act_quant_transpose(x.data(), x.xt, raw(c.y), f32(c.s), raw(c.yt), f32(c.st), x.M, x.K, x.rs, x.cs, PM, x.K, fmt_mode(fmt), stream));
    }
    return c;
}

// 128x128 blocks of a weight, rows padded to PN and columns to PK
Copies weight_copies(const Mat& w, bool rows, bool transposed, int64_t PN, int64_t PK, ScalarType type, int mode, void* stream) {
    Copies c;
    if (rows) {
        c.y = make({PN, PK}, type, w.dev());
        c.s = make({PN / 128, PK / 128}, ScalarType::Float, w.dev());
    }
    if (transposed) {
        c.yt = make({PK, PN}, type, w.dev());
        c.st = make({PK / 128, PN / 128}, ScalarType::Float, w.dev());
    }
    done(mdy_weight_quant_typed(w.data(), w.xt, raw(c.y), f32(c.s), raw(c.yt), f32(c.st), w.M, w.K, w.rs, w.cs, PN, PK, mode, stream));
    return c;
}

// bf16 [sizes] = a . b^T, M rows of a (scales a_s[m * rs + kb * cs]) against N rows of b; the callers have asked gemm_shape_ok
Tensor product(const Tensor& a, const Tensor& a_s, int64_t rs, int64_t cs, const Tensor& b, const Tensor& b_s, const void* bias, int bias_mode,
               int64_t M, int64_t N, int64_t K, int fmt, at::IntArrayRef sizes, void* stream) {
    Tensor c = make(sizes, ScalarType::BFloat16, a.device());
    const int64_t bytes = mdy_fp8_gemm_workspace_bytes(M, N, K);
    const Scratch ws(bytes);
    done(mdy_fp8_gemm_nt_ex(raw(a), f32(a_s), rs, cs, raw(b), f32(b_s), raw(c), bias, bias_mode, M, N, K, fmt, MDY_DT_BF16, ws.at(0), bytes > 0 ? bytes : 0,
                            stream));
    return c;
}

// bf16 [M, N] = a . b^T with a scale per row and 128 columns on both sides
Tensor row_scaled(const Tensor& a, const Tensor& a_s, const Tensor& b, const Tensor& b_s, int64_t M, int64_t N, int64_t K, int fmt, void* stream) {
    Tensor c = make({M, N}, ScalarType::BFloat16, a.device());
    const int64_t bytes = mdy_fp8_gemm_rowscaled_workspace_bytes(M, N, K);
    const Scratch ws(bytes);
    done(mdy_fp8_gemm_nt_rowscaled_ws(raw(a), f32(a_s), a_s.stride(0), a_s.stride(1), raw(b), f32(b_s), b_s.stride(0), b_s.stride(1), raw(c), M, N, K, fmt,
                                      MDY_DT_BF16, ws.at(0), bytes > 0 ? bytes : 0, stream));
    return c;
}

PyObject* wrap_or_none(const Tensor& t) {
    if (!t.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(t);
}
PyObject* tuple_of(std::initializer_list<Tensor> ts) {
    PyObject* r = PyTuple_New((Py_ssize_t)ts.size());
    if (r == nullptr) return nullptr;
    Py_ssize_t i = 0;
    for (const Tensor& t : ts) PyTuple_SET_ITEM(r, i++, wrap_or_none(t));
    return r;
}
bool tensor_or_none(PyObject* o, int& device, Tensor& t) {
    if (o == Py_None) return true;
    const Tensor* p = plain(o, device);
    if (p == nullptr) return false;
    t = *p;
    return true;
}

// Are y [>= rows, cols] and s [>= s_rows, s_cols] a quantized copy and its fp32 scales as the kernels read them?  What comes back from
// autograd's saved tensors has been through the user's hooks, and a cached copy through the caller's hands.
bool copy_ok(const Tensor& y, const Tensor& s, ScalarType type, int64_t rows, int64_t cols, int64_t s_rows, int64_t s_cols) {
    return y.defined() && s.defined() && y.scalar_type() == type && s.scalar_type() == ScalarType::Float && y.dim() == 2 && s.dim() == 2 &&
           y.size(0) >= rows && y.size(1) == cols && s.size(0) >= s_rows && s.size(1) == s_cols && y.is_contiguous() && s.is_contiguous() && aligned16(y);
}

// ordinary(tensors...) -> True if every one is a plain tensor here: an autograd function may then be passed by
PyObject* ordinary(PyObject*, PyObject* const* args, Py_ssize_t n) {
    int device = -1;
    for (Py_ssize_t i = 0; i < n; ++i)
        if (plain(args[i], device) == nullptr) Py_RETURN_NONE;
    Py_RETURN_TRUE;
}

// deep_forward(x, weight, cached (y, s, yt, st) or None, bias or None, bias_mode, need_dx, need_dw) -> (out, xt, xt_s, wt, wt_s):
// fp8.py:316-329; the transposed copies that the backward pass will need, else None
PyObject* deep_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 7 || !PyLong_CheckExact(args[4])) Py_RETURN_NONE;
    int device = -1;
    Mat x, w;
    if (!mat_arg(args[0], device, x) || !mat_arg(args[1], device, w) || w.t->dim() != 2 || w.K != x.K) Py_RETURN_NONE;
    const bool need_dx = flag(args[5]), need_dw = flag(args[6]);
    const int64_t N = w.M, PK = cdiv(x.K, 256) * 256, PN = cdiv(N, need_dx ? 256 : 128) * (need_dx ? 256 : 128);
    Copies wc;
    if (args[2] != Py_None) {
        if (!PyTuple_CheckExact(args[2]) || PyTuple_GET_SIZE(args[2]) != 4 || !tensor_or_none(PyTuple_GET_ITEM(args[2], 0), device, wc.y) ||
            !tensor_or_none(PyTuple_GET_ITEM(args[2], 1), device, wc.s) || !tensor_or_none(PyTuple_GET_ITEM(args[2], 2), device, wc.yt) ||
            !tensor_or_none(PyTuple_GET_ITEM(args[2], 3), device, wc.st) || !wc.y.defined() || !wc.s.defined() || (need_dx && !wc.yt.defined()))
            Py_RETURN_NONE;
        if (wc.y.scalar_type() != kE4m3 || wc.s.scalar_type() != ScalarType::Float || wc.y.dim() != 2 || wc.s.dim() != 2 || wc.y.size(0) < N ||
            wc.y.size(1) != PK || wc.s.size(0) < cdiv(N, 128) || wc.s.size(1) != PK / 128 || !wc.y.is_contiguous() || !wc.s.is_contiguous() ||
            !aligned16(wc.y))
            Py_RETURN_NONE;
    }
    const void* bias;
    if (!bias_arg(args[3], N, device, bias)) Py_RETURN_NONE;
    if (!need_dw && (x.cs != 1 || x.rs < x.K)) Py_RETURN_NONE;
    const int64_t pad = need_dw ? 256 : 4, PM = cdiv(x.M, pad) * pad;
    if (!gemm_shape_ok(x.M, N, PK, 1, PM)) Py_RETURN_NONE;
    const int mode = (int)PyLong_AsLong(args[4]);
    Copies xc;
    Tensor out = unlocked([&] {
        void* stream = stream_of(device);
        if (need_dw) {
            xc = deep_copies(x, 1, Tensor(), stream);
        } else if (!quantize_rows(Rows{x.t, x.M, x.K, x.rs, x.xt}, xc.y, xc.s, stream)) {
            throw Rejected();
        }
        if (!wc.y.defined()) wc = weight_copies(w, true, need_dx, PN, PK, kE4m3, MDY_QUANT_DEEPLINEAR, stream);
        auto sizes = x.t->sizes().vec();
        sizes.back() = N;
        return product(xc.y, xc.s, 1, PM, wc.y, wc.s, bias, mode, x.M, N, PK, MDY_FMT_E4M3, sizes, stream);
    });
    return tuple_of({out, xc.yt, xc.st, wc.yt, wc.st});
}

// deep_backward(dy, xt, xt_s, wt, wt_s, K, need_dx, need_dw, need_db) -> (dx [M, K], dw [N, K], db [N]): fp8.py:330-343
PyObject* deep_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 9 || !PyLong_CheckExact(args[5])) Py_RETURN_NONE;
    int device = -1;
    Mat dy;
    Copies xc, wc;
    if (!mat_arg(args[0], device, dy) || dy.xt != MDY_XT_BF16 || !tensor_or_none(args[1], device, xc.yt) || !tensor_or_none(args[2], device, xc.st) ||
        !tensor_or_none(args[3], device, wc.yt) || !tensor_or_none(args[4], device, wc.st))
        Py_RETURN_NONE;
    const bool need_dx = flag(args[6]), need_dw = flag(args[7]), need_db = flag(args[8]);
    const int64_t M = dy.M, N = dy.K, K = PyLong_AsLongLong(args[5]), PM = cdiv(M, 256) * 256, PN = cdiv(N, 256) * 256;
    if ((need_dx && !copy_ok(wc.yt, wc.st, kE4m3, K, PN, cdiv(K, 128), PN / 128)) || (need_dw && !copy_ok(xc.yt, xc.st, kE4m3, K, PM, cdiv(K, 128), PM / 128)))
        Py_RETURN_NONE;
    if ((need_dx && !gemm_shape_ok(M, K, PN, 1, PM)) || (need_dw && !gemm_shape_ok(N, K, PM, 1, PN))) Py_RETURN_NONE;
    Tensor db, dx, dw;
    unlocked([&] {
        void* stream = stream_of(device);
        if (need_db) db = make({N}, ScalarType::BFloat16, dy.dev());
        const Copies dc = deep_copies(dy, 0, db, stream);
        if (need_dx) dx = product(dc.y, dc.s, 1, PM, wc.yt, wc.st, nullptr, 0, M, K, PN, MDY_FMT_E4M3, {M, K}, stream);
        if (need_dw) dw = product(dc.yt, dc.st, 1, PN, xc.yt, xc.st, nullptr, 0, N, K, PM, MDY_FMT_E4M3, {N, K}, stream);
    });
    return tuple_of({dx, dw, db});
}

// An empty tensor that shares t's version counter.  Saved for a backward pass in place of t it has autograd refuse the pass when t
// was changed in place in between, and keeps none of t's memory.
Tensor version_of(const Tensor& t) {
    Tensor g = make({0}, t.scalar_type(), t.device());
    torch::autograd::impl::set_version_counter(g, torch::autograd::impl::version_counter(t));
    return g;
}
PyObject* version_guard(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 1 || !THPVariable_Check(args[0])) Py_RETURN_NONE;
    const Tensor& t = THPVariable_Unpack(args[0]);
    if (!t.defined() || t.is_inference()) Py_RETURN_NONE;
    return THPVariable_Wrap(version_of(t));
}

// official_forward(x, w, bias or None, fmt, keep_xt, keep_wt, versions) -> (y, xt, xt_s, wt, wt_s, version of x, version of w):
// fp8_kernel.py:261-272; None for what is not asked for
PyObject* official_forward(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 7 || !PyLong_CheckExact(args[3])) Py_RETURN_NONE;
    int device = -1;
    Mat x, w;
    if (!mat_arg(args[0], device, x) || !mat_arg(args[1], device, w) || w.t->dim() != 2 || w.K != x.K || x.K % 128 != 0 || w.M % 128 != 0) Py_RETURN_NONE;
    const int fmt = (int)PyLong_AsLong(args[3]);
    const bool keep_xt = flag(args[4]), keep_wt = flag(args[5]), versions = flag(args[6]);
    const int64_t N = w.M, K = x.K;
    const void* bias;
    if (!bias_arg(args[2], N, device, bias)) Py_RETURN_NONE;
    if ((!keep_xt && (x.cs != 1 || x.rs != K)) || !gemm_shape_ok(x.M, N, K, K / 128, 1)) Py_RETURN_NONE;
    if (versions && (x.t->is_inference() || w.t->is_inference())) Py_RETURN_NONE;      // save_for_backward refuses them: the wrapper lets it
    Copies xc, wc;
    Tensor y = unlocked([&] {
        void* stream = stream_of(device);
        if (keep_xt) {
            xc = official_copies(x, true, fmt, Tensor(), stream);
        } else {
            xc.y = make({x.M, K}, fmt_type(fmt), x.dev());
            xc.s = make({x.M, K / 128}, ScalarType::Float, x.dev());
            done(mdy_act_quant_typed(x.data(), x.xt, 128, raw(xc.y), f32(xc.s), x.M, K, K, x.M, K, K / 128, 1, fmt_mode(fmt), stream));
        }
        wc = weight_copies(w, true, keep_wt, N, K, fmt_type(fmt), fmt_mode(fmt), stream);
        auto sizes = x.t->sizes().vec();
        sizes.back() = N;
        return product(xc.y, xc.s, K / 128, 1, wc.y, wc.s, bias, MDY_BIAS_IN_SUM, x.M, N, K, fmt, sizes, stream);
    });
    return tuple_of({y, xc.yt, xc.st, wc.yt, wc.st, versions ? version_of(*x.t) : Tensor(), versions ? version_of(*w.t) : Tensor()});
}

// official_backward(dy, xt, xt_s, wt, wt_s, fmt, need_dx, need_dw, need_db, w or None) -> (dx, dw, db): fp8_kernel.py:274-301; wt, wt_s
// None: from w
PyObject* official_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 10 || !PyLong_CheckExact(args[5])) Py_RETURN_NONE;
    int device = -1;
    Mat dy;
    Copies xc, wc;
    if (!mat_arg(args[0], device, dy) || dy.xt != MDY_XT_BF16 || dy.K % 128 != 0 || !tensor_or_none(args[1], device, xc.yt) ||
        !tensor_or_none(args[2], device, xc.st) || !tensor_or_none(args[3], device, wc.yt) || !tensor_or_none(args[4], device, wc.st))
        Py_RETURN_NONE;
    const int fmt = (int)PyLong_AsLong(args[5]);
    const bool need_dx = flag(args[6]), need_dw = flag(args[7]), need_db = flag(args[8]);
    const int64_t M = dy.M, N = dy.K, PM = cdiv(M, 128) * 128;
    if (!need_dx && !need_dw) Py_RETURN_NONE;
    Mat w;      // to be quantized here
    if (need_dx && !wc.yt.defined()) {
        if (!mat_arg(args[9], device, w) || w.t->dim() != 2 || w.M != N || w.K % 128 != 0) Py_RETURN_NONE;
    } else if (need_dx && (wc.yt.dim() != 2 || !copy_ok(wc.yt, wc.st, fmt_type(fmt), 0, N, cdiv(wc.yt.size(0), 128), N / 128))) {
        Py_RETURN_NONE;
    }
    if (need_dw && (!xc.yt.defined() || xc.yt.dim() != 2 || !copy_ok(xc.yt, xc.st, fmt_type(fmt), 0, PM, xc.yt.size(0), PM / 128))) Py_RETURN_NONE;
    const int64_t K = w.t != nullptr ? w.K : need_dx ? wc.yt.size(0) : 0;
    if ((need_dx && !gemm_shape_ok(M, K, N, N / 128, 1)) || (need_dw && !row_scaled_shape_ok(N, xc.yt.size(0), PM, PM / 128, 1, PM / 128, 1))) Py_RETURN_NONE;
    Tensor db, dx, dw;
    unlocked([&] {
        void* stream = stream_of(device);
        if (need_db) db = make({N}, ScalarType::BFloat16, dy.dev());
        const Copies dc = official_copies(dy, need_dx, fmt, db, stream);
        if (w.t != nullptr) wc = weight_copies(w, false, true, N, K, fmt_type(fmt), fmt_mode(fmt), stream);
        if (need_dx) dx = product(dc.y, dc.s, N / 128, 1, wc.yt, wc.st, nullptr, 0, M, K, N, fmt, {M, K}, stream);
        if (need_dw) dw = row_scaled(dc.yt, dc.st, xc.yt, xc.st, N, xc.yt.size(0), PM, fmt, stream);
    });
    return tuple_of({dx, dw, db});
}

// official_copies(x, rows, fmt) -> (y or None, s or None, yt, st), padded rows
PyObject* act_copies(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 3 || !PyLong_CheckExact(args[2])) Py_RETURN_NONE;
    int device = -1;
    Mat x;
    if (!mat_arg(args[0], device, x) || x.t->dim() != 2 || x.K % 128 != 0) Py_RETURN_NONE;
    const bool rows = flag(args[1]);
    const int fmt = (int)PyLong_AsLong(args[2]);
    const Copies c = unlocked([&] { return official_copies(x, rows, fmt, Tensor(), stream_of(device)); });
    return tuple_of({c.y, c.s, c.yt, c.st});
}

// block_copies(w, rows, transposed, fmt) -> (y, s, yt, st), None for what is not asked for
PyObject* block_copies(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 4 || !PyLong_CheckExact(args[3])) Py_RETURN_NONE;
    int device = -1;
    Mat w;
    const bool rows = flag(args[1]), transposed = flag(args[2]);
    if (!mat_arg(args[0], device, w) || w.t->dim() != 2 || w.K % 128 != 0 || w.M % 128 != 0 || (!rows && !transposed)) Py_RETURN_NONE;
    const int fmt = (int)PyLong_AsLong(args[3]);
    const Copies c = unlocked([&] { return weight_copies(w, rows, transposed, w.M, w.K, fmt_type(fmt), fmt_mode(fmt), stream_of(device)); });
    return tuple_of({c.y, c.s, c.yt, c.st});
}

// quant_weight(w, only_forward) -> (y, s, yt, st) of the DeepLinear dialect (fp8.py:206-247)
PyObject* quant_weight(PyObject*, PyObject* const* args, Py_ssize_t n) {
    int device = -1;
    Mat w;
    if (n != 2 || !mat_arg(args[0], device, w) || w.t->dim() != 2) Py_RETURN_NONE;
    const bool only_forward = flag(args[1]);
    const int64_t b = only_forward ? 128 : 256;
    const Copies c = unlocked([&] {
        return weight_copies(w, true, !only_forward, cdiv(w.M, b) * b, cdiv(w.K, 256) * 256, kE4m3, MDY_QUANT_DEEPLINEAR, stream_of(device));
    });
    return tuple_of({c.y, c.s, c.yt, c.st});
}

// quant_transposed(x, t_mode) -> (y, s, yt, st) of the DeepLinear dialect's two training quantizers
PyObject* quant_transposed(PyObject*, PyObject* const* args, Py_ssize_t n) {
    int device = -1;
    Mat x;
    if (n != 2 || !PyLong_CheckExact(args[1]) || !mat_arg(args[0], device, x) || x.t->dim() != 2) Py_RETURN_NONE;
    const int t_mode = (int)PyLong_AsLong(args[1]);
    const Copies c = unlocked([&] { return deep_copies(x, t_mode, Tensor(), stream_of(device)); });
    return tuple_of({c.y, c.s, c.yt, c.st});
}

// row_scaled(x [M, K], w [N, K], sx, sw, fmt) -> bf16 [M, N]; K % 128 == 0, both scales one per row and 128 columns, any strides
PyObject* row_scaled_product(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 5 || !PyLong_CheckExact(args[4])) Py_RETURN_NONE;
    int device = -1;
    const Tensor *a = plain(args[0], device), *b = plain(args[1], device), *as = plain(args[2], device), *bs = plain(args[3], device);
    if (a == nullptr || b == nullptr || as == nullptr || bs == nullptr) Py_RETURN_NONE;
    const int fmt = (int)PyLong_AsLong(args[4]);
    if (a->scalar_type() != fmt_type(fmt) || b->scalar_type() != fmt_type(fmt) || as->scalar_type() != ScalarType::Float ||
        bs->scalar_type() != ScalarType::Float || a->dim() != 2 || b->dim() != 2 || as->dim() != 2 || bs->dim() != 2 || a->numel() == 0 ||
        b->numel() == 0 || !a->is_contiguous() || !b->is_contiguous() || !aligned16(*a) || !aligned16(*b))
        Py_RETURN_NONE;
    const int64_t M = a->size(0), K = a->size(1), N = b->size(0);
    if (b->size(1) != K || as->size(0) != M || as->size(1) != K / 128 || bs->size(0) != N || bs->size(1) != K / 128 ||
        !row_scaled_shape_ok(M, N, K, as->stride(0), as->stride(1), bs->stride(0), bs->stride(1)))
        Py_RETURN_NONE;
    return THPVariable_Wrap(unlocked([&] { return row_scaled(*a, *as, *b, *bs, M, N, K, fmt, stream_of(device)); }));
}

// silu_fwd(x [..., 2N], gate_first) -> bf16 [..., N];  silu_bwd(dy, x, gate_first) -> dx like x
PyObject* silu_fwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
    int device = -1;
    if (n != 2 || !PyLong_CheckExact(args[1])) Py_RETURN_NONE;
    const Tensor* x = plain(args[0], device);
    if (x == nullptr || x->scalar_type() != ScalarType::BFloat16 || x->dim() < 1 || x->numel() == 0 || !x->is_contiguous() || x->size(-1) % 2 != 0)
        Py_RETURN_NONE;
    auto sizes = x->sizes().vec();
    const int64_t N = sizes.back() / 2, M = x->numel() / (2 * N);
    sizes.back() = N;
    const int gate_first = flag(args[1]);
    Tensor y = unlocked([&] {
        Tensor t = make(sizes, ScalarType::BFloat16, x->device());
        done(mdy_swiglu(x->data_ptr(), raw(t), nullptr, nullptr, M, N, 2 * N, gate_first, 0, 0, 0, 0, 0, stream_of(device)));
        return t;
    });
    return THPVariable_Wrap(std::move(y));
}
PyObject* silu_bwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
    int device = -1;
    if (n != 3 || !PyLong_CheckExact(args[2])) Py_RETURN_NONE;
    const Tensor *dy = plain(args[0], device), *x = plain(args[1], device);
    if (x == nullptr || dy == nullptr || x->scalar_type() != ScalarType::BFloat16 || dy->scalar_type() != ScalarType::BFloat16 || x->dim() < 1 ||
        x->numel() == 0 || !x->is_contiguous() || !dy->is_contiguous() || x->size(-1) % 2 != 0 || dy->numel() * 2 != x->numel())
        Py_RETURN_NONE;
    const int64_t N = x->size(-1) / 2, M = x->numel() / (2 * N);
    const int gate_first = flag(args[2]);
    Tensor dx = unlocked([&] {
        Tensor t = make(x->sizes(), ScalarType::BFloat16, x->device());
        done(mdy_swiglu_bwd(x->data_ptr(), dy->data_ptr(), raw(t), M, N, 2 * N, gate_first, stream_of(device)));
        return t;
    });
    return THPVariable_Wrap(std::move(dx));
}

// ---------------------------------------------------------------------------------------------------------------------------
// expert groups
// ---------------------------------------------------------------------------------------------------------------------------
bool ints_arg(PyObject* o, std::vector<int64_t>& v) {
    const bool list = PyList_CheckExact(o);
    if (!list && !PyTuple_CheckExact(o)) return false;
    const Py_ssize_t n = list ? PyList_GET_SIZE(o) : PyTuple_GET_SIZE(o);
    if (n > (1 << 20)) return false;
    v.resize((size_t)n);
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* e = list ? PyList_GET_ITEM(o, i) : PyTuple_GET_ITEM(o, i);
        if (!PyLong_CheckExact(e)) return false;
        const long long x = PyLong_AsLongLong(e);
        if (x < 0 || x > ((int64_t)1 << 40)) return false;      // also an overflow, cleared by the caller; sums of them fit 64 bits
        v[(size_t)i] = x;
    }
    return true;
}
int64_t sum_of(const std::vector<int64_t>& v) {
    int64_t t = 0;
    for (int64_t x : v) t += x;
    return t;
}

// A tensor over a part of `buffer` with a version counter of its own (a view shares its base's): parts that do not overlap are changed
// and saved for backward passes without each other.
Tensor part_of(const Tensor& buffer, int64_t offset, at::IntArrayRef sizes, at::IntArrayRef strides) {
    auto impl = c10::make_intrusive<c10::TensorImpl>(c10::TensorImpl::VIEW, c10::Storage(buffer.storage()), buffer.key_set(), buffer.dtype());
    impl->set_storage_offset(offset);
    impl->set_sizes_and_strides(sizes, strides);
    return Tensor(std::move(impl));
}

// group_cast(x [M, N], m_splits) -> (y, s, [yt], [st]): megatron_patchs/fp8_matmul.py:218-247.  Every group's copy is a tensor of its own;
// the scales, a thirty-second of the copies, lie in one allocation (8 groups: 15.6 -> 12 us a call).
PyObject* group_cast(PyObject*, PyObject* const* args, Py_ssize_t n) {
    int device = -1;
    Mat x;
    std::vector<int64_t> splits;
    if (n != 2 || !mat_arg(args[0], device, x) || x.t->dim() != 2 || !ints_arg(args[1], splits) || sum_of(splits) != x.M || x.K % 256 != 0) Py_RETURN_NONE;
    for (int64_t m : splits)
        if (m % 256 != 0) Py_RETURN_NONE;
    const size_t G = splits.size();
    Tensor y, s;
    std::vector<Tensor> yt(G), st(G);
    unlocked([&] {
        y = make({x.M, x.K}, kE4m3, x.dev());
        s = make_strided({x.M, x.K / 128}, {1, x.M}, ScalarType::Float, x.dev());
        std::vector<void*> ytp(G);
        std::vector<float*> stp(G);
        const Tensor scales = make({x.M / 128 * x.K}, ScalarType::Float, x.dev());
        int64_t row = 0;
        for (size_t g = 0; g < G; ++g) {
            yt[g] = make({x.K, splits[g]}, kE4m3, x.dev());
            st[g] = part_of(scales, row / 128 * x.K, {x.K, splits[g] / 128}, {1, x.K});
            ytp[g] = raw(yt[g]);
            stp[g] = f32(scales) + row / 128 * x.K;
            row += splits[g];
        }
        done(mdy_quant_transpose_grouped(x.data(), x.xt, raw(y), f32(s), ytp.data(), stp.data(), splits.data(), (int64_t)G, x.K, x.rs, x.cs,
                                         stream_of(device)));
    });
    PyObject* r = PyTuple_New(4);
    PyObject *lt = PyList_New((Py_ssize_t)G), *ls = PyList_New((Py_ssize_t)G);
    if (r == nullptr || lt == nullptr || ls == nullptr) return nullptr;
    for (size_t g = 0; g < G; ++g) {
        PyList_SET_ITEM(lt, (Py_ssize_t)g, THPVariable_Wrap(std::move(yt[g])));
        PyList_SET_ITEM(ls, (Py_ssize_t)g, THPVariable_Wrap(std::move(st[g])));
    }
    PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(y)));
    PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(s)));
    PyTuple_SET_ITEM(r, 2, lt);
    PyTuple_SET_ITEM(r, 3, ls);
    return r;
}

// grouped_matmul(qa [M, K], sa, qb [G, N, K], sb, m_splits, bias [G, N] or None) -> bf16 [M, N]
PyObject* grouped_matmul(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 6) Py_RETURN_NONE;
    int device = -1;
    const Tensor *a = plain(args[0], device), *as = plain(args[1], device), *b = plain(args[2], device), *bs = plain(args[3], device);
    std::vector<int64_t> splits;
    if (a == nullptr || as == nullptr || b == nullptr || bs == nullptr || !ints_arg(args[4], splits)) Py_RETURN_NONE;
    if (a->scalar_type() != kE4m3 || b->scalar_type() != kE4m3 || as->scalar_type() != ScalarType::Float || bs->scalar_type() != ScalarType::Float ||
        a->dim() != 2 || b->dim() != 3 || as->dim() != 2 || bs->dim() != 3 || !a->is_contiguous() || !b->is_contiguous() || !bs->is_contiguous())
        Py_RETURN_NONE;
    const int64_t M = a->size(0), K = a->size(1), G = b->size(0), N = b->size(1), KB = K / 128;
    const void* bias;
    if (b->size(2) != K || !gemm_shape_ok(M, N, K, as->stride(0), as->stride(1)) || as->size(0) != M || as->size(1) != KB || bs->size(0) != G ||
        bs->size(1) != cdiv(N, 128) || bs->size(2) != KB || (int64_t)splits.size() != G || sum_of(splits) != M || !bias_arg(args[5], G * N, device, bias))
        Py_RETURN_NONE;
    if (args[5] != Py_None && THPVariable_Unpack(args[5]).dim() != 2) Py_RETURN_NONE;
    Tensor c = unlocked([&] {
        Tensor t = make({M, N}, ScalarType::BFloat16, a->device());
        done(mdy_fp8_grouped_gemm_nt(raw(*a), f32(*as), as->stride(0), as->stride(1), raw(*b), f32(*bs), raw(t), bias, splits.data(), G, N, K, MDY_DT_BF16,
                                     stream_of(device)));
        return t;
    });
    return THPVariable_Wrap(std::move(c));
}

// move_rows(x [rows, H] contiguous, m_splits, unpad, multiple) -> padded or unpadded rows
PyObject* move_rows(PyObject*, PyObject* const* args, Py_ssize_t n) {
    int device = -1;
    std::vector<int64_t> splits;
    if (n != 4 || !PyLong_CheckExact(args[3])) Py_RETURN_NONE;
    const Tensor* x = plain(args[0], device);
    const int64_t multiple = PyLong_AsLongLong(args[3]);
    if (x == nullptr || x->dim() != 2 || x->numel() == 0 || !x->is_contiguous() || multiple < 1 || multiple > (1 << 20) || !ints_arg(args[1], splits)) Py_RETURN_NONE;
    const bool unpad = flag(args[2]);
    int64_t padded = 0;
    for (int64_t m : splits) padded += cdiv(m, multiple) * multiple;
    const int64_t rows = sum_of(splits);
    if (x->size(0) != (unpad ? padded : rows)) Py_RETURN_NONE;
    if ((unpad ? rows : padded) == 0) Py_RETURN_NONE;
    Tensor y = unlocked([&] {
        Tensor t = make({unpad ? rows : padded, x->size(1)}, x->scalar_type(), x->device());
        done(mdy_group_pad_rows(x->data_ptr(), raw(t), splits.data(), (int64_t)splits.size(), x->size(1) * (int64_t)x->element_size(), multiple,
                                unpad ? 1 : 0, stream_of(device)));
        return t;
    });
    return THPVariable_Wrap(std::move(y));
}

// silu_act_quant(x [..., 2N] bf16 contiguous, gate_first, deeplinear) -> (y, s) as the wrapper of that name returns them
PyObject* silu_act_quant(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 3 || !PyLong_CheckExact(args[1]) || !PyLong_CheckExact(args[2])) Py_RETURN_NONE;
    int device = -1;
    const Tensor* x = plain(args[0], device);
    if (x == nullptr || x->scalar_type() != ScalarType::BFloat16 || x->dim() < 1 || x->numel() == 0 || !x->is_contiguous() || x->size(-1) % 2 != 0)
        Py_RETURN_NONE;
    const bool deep = PyLong_AsLong(args[2]) != 0;
    const int64_t N = x->size(-1) / 2, M = x->numel() / (2 * N);
    const int64_t PM = deep ? cdiv(M, 4) * 4 : M, PN = deep ? cdiv(N, 256) * 256 : N;
    if (PN % 128 != 0) Py_RETURN_NONE;
    const int gate_first = flag(args[1]);
    Tensor y, s;
    const int rc = unlocked([&] {
        if (deep) {
            y = make({PM, PN}, kE4m3, x->device());
            s = make_strided({PM, PN / 128}, {1, PM}, ScalarType::Float, x->device());
        } else {
            auto sizes = x->sizes().vec();
            sizes.back() = N;
            y = make(sizes, kE4m3, x->device());
            sizes.back() = N / 128;
            s = make(sizes, ScalarType::Float, x->device());
        }
        return mdy_swiglu(x->data_ptr(), nullptr, y.data_ptr(), (float*)s.data_ptr(), M, N, 2 * N, gate_first, PM, PN, deep ? 1 : N / 128,
                          deep ? PM : 1, deep ? MDY_QUANT_DEEPLINEAR : MDY_QUANT_OFFICIAL, stream_of(device));
    });
    if (rc != 0) Py_RETURN_NONE;
    return tuple2(std::move(y), std::move(s));
}

// mlp(x [..., K], qwu [>= 2I, PK], swu, 2I, qwd [>= N, PI], swd, N, gate_first, deep) -> bf16 [..., N]: the forward pass of a SwiGLU MLP on
// e4m3fn weights that are quantized already: x quantized (fp8.py:164-204 with deep, act_quant without), up/gate projection,
// activation quantized (silu_act_quant), down projection
PyObject* mlp(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 9 || !PyLong_CheckExact(args[3]) || !PyLong_CheckExact(args[6])) Py_RETURN_NONE;
    int device = -1;
    Rows r;
    if (!rows_arg(args[0], device, r)) Py_RETURN_NONE;
    const Tensor *qwu = plain(args[1], device), *swu = plain(args[2], device), *qwd = plain(args[4], device), *swd = plain(args[5], device);
    if (qwu == nullptr || swu == nullptr || qwd == nullptr || swd == nullptr) Py_RETURN_NONE;
    const int64_t M = r.M, N2 = PyLong_AsLongLong(args[3]), I = N2 / 2, N = PyLong_AsLongLong(args[6]);
    const int gate_first = flag(args[7]);
    const bool deep = flag(args[8]);
    const int64_t pad = deep ? 256 : 1, K = cdiv(r.K, pad) * pad, PI = cdiv(I, pad) * pad, PM = deep ? cdiv(M, 4) * 4 : M;
    const int64_t rs = deep ? 1 : K / 128, cs = deep ? PM : 1, act_rs = deep ? 1 : PI / 128;
    if (N2 < 2 || N2 % 2 != 0 || N < 1 || PI % 128 != 0 || (!deep && r.stride != K) || !copy_ok(*qwu, *swu, kE4m3, N2, K, cdiv(N2, 128), K / 128) ||
        !copy_ok(*qwd, *swd, kE4m3, N, PI, cdiv(N, 128), PI / 128) || !gemm_shape_ok(M, N2, K, rs, cs) || !gemm_shape_ok(M, N, PI, act_rs, cs))
        Py_RETURN_NONE;
    const int mode = deep ? MDY_QUANT_DEEPLINEAR : MDY_QUANT_OFFICIAL;
    auto sizes = r.t->sizes().vec();
    sizes.back() = N;
    return THPVariable_Wrap(unlocked([&] {
        const at::Device dev = r.t->device();
        void* stream = stream_of(device);
        const int64_t bytes = mdy_fp8_gemm_swiglu_workspace_bytes(M, N2, K), s_at = round_up(PM * K, 512), ws_at = round_up(s_at + PM * (K / 128) * 4, 512),
                      act_s_at = round_up(PM * PI, 512);
        const Scratch act(act_s_at + PM * (PI / 128) * 4);      // quantized activation and its scales, written [PI / 128, PM] with deep
        {
            const Scratch room(ws_at + std::max<int64_t>(bytes, 0));      // quantized x, its scales, workspace: the down projection finds room where these were
            done(mdy_act_quant_typed(r.t->data_ptr(), r.xt, 128, room.at(0), (float*)room.at(s_at), M, r.K, r.stride, PM, K, rs, cs, mode, stream));
            done(mdy_fp8_gemm_swiglu(room.at(0), (float*)room.at(s_at), rs, cs, raw(*qwu), f32(*swu), M, N2, K, gate_first, act.at(0), (float*)act.at(act_s_at), PM,
                                     PI, act_rs, cs, mode, bytes > 0 ? room.at(ws_at) : nullptr, bytes > 0 ? bytes : 0, stream));
        }
        Tensor c = make(sizes, ScalarType::BFloat16, dev);
        if (!gemm(act.at(0), (const float*)act.at(act_s_at), act_rs, cs, raw(*qwd), f32(*swd), raw(c), nullptr, 0, M, N, PI, MDY_FMT_E4M3, MDY_DT_BF16, stream))
            throw Rejected();
        return c;
    }));
}

// mlp_backward(dy [M, H'], x [M, H], w_up_gate [2I, H], w_down [H', I], gate_first, fmt, deep) -> (dx, dw_up_gate, dw_down): the backward pass of
// a SwiGLU MLP that kept its input only (fp8_kernel.py:452-494): the up/gate projection again, then the activation and the gradients
PyObject* mlp_backward(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 7 || !PyLong_CheckExact(args[5])) Py_RETURN_NONE;
    int device = -1;
    Mat dy, x, wu, wd;
    if (!mat_arg(args[0], device, dy) || !mat_arg(args[1], device, x) || !mat_arg(args[2], device, wu) || !mat_arg(args[3], device, wd)) Py_RETURN_NONE;
    const int gate_first = flag(args[4]), fmt = (int)PyLong_AsLong(args[5]);
    const bool deep = flag(args[6]);
    const int64_t M = x.M, H = x.K, N2 = wu.M, I = wd.K, O = wd.M, tile = deep ? 256 : 128;
    if (dy.t->dim() != 2 || x.t->dim() != 2 || wu.t->dim() != 2 || wd.t->dim() != 2 || dy.xt != MDY_XT_BF16 || dy.M != M || dy.K != O || wu.K != H ||
        N2 != 2 * I || I % 128 != 0 || (!deep && (H % 128 != 0 || O % 128 != 0)) || (deep && fmt != MDY_FMT_E4M3))
        Py_RETURN_NONE;
    const auto padded = [&](int64_t v) { return cdiv(v, tile) * tile; };
    const int64_t PM = padded(M), PH = padded(H), PI = padded(I), PO = padded(O);      // 2 I is a multiple of 256
    const auto block_ok = [&](int64_t m, int64_t nn, int64_t k) { return deep ? gemm_shape_ok(m, nn, k, 1, PM) : gemm_shape_ok(m, nn, k, k / 128, 1); };
    const auto row_ok = [&](int64_t m, int64_t nn, int64_t pm) {      // of a weight's gradient: contraction over the tokens
        return deep ? gemm_shape_ok(m, nn, PM, 1, pm) : row_scaled_shape_ok(m, nn, PM, PM / 128, 1, PM / 128, 1);
    };
    if (!block_ok(M, N2, PH) || !block_ok(M, I, PO) || !block_ok(M, H, N2) || !row_ok(O, I, PO) || !row_ok(N2, H, N2)) Py_RETURN_NONE;
    const int mode = deep ? MDY_QUANT_DEEPLINEAR : fmt_mode(fmt);
    const ScalarType type = fmt_type(fmt);
    Tensor dx, dwu, dwd;
    unlocked([&] {
        void* stream = stream_of(device);
        const at::Device dev = x.dev();
        const auto copies = [&](const Mat& m, int t_mode) { return deep ? deep_copies(m, t_mode, Tensor(), stream) : official_copies(m, true, fmt, Tensor(), stream); };
        // m rows of a against the block-quantized b; a's K blocks as columns of scales
        const auto blocks = [&](const Tensor& a, const Tensor& as, const Copies& w, bool transposed, int64_t nn, int64_t k) {
            return product(a, as, deep ? 1 : k / 128, deep ? PM : 1, transposed ? w.yt : w.y, transposed ? w.st : w.s, nullptr, 0, M, nn, k, fmt, {M, nn}, stream);
        };
        const auto weight_gradient = [&](const Tensor& a, const Tensor& as, const Tensor& b, const Tensor& bs, int64_t m, int64_t nn, int64_t pm) {
            return deep ? product(a, as, 1, pm, b, bs, nullptr, 0, m, nn, PM, fmt, {m, nn}, stream) : row_scaled(a, as, b, bs, m, nn, PM, fmt, stream);
        };
        Copies xc = copies(x, 1), wuc = weight_copies(wu, true, true, N2, PH, type, mode, stream);
        Tensor up_gate = blocks(xc.y, xc.s, wuc, false, N2, PH);
        xc.y.reset(), xc.s.reset(), wuc.y.reset(), wuc.s.reset();
        Copies dc = copies(dy, 0);
        Tensor dact = blocks(dc.y, dc.s, weight_copies(wd, false, true, PO, PI, type, mode, stream), true, I, PO);
        dc.y.reset(), dc.s.reset();
        const Tensor act_t = make({PI, PM}, type, dev), act_ts = make({deep ? PI / 128 : PI, PM / 128}, ScalarType::Float, dev);
        Copies gc;
        gc.y = make({PM, N2}, type, dev);
        gc.s = make({PM * (N2 / 128)}, ScalarType::Float, dev);
        gc.yt = make({N2, PM}, type, dev);
        gc.st = deep ? make_strided({N2, PM / 128}, {1, N2}, ScalarType::Float, dev) : make({N2, PM / 128}, ScalarType::Float, dev);
        done(mdy_swiglu_bwd_quant(raw(up_gate), raw(dact), raw(act_t), f32(act_ts), raw(gc.y), f32(gc.s), raw(gc.yt), f32(gc.st), M, I, gate_first, PM, PI, mode,
                                  stream));
        up_gate.reset(), dact.reset();
        dwd = weight_gradient(dc.yt, dc.st, act_t, act_ts, O, I, PO);
        dx = blocks(gc.y, gc.s, wuc, true, H, N2);
        dwu = weight_gradient(gc.yt, gc.st, xc.yt, xc.st, N2, H, N2);
    });
    return tuple_of({dx, dwu, dwd});
}

// A C++ exception (a call that the library rejects, an allocation that fails) becomes None as well: the wrapper meets it again and reports it as torch does.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    try {
        PyObject* r = F(self, args, n);
        if (r == Py_None) PyErr_Clear();      // a number that did not fit: the wrapper meets it again
        return r;
    } catch (...) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

#define MDY_METHOD(F) {#F, (PyCFunction)(void (*)(void))guarded<F>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {MDY_METHOD(act_quant), MDY_METHOD(fp8_gemm), MDY_METHOD(weight_dequant), MDY_METHOD(matmul), MDY_METHOD(quant_input),
                         MDY_METHOD(deep_linear), MDY_METHOD(parameter), MDY_METHOD(cached_weight), MDY_METHOD(silu_act_quant), MDY_METHOD(deep_forward), MDY_METHOD(deep_backward),
                         MDY_METHOD(official_forward), MDY_METHOD(ordinary), MDY_METHOD(version_guard), MDY_METHOD(official_backward), MDY_METHOD(act_copies), MDY_METHOD(block_copies),
                         MDY_METHOD(quant_weight), MDY_METHOD(quant_transposed), MDY_METHOD(row_scaled_product), MDY_METHOD(silu_fwd),
                         MDY_METHOD(silu_bwd), MDY_METHOD(mlp), MDY_METHOD(mlp_backward), MDY_METHOD(group_cast), MDY_METHOD(grouped_matmul), MDY_METHOD(move_rows),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    if (mdy_fp8_abi_version() != MDY_FP8_ABI_VERSION) {
        PyErr_SetString(PyExc_ImportError, "libmdyfp8.so and _host.so were built from different sources: rebuild");
        return nullptr;
    }
    return PyModule_Create(&module);
}
