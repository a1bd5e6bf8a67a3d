// Host side of the serving operators in native code: argument checks, output allocation, the current stream and the call
// into libmdyfp8.so, for the calls whose kernels take a few microseconds (one call of a Python wrapper cost 7.5 us of
// host time against 2.3-4 us of kernel at one token).
//
// Every function takes the ordinary case - plain tensors on the current device, the layouts the operators document - and
// returns None for anything else, before anything is allocated or launched: the Python wrapper then goes its own way, which
// handles or rejects the rest with its own messages.  A call that the library rejects also returns None and is repeated there.
// Outputs come from torch's caching allocator on the current stream, as torch.empty gives them; nothing is kept between calls.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DefaultDtype.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/mdy_fp8.h"

namespace {

using at::ScalarType;
using at::Tensor;

constexpr ScalarType kE4m3 = ScalarType::Float8_e4m3fn;

// the tensor behind a Python object if it is a plain tensor on `device` (device < 0: on the current one, which is returned)
const Tensor* plain(PyObject* o, int& device) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.is_conj() || t.is_neg()) return nullptr;
    if (device < 0) device = (int)c10::hip::current_device();
    return t.get_device() == device ? &t : nullptr;
}

void* stream_of(int device) { return (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

Tensor make(at::IntArrayRef sizes, ScalarType dtype, const at::Device& dev) {
    return Tensor(at::detail::empty_cuda(sizes, dtype, dev, std::nullopt));
}
Tensor make_strided(at::IntArrayRef sizes, at::IntArrayRef strides, ScalarType dtype, const at::Device& dev) {
    return Tensor(at::detail::empty_strided_cuda(sizes, strides, dtype, dev));
}

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
          int64_t M, int64_t N, int64_t K, int out_code, const at::Device& dev, void* stream) {
    const int64_t bytes = mdy_fp8_gemm_workspace_bytes(M, N, K);
    Tensor ws;      // handed back as soon as the launch is enqueued: the allocator reuses it in stream order only
    if (bytes > 0) ws = make({bytes}, ScalarType::Byte, dev);
    return mdy_fp8_gemm_nt_ex(a, a_s, rs, cs, b, b_s, c, bias, bias_mode, M, N, K, MDY_FMT_E4M3, out_code, bytes > 0 ? ws.data_ptr() : nullptr,
                              bytes > 0 ? bytes : 0, stream) == 0;
}
// What the MFMA kernels need of a GEMM (anything else may run the scalar kernel, about which the wrapper warns)
bool gemm_shape_ok(int64_t M, int64_t N, int64_t K, int64_t rs, int64_t cs) {
    return M > 0 && N > 0 && K > 0 && K % 128 == 0 && K <= 65536 && rs >= 0 && cs >= 0 &&
           ((M - 1) * rs + (K / 128 - 1) * cs + 1) * 4 < ((int64_t)1 << 31);
}

// act_quant(x, block_size) -> (y, s)
PyObject* act_quant(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 2 || !PyLong_CheckExact(args[1])) Py_RETURN_NONE;
    int device = -1;
    const Tensor* x = plain(args[0], device);
    const long bs = PyLong_AsLong(args[1]);
    if (x == nullptr || bs < 8 || bs > 512 || (bs & (bs - 1)) != 0 || x->dim() < 1 || x->numel() == 0 || !x->is_contiguous()) Py_RETURN_NONE;
    const int xt = xt_code(x->scalar_type());
    const int64_t K = x->size(-1), M = x->numel() / K;
    if (xt < 0 || K % bs != 0) Py_RETURN_NONE;
    Tensor y = make(x->sizes(), kE4m3, x->device());
    auto sizes = x->sizes().vec();
    sizes.back() = K / bs;
    Tensor s = make(sizes, ScalarType::Float, x->device());
    if (mdy_act_quant_typed(x->data_ptr(), xt, (int)bs, y.data_ptr(), (float*)s.data_ptr(), M, K, K, M, K, K / bs, 1, MDY_QUANT_OFFICIAL, stream_of(device)) != 0)
        Py_RETURN_NONE;
    return tuple2(std::move(y), std::move(s));
}

// fp8_gemm(a, a_s, b, b_s, out_dtype or None, bias or None) -> c
PyObject* fp8_gemm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 6) Py_RETURN_NONE;
    int device = -1;
    const Tensor *a = plain(args[0], device), *as = plain(args[1], device), *b = plain(args[2], device), *bs = plain(args[3], device);
    if (a == nullptr || as == nullptr || b == nullptr || bs == nullptr) Py_RETURN_NONE;
    if (args[4] != Py_None && !THPDtype_Check(args[4])) Py_RETURN_NONE;
    const ScalarType out = args[4] == Py_None ? c10::get_default_dtype_as_scalartype() : reinterpret_cast<THPDtype*>(args[4])->scalar_type;
    const int code = out == ScalarType::BFloat16 ? MDY_DT_BF16 : out == ScalarType::Float ? MDY_DT_F32 : -1;
    if (code < 0 || a->scalar_type() != kE4m3 || b->scalar_type() != kE4m3 || as->scalar_type() != ScalarType::Float ||
        bs->scalar_type() != ScalarType::Float || a->dim() < 1 || b->dim() != 2 || bs->dim() != 2 || a->numel() == 0 || !a->is_contiguous() ||
        !b->is_contiguous() || !as->is_contiguous() || !bs->is_contiguous())
        Py_RETURN_NONE;
    const int64_t K = a->size(-1), M = a->numel() / K, N = b->size(0), KB = K / 128;
    const void* bias;
    if (b->size(1) != K || !gemm_shape_ok(M, N, K, KB, 1) || as->numel() != M * KB || bs->size(0) != cdiv(N, 128) || bs->size(1) != KB ||
        !aligned16(*a) || !aligned16(*b) || !bias_arg(args[5], N, device, bias))
        Py_RETURN_NONE;
    auto sizes = a->sizes().vec();
    sizes.back() = N;
    Tensor c = make(sizes, out, a->device());
    if (!gemm(a->data_ptr(), (const float*)as->data_ptr(), KB, 1, b->data_ptr(), (const float*)bs->data_ptr(), c.data_ptr(), bias, MDY_BIAS_IN_SUM, M, N,
              K, code, a->device(), stream_of(device)))
        Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(c));
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
    Tensor c = make({M, N}, ScalarType::BFloat16, a->device());
    if (!gemm(a->data_ptr(), (const float*)as->data_ptr(), rs, cs, b->data_ptr(), (const float*)bs->data_ptr(), c.data_ptr(), bias,
              (int)PyLong_AsLong(args[5]), M, N, K, MDY_DT_BF16, a->device(), stream_of(device)))
        Py_RETURN_NONE;
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
    if (!quantize_rows(r, y, s, stream_of(device))) Py_RETURN_NONE;
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
    void* stream = stream_of(device);
    Tensor y, s;
    if (!quantize_rows(r, y, s, stream)) Py_RETURN_NONE;
    auto sizes = r.t->sizes().vec();
    sizes.back() = N;
    Tensor c = make(sizes, ScalarType::BFloat16, r.t->device());
    if (!gemm(y.data_ptr(), (const float*)s.data_ptr(), 1, PM, b->data_ptr(), (const float*)bs->data_ptr(), c.data_ptr(), bias,
              (int)PyLong_AsLong(args[5]), r.M, N, PK, MDY_DT_BF16, r.t->device(), stream))
        Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(c));
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
    Tensor y, s;
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
    if (mdy_swiglu(x->data_ptr(), nullptr, y.data_ptr(), (float*)s.data_ptr(), M, N, 2 * N, PyLong_AsLong(args[1]) != 0, PM, PN, deep ? 1 : N / 128,
                   deep ? PM : 1, deep ? MDY_QUANT_DEEPLINEAR : MDY_QUANT_OFFICIAL, stream_of(device)) != 0)
        Py_RETURN_NONE;
    return tuple2(std::move(y), std::move(s));
}

// A C++ exception (an allocation that fails) becomes None as well: the wrapper meets it again and reports it as torch does.
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    try {
        return F(self, args, n);
    } catch (...) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

#define MDY_METHOD(F) {#F, (PyCFunction)(void (*)(void))guarded<F>, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {MDY_METHOD(act_quant), MDY_METHOD(fp8_gemm), MDY_METHOD(matmul), MDY_METHOD(quant_input),
                         MDY_METHOD(deep_linear), MDY_METHOD(silu_act_quant), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    if (mdy_fp8_abi_version() != MDY_FP8_ABI_VERSION) {
        PyErr_SetString(PyExc_ImportError, "libmdyfp8.so and _host.so were built from different sources: rebuild");
        return nullptr;
    }
    return PyModule_Create(&module);
}
