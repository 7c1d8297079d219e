// Native caller of the C ABI (include/aiter_amd.h) for the Python package: one
// CPython function per entry point, with the entry's own argument list.
//
// Why: a decode call runs 4-10 us on the GPU, while building its tensor
// descriptors field by field through ctypes cost 3 us per tensor, 12-16 us per
// entry.  Here the descriptors are filled from the tensor's own fields on the
// C++ stack.
//
// A function takes the entry's arguments without the trailing stream: tensors
// (None: NULL), ints, floats, strings (None: NULL).  The stream is the current
// one of the first tensor's device (0 without a GPU tensor).  Returns True, or
// False without calling when an argument is something else (the caller then
// goes through ctypes, which reports it).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <string>
#include <tuple>
#include <type_traits>
#include <utility>

#include "aiter_amd.h"

namespace {

int dtype_id(at::ScalarType t) {
    switch (t) {
        case at::kHalf: return AITER_DTYPE_fp16;
        case at::kBFloat16: return AITER_DTYPE_bf16;
        case at::kFloat: return AITER_DTYPE_fp32;
        case at::kUInt32: return AITER_DTYPE_u32;
        case at::kInt: return AITER_DTYPE_i32;
        case at::kShort: return AITER_DTYPE_i16;
        case at::kChar: return AITER_DTYPE_i8;
        case at::kByte: return AITER_DTYPE_u8;
        case at::kLong: return AITER_DTYPE_i64;
        case at::kUInt64: return AITER_DTYPE_u64;
        case at::kFloat8_e4m3fn: return AITER_DTYPE_fp8;
#if AITER_AMD_TORCH_E8M0
        case at::kFloat8_e8m0fnu: return AITER_DTYPE_fp8_e8m0;
#endif
#if AITER_AMD_TORCH_FP4
        case at::kFloat4_e2m1fn_x2: return AITER_DTYPE_fp4x2;
#endif
        default: return -1;
    }
}

enum Conv { kOk, kElsewhere, kError };   // kElsewhere: not for this path

struct Call {
    int device = -2;   // device of the first tensor (-1: CPU; -2: none yet)
};

template <typename T>
struct Arg;

template <>
struct Arg<aiter_tensor_t*> {
    aiter_tensor_t t{};
    aiter_tensor_t* value = nullptr;

    Conv from(PyObject* o, Call& call) {
        if (o == Py_None) return kOk;
        if (!THPVariable_CheckExact(o)) return kElsewhere;
        const at::Tensor& x = THPVariable_Unpack(o);
        const int64_t nd = x.dim();
        const int dt = dtype_id(x.scalar_type());
        if (nd > 8 || dt < 0 || x.layout() != at::kStrided) return kElsewhere;
        t.numel = (size_t)x.numel();
        t.ptr = t.numel ? x.data_ptr() : nullptr;
        t.ndim = (int)nd;
        const auto sizes = x.sizes(), strides = x.strides();
        for (int64_t i = 0; i < nd; ++i) {
            t.shape[i] = sizes[i];
            t.strides[i] = strides[i];
        }
        t.dtype = decltype(t.dtype)(dt);
        t.device_id = x.is_cuda() ? (int)x.get_device() : -1;
        if (call.device == -2) call.device = t.device_id;
        value = &t;
        return kOk;
    }
};

template <>
struct Arg<const char*> {
    const char* value = nullptr;
    Conv from(PyObject* o, Call&) {
        if (o == Py_None) return kOk;
        if (!PyUnicode_Check(o)) return kElsewhere;
        value = PyUnicode_AsUTF8(o);
        return value ? kOk : kError;
    }
};

template <>
struct Arg<int> {
    int value = 0;
    Conv from(PyObject* o, Call&) {
        if (!PyLong_Check(o)) return kElsewhere;
        const long v = PyLong_AsLong(o);
        if (v == -1 && PyErr_Occurred()) PyErr_Clear();
        else if (v == (int)v) {
            value = (int)v;
            return kOk;
        }
        return kElsewhere;
    }
};

template <>
struct Arg<float> {
    float value = 0;
    Conv from(PyObject* o, Call&) {
        if (PyFloat_Check(o)) value = (float)PyFloat_AS_DOUBLE(o);
        else if (PyLong_Check(o)) value = (float)PyLong_AsDouble(o);
        else return kElsewhere;
        return PyErr_Occurred() ? kError : kOk;
    }
};

template <typename>
struct Entry;

template <typename... A>
struct Entry<int (*)(A...)> {
    // every argument but the trailing stream
    static constexpr size_t kArgs = sizeof...(A) - 1;
    using All = std::tuple<A...>;
    static_assert(std::is_same_v<std::tuple_element_t<kArgs, All>, aiter_stream_t>, "the stream comes last");

    template <size_t... I>
    static PyObject* run(const char* name, int (*fn)(A...), PyObject* const* args, Py_ssize_t n,
                         std::index_sequence<I...>) {
        if (n != (Py_ssize_t)kArgs) Py_RETURN_FALSE;
        std::tuple<Arg<std::tuple_element_t<I, All>>...> v;
        Call call;
        Conv c = kOk;
        ((c = c == kOk ? std::get<I>(v).from(args[I], call) : c), ...);
        if (c == kError) return nullptr;
        if (c == kElsewhere) Py_RETURN_FALSE;
        aiter_stream_t st = call.device >= 0
                                ? (aiter_stream_t)c10::hip::getCurrentHIPStream((c10::DeviceIndex)call.device).stream()
                                : aiter_stream_t{};
        int rc;
        std::string msg;
        Py_BEGIN_ALLOW_THREADS;
        rc = fn(std::get<I>(v).value..., st);
        if (rc != 0) {
            const char* m = aiter_get_last_error();
            msg = m ? m : "unknown error";
        }
        Py_END_ALLOW_THREADS;
        if (rc != 0) {
            PyErr_Format(PyExc_RuntimeError, "%s failed: %s", name, msg.c_str());
            return nullptr;
        }
        Py_RETURN_TRUE;
    }
};

template <auto Fn>
PyObject* entry(const char* name, PyObject* const* args, Py_ssize_t n) {
    using E = Entry<decltype(Fn)>;
    try {
        return E::run(name, Fn, args, n, std::make_index_sequence<E::kArgs>{});
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}

#define AA_ENTRY(F)                                                                  \
    {#F, (PyCFunction)(void (*)(void))(+[](PyObject*, PyObject* const* a, Py_ssize_t n) -> PyObject* { \
         return entry<&F>(#F, a, n);                                                 \
     }), METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    AA_ENTRY(gemm_a4w4_asm), AA_ENTRY(gemm_a4w4_blockscale), AA_ENTRY(gemm_a4w4_asm_noalloc),
    AA_ENTRY(mxfp8_mxfp4_gemm_asm), AA_ENTRY(mxfp4_gemm_asm), AA_ENTRY(gemm_a16w16_asm), AA_ENTRY(opus_gemm),
    AA_ENTRY(opus_gemm_a16w16_tune), AA_ENTRY(batched_gemm_bf16), AA_ENTRY(batched_gemm_bf16_tune),
    AA_ENTRY(dynamic_per_group_scaled_quant), AA_ENTRY(quant_mxfp4), AA_ENTRY(dynamic_mxfp4_quant),
    AA_ENTRY(dynamic_mxfp8_quant), AA_ENTRY(fused_rms_mx_quant), AA_ENTRY(fused_gemm_afp4wfp4_mul_add),
    AA_ENTRY(fused_gemm_afp4wfp4_split_cat), AA_ENTRY(fused_gemm_afp4wfp4_a16w16), AA_ENTRY(moe_sorting_fwd),
    AA_ENTRY(moe_sorting_mx_quant), AA_ENTRY(fused_dynamic_mx_quant_moe_sort_hip), AA_ENTRY(mxfp4_moe_sort_hip),
    AA_ENTRY(ck_moe_stage1), AA_ENTRY(ck_moe_stage1_fuse_quant), AA_ENTRY(moe_stage1_stream),
    AA_ENTRY(ck_moe_stage2), AA_ENTRY(moe_stage2_reduce), AA_ENTRY(moe_sum),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", AITER_AMD_TORCH) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
