// Compiled calls of the C ABI (include/modelopt_hip.h) for the Python layer.
//
// A call through ctypes converts every argument by its declared type at run time: 4.1 us for the fourteen
// arguments of mo_row_qdq with its launch, which is most of what a fake quantisation of a few tokens costs; 3.2 compiled,
// nearly all of it the launch.  The converters here are generated from the declarations of the header.  The
// functions' addresses come from the library that the Python layer has loaded: this file links none of it.
//
// Two quantizer calls are whole here, output tensor, scratch memory and stream included: x of 8 x 4096 under NVFP4
// 6.9 us from Python through ctypes (empty_like 1.2, the call 4.8), 4.3 so; the quantizer's forward 9.6 and 8.1.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <cstring>
#include <tuple>
#include <type_traits>
#include <utility>
#include <vector>

#include "modelopt_hip.h"

namespace {

// Every entry point whose pointers are device addresses (or None): host arrays and results by
// reference stay with ctypes.
#define MO_FUNCTIONS(X)                                                                                       \
    X(mo_absmax) X(mo_absmax_hinted) X(mo_absmax_tensor) X(mo_dynamic_qdq) X(mo_nvfp4_quantize_dynamic)       \
    X(mo_absmax_pair) X(mo_awq_pick_scale) X(mo_smooth_scales) X(mo_absmax_cols_staged)                       \
    X(mo_absmax_cols_noalloc) X(mo_fp8_qdq) X(mo_int_qdq) X(mo_ste_mask) X(mo_wgrad_masked) X(mo_row_qdq)     \
    X(mo_input_grad_splits) X(mo_input_grad_tile) X(mo_input_grad)                                            \
    X(mo_nvfp4_qdq) X(mo_qdq_sq_err) X(mo_mxfp4_quantize) X(mo_mxfp4_dequantize) X(mo_block_fp_qdq)           \
    X(mo_convert_to_format) X(mo_nvfp4_quantize) X(mo_nvfp4_quantize_fused) X(mo_fused_amax_qdq)              \
    X(mo_nvfp4_dequantize) X(mo_real_quantize) X(mo_real_dequantize) X(mo_int4_block_quantize)                \
    X(mo_int4_block_dequantize) X(mo_cast_fp4) X(mo_fp8_qdq_blocks2d) X(mo_int_qdq_blocks2d)                  \
    X(mo_absmax_blocks2d) X(mo_real_quantize_blocks2d) X(mo_real_dequantize_blocks2d) X(mo_int4_pack_rows)    \
    X(mo_int4_pack_rows_via) X(mo_nf4_quantize) X(mo_nf4_scales_quantize) X(mo_nf4_dequantize_double)         \
    X(mo_nf4_dequantize) X(mo_mul_cols) X(mo_scale_block_int_qdq) X(mo_awq_scale_grid)                        \
    X(mo_awq_scale_activations) X(mo_awq_search_losses) X(mo_awq_search_losses_biased) X(mo_awq_best_clip)    \
    X(mo_abs_colsum) X(mo_abs_colsum_staged) X(mo_weight_scale_colsum) X(mo_sq_diff_sum)

// Of those the ones that the calls below make themselves
#define MO_INSIDE(X) X(mo_value_ranges) X(mo_amax_fold)

enum Slot {
#define X(f) k_##f,
    MO_FUNCTIONS(X) kCalls, kBeforeInside = kCalls - 1, MO_INSIDE(X) kSlots
#undef X
};
const char* const kNames[] = {
#define X(f) #f,
    MO_FUNCTIONS(X) MO_INSIDE(X)
#undef X
};
void* g_address[kSlots];

template <typename T>
bool convert(PyObject* o, T& out) {
    if constexpr (std::is_pointer_v<T>) {
        out = nullptr;
        if (o == Py_None) return true;
        out = (T)PyLong_AsVoidPtr(o);
    } else if constexpr (std::is_floating_point_v<T>) {
        out = (T)PyFloat_AsDouble(o);
    } else if constexpr (sizeof(T) == 8) {
        out = (T)PyLong_AsLongLong(o);
    } else {
        const long long v = PyLong_AsLongLong(o);
        out = (T)v;
        if ((long long)out != v && !PyErr_Occurred())
            PyErr_SetString(PyExc_OverflowError, "argument does not fit its type");
    }
    return !PyErr_Occurred();
}

template <int SLOT, typename F>
struct Call;
template <int SLOT, typename... A>
struct Call<SLOT, int (*)(A...)> {
    using Args = std::tuple<A...>;
    template <size_t... I>
    static PyObject* run(PyObject* const* args, Py_ssize_t n, std::index_sequence<I...>) {
        if (n != (Py_ssize_t)sizeof...(A) || !g_address[SLOT]) {
            PyErr_Format(PyExc_TypeError, "%s: %zd arguments given, %zd taken", kNames[SLOT], n, (Py_ssize_t)sizeof...(A));
            return nullptr;
        }
        Args a{};
        if (!(convert(args[I], std::get<I>(a)) && ...)) return nullptr;
        int rc;
        Py_BEGIN_ALLOW_THREADS
        rc = ((int (*)(A...))g_address[SLOT])(std::get<I>(a)...);
        Py_END_ALLOW_THREADS
        return PyLong_FromLong(rc);
    }
    static PyObject* fast(PyObject*, PyObject* const* args, Py_ssize_t n) {
        return run(args, n, std::index_sequence_for<A...>{});
    }
};

template <typename F>
F bound(Slot slot, F) {
    return (F)g_address[slot];
}
#define BOUND(f) bound(k_##f, &f)

// -------------------------------------------------------------------------- whole quantizer calls

int code_of(at::ScalarType t) {
    return t == at::kFloat ? MO_F32 : t == at::kHalf ? MO_F16 : t == at::kBFloat16 ? MO_BF16 : -1;
}

// A contiguous tensor in the memory of the current GPU, of a type that the kernels take
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_Check(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda() || !t.is_contiguous() || code_of(t.scalar_type()) < 0 ||
        t.get_device() != c10::hip::current_device())
        return nullptr;
    return &t;
}

struct Kind {
    int kind, p0, p1, p2;
};
bool kind_of(PyObject* const* a, Kind& k) {
    return convert(a[0], k.kind) && convert(a[1], k.p0) && convert(a[2], k.p1) && convert(a[3], k.p2);
}

PyObject* finish(int rc, const at::Tensor& y) {
    if (rc == MO_OK) return THPVariable_Wrap(y);
    return PyLong_FromLong(rc);   // the caller raises, with the name of the code
}

// row_qdq(x, pre_scale, kind, p0, p1, p2, amax): the tensor, a status other than MO_OK, or None where the arguments
// are for the general path to take or to refuse
PyObject* row_qdq(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Kind k;
    if (n != 7 || !g_address[k_mo_row_qdq]) Py_RETURN_NONE;
    const at::Tensor* xp = plain(a[0]);
    const at::Tensor* sp = a[1] == Py_None ? nullptr : plain(a[1]);
    const at::Tensor* ap = a[6] == Py_None ? nullptr : plain(a[6]);
    if (!xp || (a[1] != Py_None && !sp) || (a[6] != Py_None && !ap) || xp->dim() == 0 || xp->numel() == 0) Py_RETURN_NONE;
    if (!kind_of(a + 2, k)) return nullptr;
    const at::Tensor x = *xp;
    const int64_t cols = x.size(-1);
    if (sp && (sp->scalar_type() != x.scalar_type() || sp->numel() != cols)) Py_RETURN_NONE;
    const void* scale = sp ? sp->const_data_ptr() : nullptr;
    const void* amax = ap ? ap->const_data_ptr() : nullptr;
    const int amax_dtype = ap ? code_of(ap->scalar_type()) : MO_F32;
    at::Tensor y;
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        y = at::empty_like(x);
        rc = BOUND(mo_row_qdq)(x.const_data_ptr(), y.mutable_data_ptr(), x.numel() / cols, cols, code_of(x.scalar_type()),
                               scale, k.kind, k.p0, k.p1, k.p2, amax, amax_dtype,
                               c10::hip::getCurrentHIPStream().stream());
    }
    return finish(rc, y);
    END_HANDLE_TH_ERRORS
}

// dynamic_qdq(x, kind, p0, p1, p2, scratch bytes)
PyObject* dynamic_qdq(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    Kind k;
    int64_t bytes;
    if (n != 6 || !g_address[k_mo_dynamic_qdq]) Py_RETURN_NONE;
    const at::Tensor* xp = plain(a[0]);
    if (!xp || xp->numel() == 0 || ((uintptr_t)xp->const_data_ptr() & 15u)) Py_RETURN_NONE;
    if (!kind_of(a + 1, k) || !convert(a[5], bytes)) return nullptr;
    const at::Tensor x = *xp;
    const int64_t cols = x.dim() ? x.size(-1) : 1;
    at::Tensor y;
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        y = at::empty_like(x);
        const at::Tensor parts = at::empty({bytes}, x.options().dtype(at::kByte));
        rc = BOUND(mo_dynamic_qdq)(x.const_data_ptr(), y.mutable_data_ptr(), x.numel() / cols, cols,
                                   code_of(x.scalar_type()), k.kind, k.p0, k.p1, k.p2, parts.mutable_data_ptr(),
                                   c10::hip::getCurrentHIPStream().stream());
    }
    return finish(rc, y);
    END_HANDLE_TH_ERRORS
}

// value_ranges(tensors, most tensors, elements of a chunk, most chunks): (the kernel's output, [chunks of each tensor]),
// or None where the list is not covered
PyObject* value_ranges(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int64_t most, chunk, most_chunks;
    if (n != 4 || !PyList_Check(a[0]) || !g_address[k_mo_value_ranges]) Py_RETURN_NONE;
    if (!convert(a[1], most) || !convert(a[2], chunk) || !convert(a[3], most_chunks)) return nullptr;
    const int64_t count = PyList_GET_SIZE(a[0]);
    if (count == 0 || count > most || count > 64) Py_RETURN_NONE;
    const void* xs[64];
    int64_t counts[64], chunks[64], total = 0;
    int dtypes[64];
    std::vector<at::Tensor> held;
    for (int64_t i = 0; i < count; ++i) {
        const at::Tensor* t = plain(PyList_GET_ITEM(a[0], i));
        if (!t) Py_RETURN_NONE;
        held.push_back(*t);
        xs[i] = t->const_data_ptr();
        counts[i] = t->numel();
        dtypes[i] = code_of(t->scalar_type());
        chunks[i] = std::max<int64_t>(1, (counts[i] + chunk - 1) / chunk);
        total += chunks[i];
    }
    if (total > most_chunks) Py_RETURN_NONE;
    at::Tensor out;
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        out = at::empty({3 * total}, held[0].options().dtype(at::kFloat));
        rc = BOUND(mo_value_ranges)(xs, counts, dtypes, (int)count, out.mutable_data_ptr<float>(), total,
                                    c10::hip::getCurrentHIPStream().stream());
    }
    if (rc != MO_OK) return PyLong_FromLong(rc);
    pybind11::list each;
    for (int64_t i = 0; i < count; ++i) each.append(chunks[i]);
    return pybind11::make_tuple(pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(out)), each).release().ptr();
    END_HANDLE_TH_ERRORS
}

// amax_fold([accumulator], [[parts]], [dtype code]): the folded maximum of each as a tensor of no dims in its type (mo_amax_fold),
// a status, or None where an accumulator is not one fp32 element on the current GPU
PyObject* amax_fold(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3 || !PyList_Check(a[0]) || !PyList_Check(a[1]) || !PyList_Check(a[2]) || !g_address[k_mo_amax_fold]) Py_RETURN_NONE;
    const Py_ssize_t count = PyList_GET_SIZE(a[0]);
    if (count == 0 || PyList_GET_SIZE(a[1]) != count || PyList_GET_SIZE(a[2]) != count) Py_RETURN_NONE;
    std::vector<at::Tensor> held, outs;
    std::vector<float*> accs;
    std::vector<void*> out_ptrs;
    std::vector<int> dtypes, first{0};
    std::vector<const uint32_t*> parts;
    std::vector<int64_t> words;
    static const at::ScalarType kTypes[3] = {at::kFloat, at::kHalf, at::kBFloat16};
    for (Py_ssize_t i = 0; i < count; ++i) {
        const at::Tensor* acc = plain(PyList_GET_ITEM(a[0], i));
        PyObject* runs = PyList_GET_ITEM(a[1], i);
        int code;
        if (!convert(PyList_GET_ITEM(a[2], i), code)) return nullptr;
        if (!acc || acc->numel() != 1 || acc->scalar_type() != at::kFloat || !PyList_Check(runs) || code < MO_F32 || code > MO_BF16)
            Py_RETURN_NONE;
        held.push_back(*acc);
        for (Py_ssize_t j = 0; j < PyList_GET_SIZE(runs); ++j) {
            PyObject* r = PyList_GET_ITEM(runs, j);
            if (!THPVariable_Check(r)) Py_RETURN_NONE;
            const at::Tensor& t = THPVariable_Unpack(r);
            if (t.scalar_type() != at::kInt || !t.is_contiguous() || !t.is_cuda() || t.device() != acc->device()) Py_RETURN_NONE;
            held.push_back(t);
            parts.push_back((const uint32_t*)t.const_data_ptr());
            words.push_back(t.numel());
        }
        first.push_back((int)parts.size());
        accs.push_back((float*)acc->mutable_data_ptr());
        dtypes.push_back(code);
    }
    int rc;
    {
        pybind11::gil_scoped_release no_gil;
        for (Py_ssize_t i = 0; i < count; ++i) {
            outs.push_back(at::empty({}, held[0].options().dtype(kTypes[dtypes[i]])));
            out_ptrs.push_back(outs.back().mutable_data_ptr());
        }
        rc = BOUND(mo_amax_fold)(accs.data(), out_ptrs.data(), dtypes.data(), first.data(), parts.data(), words.data(),
                                 (int)count, c10::hip::getCurrentHIPStream().stream());
    }
    if (rc != MO_OK) return PyLong_FromLong(rc);
    pybind11::list made;
    for (const at::Tensor& t : outs) made.append(pybind11::reinterpret_steal<pybind11::object>(THPVariable_Wrap(t)));
    return made.release().ptr();
    END_HANDLE_TH_ERRORS
}

// bind({name: address}): where the calls go; a name left out has no compiled call.  Returns the names of those that have one.
PyObject* bind(PyObject*, PyObject* table) {
    PyObject* names = PyList_New(0);
    if (!names) return nullptr;
    for (int i = 0; i < kSlots; ++i) {
        PyObject* v = PyDict_GetItemString(table, kNames[i]);
        if (!v) continue;
        void* p = PyLong_AsVoidPtr(v);
        if (!PyErr_Occurred() && i >= kCalls) {
            g_address[i] = p;
            continue;
        }
        PyObject* name = PyErr_Occurred() ? nullptr : PyUnicode_FromString(kNames[i]);
        if (!name || PyList_Append(names, name)) {
            Py_XDECREF(name);
            Py_DECREF(names);
            return nullptr;
        }
        Py_DECREF(name);
        g_address[i] = p;
    }
    return names;
}

PyMethodDef kMethods[] = {
#define X(f) {#f, (PyCFunction)(void (*)(void))Call<k_##f, decltype(&f)>::fast, METH_FASTCALL, nullptr},
    MO_FUNCTIONS(X)
#undef X
    {"row_qdq", (PyCFunction)(void (*)(void))row_qdq, METH_FASTCALL, nullptr},
    {"dynamic_qdq", (PyCFunction)(void (*)(void))dynamic_qdq, METH_FASTCALL, nullptr},
    {"value_ranges", (PyCFunction)(void (*)(void))value_ranges, METH_FASTCALL, nullptr},
    {"amax_fold", (PyCFunction)(void (*)(void))amax_fold, METH_FASTCALL, nullptr},
    {"bind", bind, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_launch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__launch(void) { return PyModule_Create(&kModule); }
