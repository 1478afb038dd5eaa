// The Python side of a call: the library's functions taking torch tensors as their pointers, and the checks that stand before most of them.
// Built into the module research_amd._host (plain C++; it finds the functions in the library that _lib.py has loaded).
//
// A call of a small shape is as long as its host side.  us a pass with ctypes and each tensor's pointer, type, shape and strides asked for from
// Python -> this: mLSTM, 34 rows and two tokens behind them 49.5 -> 30.8; SSD, 235 rows and a token 32.7 -> 21.2; delta rule, 37 rows and three
// tokens 66 -> 43.5; attention with score terms, a token 10.3 -> 5.8; experts of 235 rows 54 -> 42.
#include <Python.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <tuple>
#include <utility>

#include "../../include/paged_attn.h"

// The functions that ops.py calls
#define PA_CALLS(X)                                                                                                                     \
    X(pa_kv_scatter) X(pa_kv_gather) X(pa_decode) X(pa_decode_split) X(pa_decode_reduce) X(pa_decode_static) X(pa_prefill_paged)         \
    X(pa_prefill_paged_ws) X(pa_prefill_paged_rowwise) X(pa_attend_masked) X(pa_quantize_kv_e4m3) X(pa_kv_append_e4m3)                   \
    X(pa_dequantize_blocks_e4m3) X(pa_rope_kv_append) X(pa_rope_kv_append_e4m3) X(pa_residual_norm) X(pa_bias_act) X(pa_rms_gate)        \
    X(pa_softcap) X(pa_glu) X(pa_head_gate) X(pa_qkv_conv_append) X(pa_lightning_recurrent) X(pa_lightning_chunked) X(pa_short_conv)     \
    X(pa_gated_linear) X(pa_narrow_linear) X(pa_moe_workspace_bytes) X(pa_moe_choose) X(pa_moe_product) X(pa_delta) X(pa_hyper_norm)     \
    X(pa_latent_append) X(pa_latent_gather) X(pa_scored_attention) X(pa_talking_attention) X(pa_channel_linear)

namespace {

enum Function {
#define X(name) k_##name,
    PA_CALLS(X)
#undef X
    kFunctions
};
const char *const kNames[] = {
#define X(name) #name,
    PA_CALLS(X)
#undef X
};
void *bound[kFunctions];  // (set once by bind, before any call)

const at::Tensor *tensor_of(PyObject *x) { return THPVariable_Check(x) ? &THPVariable_Unpack(x) : nullptr; }

// One argument from Python; false with an exception set.  Integers wrap to the parameter's size, as ctypes has it.
template <typename T> bool take(PyObject *x, T *&to) {
    if (x == Py_None) {
        to = nullptr;
    } else if (const at::Tensor *t = tensor_of(x)) {
        to = static_cast<T *>(t->data_ptr());
    } else {
        if (!PyLong_Check(x)) {
            PyErr_Format(PyExc_TypeError, "expected a tensor, None or an address, got %s", Py_TYPE(x)->tp_name);
            return false;
        }
        const unsigned long long v = PyLong_AsUnsignedLongLongMask(x);
        if (v == ~0ull && PyErr_Occurred()) return false;
        to = reinterpret_cast<T *>(static_cast<uintptr_t>(v));
    }
    return true;
}
template <typename T> std::enable_if_t<std::is_integral_v<T>, bool> take(PyObject *x, T &to) {
    const unsigned long long v = PyLong_AsUnsignedLongLongMask(x);
    if (v == ~0ull && PyErr_Occurred()) return false;
    to = static_cast<T>(v);
    return true;
}
bool take(PyObject *x, float &to) {
    const double v = PyFloat_AsDouble(x);
    if (v == -1.0 && PyErr_Occurred()) return false;
    to = static_cast<float>(v);
    return true;
}

struct Unlocked {  // other Python threads run meanwhile (also while an exception leaves the library)
    PyThreadState *state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};

template <int I, typename F> struct Call;
template <int I, typename R, typename... A> struct Call<I, R (*)(A...)> {
    template <size_t... N> static bool take_all(PyObject *const *args, std::tuple<A...> &to, std::index_sequence<N...>) {
        return (take(args[N], std::get<N>(to)) && ...);
    }
    static PyObject *run(PyObject *, PyObject *const *args, Py_ssize_t n) {
        HANDLE_TH_ERRORS
        if (n != (Py_ssize_t)sizeof...(A)) {
            PyErr_Format(PyExc_TypeError, "%s takes %zd arguments, got %zd", kNames[I], (Py_ssize_t)sizeof...(A), n);
            return nullptr;
        }
        if (!bound[I]) {
            PyErr_Format(PyExc_RuntimeError, "%s: the library has not been loaded", kNames[I]);
            return nullptr;
        }
        std::tuple<A...> values;
        if (!take_all(args, values, std::index_sequence_for<A...>{})) return nullptr;
        const R result = [&] {
            Unlocked unlocked;
            return std::apply(reinterpret_cast<R (*)(A...)>(bound[I]), values);
        }();
        if constexpr (std::is_signed_v<R>) return PyLong_FromLongLong((long long)result);
        else return PyLong_FromUnsignedLongLong((unsigned long long)result);
        END_HANDLE_TH_ERRORS
    }
};

// bind(handle): the functions of the library behind a dlopen handle
PyObject *bind(PyObject *, PyObject *arg) {
    void *handle = PyLong_AsVoidPtr(arg);
    if (!handle) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "no library");
        return nullptr;
    }
    void *found[kFunctions];
    for (int i = 0; i < kFunctions; ++i) {
        found[i] = dlsym(handle, kNames[i]);
        if (!found[i]) {
            PyErr_Format(PyExc_AttributeError, "the library has no %s", kNames[i]);
            return nullptr;
        }
    }
    for (int i = 0; i < kFunctions; ++i) bound[i] = found[i];
    Py_RETURN_NONE;
}

bool a_tensor(PyObject *x, const at::Tensor *&t) {
    t = tensor_of(x);
    if (!t) PyErr_Format(PyExc_TypeError, "expected a tensor, got %s", Py_TYPE(x)->tp_name);
    return t != nullptr;
}

// dense(*tensors or None): all are contiguous
PyObject *dense(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    for (Py_ssize_t i = 0; i < n; ++i) {
        const at::Tensor *t;
        if (args[i] == Py_None) continue;
        if (!a_tensor(args[i], t)) return nullptr;
        if (!t->is_contiguous()) {
            PyErr_SetString(PyExc_ValueError, "expected contiguous tensors");
            return nullptr;
        }
    }
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// typed(dtype, *tensors or None): all have that type
PyObject *typed(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 1 || !THPDtype_Check(args[0])) {
        PyErr_SetString(PyExc_TypeError, "expected a dtype");
        return nullptr;
    }
    const at::ScalarType want = reinterpret_cast<THPDtype *>(args[0])->scalar_type;
    for (Py_ssize_t i = 1; i < n; ++i) {
        const at::Tensor *t;
        if (args[i] == Py_None) continue;
        if (!a_tensor(args[i], t)) return nullptr;
        if (t->scalar_type() != want) {
            PyObject *got = PyObject_GetAttrString(args[i], "dtype");
            if (got) PyErr_Format(PyExc_ValueError, "expected %S, got %S", args[0], got);
            Py_XDECREF(got);
            return nullptr;
        }
    }
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// shaped(tensor, *sizes): whether the tensor has these sizes (None: any)
PyObject *shaped(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor *t;
    if (n < 1) {
        PyErr_SetString(PyExc_TypeError, "expected a tensor");
        return nullptr;
    }
    if (!a_tensor(args[0], t)) return nullptr;
    bool same = t->dim() == n - 1;
    for (Py_ssize_t i = 1; same && i < n; ++i) {
        if (args[i] == Py_None) continue;
        const long long v = PyLong_AsLongLong(args[i]);
        if (v == -1 && PyErr_Occurred()) return nullptr;
        same = t->size(i - 1) == v;
    }
    return PyBool_FromLong(same);
    END_HANDLE_TH_ERRORS
}

// row_stride(tensor): elements between the rows of a 2-D tensor whose rows are contiguous (a column slice of a wider one)
PyObject *row_stride(PyObject *, PyObject *arg) {
    HANDLE_TH_ERRORS
    const at::Tensor *t;
    if (!a_tensor(arg, t)) return nullptr;
    if (t->dim() == 2) {
        const int64_t rows = t->size(0), cols = t->size(1), row = t->stride(0);
        if (cols <= 1 || t->stride(1) == 1) return PyLong_FromLongLong(rows > 1 ? row : row > cols ? row : cols);
    }
    PyErr_SetString(PyExc_ValueError, "expected a 2-D tensor with contiguous rows");
    return nullptr;
    END_HANDLE_TH_ERRORS
}

// nbytes(tensor or None): bytes of its elements
PyObject *nbytes(PyObject *, PyObject *arg) {
    HANDLE_TH_ERRORS
    const at::Tensor *t;
    if (arg == Py_None) return PyLong_FromLong(0);
    if (!a_tensor(arg, t)) return nullptr;
    return PyLong_FromLongLong(t->numel() * (int64_t)t->element_size());
    END_HANDLE_TH_ERRORS
}

// stream(tensor): the number of the current stream of its device
PyObject *raw_stream;  // torch._C._cuda_getCurrentRawStream: without the object that torch.cuda.current_stream makes around it
PyObject *stream(PyObject *, PyObject *arg) {
    HANDLE_TH_ERRORS
    const at::Tensor *t;
    if (!a_tensor(arg, t)) return nullptr;
    if (!t->is_cuda()) {
        PyObject *on = PyObject_GetAttrString(arg, "device");
        if (on) PyErr_Format(PyExc_RuntimeError, "libpaged_attn computes only on a HIP device; got a tensor on %S", on);
        Py_XDECREF(on);
        return nullptr;
    }
    PyObject *device = PyLong_FromLong(t->get_device());
    if (!device) return nullptr;
    PyObject *number = PyObject_CallFunctionObjArgs(raw_stream, device, nullptr);
    Py_DECREF(device);
    return number;
    END_HANDLE_TH_ERRORS
}

#define FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f))
PyMethodDef methods[] = {
#define X(name) {#name, FAST((&Call<k_##name, decltype(&name)>::run)), METH_FASTCALL, nullptr},
    PA_CALLS(X)
#undef X
    {"bind", bind, METH_O, nullptr},
    {"dense", FAST(dense), METH_FASTCALL, nullptr},
    {"typed", FAST(typed), METH_FASTCALL, nullptr},
    {"shaped", FAST(shaped), METH_FASTCALL, nullptr},
    {"row_stride", row_stride, METH_O, nullptr},
    {"nbytes", nbytes, METH_O, nullptr},
    {"stream", stream, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
    // What is read here of a tensor lies where the torch that this was built against puts it.
    PyObject *v = PyImport_ImportModule("torch.version"), *is = v ? PyObject_GetAttrString(v, "__version__") : nullptr;
    Py_XDECREF(v);
    if (!is) return nullptr;
    const bool same = PyUnicode_Check(is) && PyUnicode_CompareWithASCIIString(is, PA_TORCH_VERSION) == 0;
    if (!same) PyErr_Format(PyExc_ImportError, "built for torch " PA_TORCH_VERSION ", this is torch %S", is);
    Py_DECREF(is);
    if (!same) return nullptr;
    PyObject *c = PyImport_ImportModule("torch._C");
    if (!c) return nullptr;
    raw_stream = PyObject_GetAttrString(c, "_cuda_getCurrentRawStream");
    Py_DECREF(c);
    return raw_stream ? PyModule_Create(&module) : nullptr;
}
