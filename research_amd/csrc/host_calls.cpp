// The Python side of a call: the library's functions taking torch tensors as their pointers, and the checks that stand before most of them.
// Built into the module research_amd._host (plain C++; it finds the functions in the library that _lib.py has loaded).
//
// A call of a small shape is as long as its host side.  us a pass with ctypes and each tensor's pointer, type, shape and strides asked for from
// Python -> functions and checks in C++: mLSTM, 34 rows and two tokens behind them 49.5 -> 30.8; SSD, 235 rows and a token 32.7 -> 21.2; delta rule, 37 rows and three
// tokens 66 -> 43.5; attention with score terms, a token 10.3 -> 5.8; experts of 235 rows 54 -> 42.
#include <Python.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ops/empty.h>

#include <initializer_list>
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

// ---- Whole wrappers of ops.py for the calls that small shapes repeat most ----
// Each makes the wrapper's checks, allocates its results and calls the library.  Where anything does not fit (also another type of number than
// a wrapper's callers pass) it does nothing and answers None: the wrapper then goes its own way, and says what it is.  Else the answer is the
// results, or the library's status where that is not zero (or there are no new results).
// us a call, checks and results from Python -> this: choice of experts 14.3 -> 9.1, product of experts 6.4 -> 4.7, narrow product 4.9 -> 3.8, a token of a
// gated recurrence 5.6 -> 4.0; the expert layer of 33 rows of 1024 and 16 experts 50 -> 38, SSD of 3 prompts of 127 .. 246 rows and a token 28 -> 21.
struct Taken {  // arguments one after the other; ok: all were what was asked for
    PyObject *const *at;
    bool ok = true;
    const at::Tensor *maybe() { return *at == Py_None ? (++at, nullptr) : tensor(); }
    const at::Tensor *tensor() {
        const at::Tensor *t = tensor_of(*at++);
        ok = ok && t;
        return t;
    }
    int64_t integer() {
        int over = 0;
        const long long v = PyLong_Check(*at) ? PyLong_AsLongLongAndOverflow(*at, &over) : (over = 1);
        ++at;
        ok = ok && !over;
        return v;
    }
    float number() {
        const bool is = PyFloat_Check(*at);
        ok = ok && is;
        return (float)(is ? PyFloat_AS_DOUBLE(*at++) : (++at, 0.0));
    }
};

void *pointer(const at::Tensor *t) { return t ? t->data_ptr() : nullptr; }
template <typename T> T *pointer_of(const at::Tensor *t) { return static_cast<T *>(pointer(t)); }
bool all_dense(std::initializer_list<const at::Tensor *> ts) {
    for (const at::Tensor *t : ts)
        if (t && !t->is_contiguous()) return false;
    return true;
}
bool all_typed(at::ScalarType want, std::initializer_list<const at::Tensor *> ts) {
    for (const at::Tensor *t : ts)
        if (t && t->scalar_type() != want) return false;
    return true;
}
// rows x cols (either -1: any) with contiguous rows, and the elements between them (as row_stride)
bool in_rows(const at::Tensor *t, int64_t rows, int64_t cols, int64_t &stride) {
    if (t->dim() != 2 || (rows >= 0 && t->size(0) != rows) || (cols >= 0 && t->size(1) != cols) || (t->size(1) > 1 && t->stride(1) != 1)) return false;
    const int64_t row = t->stride(0), n = t->size(1);
    stride = t->size(0) > 1 ? row : row > n ? row : n;
    return true;
}
bool sized(const at::Tensor *t, int64_t b, int64_t c, int64_t d = -1) {  // [any, b, c] or [any, b, c, d]
    return t->dim() == (d < 0 ? 3 : 4) && t->size(1) == b && t->size(2) == c && (d < 0 || t->size(3) == d);
}
int type_code(const at::Tensor *t) {
    const at::ScalarType s = t->scalar_type();
    return s == at::kFloat ? PA_F32 : s == at::kBFloat16 ? PA_BF16 : s == at::kHalf ? PA_F16 : -1;
}
int64_t pad16(int64_t n) { return (n + 15) / 16 * 16; }
bool fits_int(std::initializer_list<int64_t> ns) {
    for (int64_t n : ns)
        if (n < 0 || n > 0x7fffffff) return false;
    return true;
}
// The current stream of the tensor's device; false, without an exception, where there is none.
bool stream_of(const at::Tensor *t, void *&to) {
    if (!t->is_cuda()) return false;
    PyObject *device = PyLong_FromLong(t->get_device()), *number = device ? PyObject_CallFunctionObjArgs(raw_stream, device, nullptr) : nullptr;
    Py_XDECREF(device);
    to = number ? PyLong_AsVoidPtr(number) : nullptr;
    Py_XDECREF(number);
    if (!PyErr_Occurred()) return true;
    PyErr_Clear();
    return false;
}
template <typename F, typename... A> int unlocked(Function which, A... args) {
    Unlocked u;
    return reinterpret_cast<F>(bound[which])(args...);
}
#define PA_UNLOCKED(name, ...) unlocked<decltype(&name)>(k_##name, __VA_ARGS__)

struct Runs {  // ctx_lens, state_slots, q_lens, q_starts, max_q_len: the new rows of a recurrence
    const at::Tensor *ctx, *slots, *lens, *starts;
    int64_t most;
    explicit Runs(Taken &a) : ctx(a.tensor()), slots(a.maybe()), lens(a.maybe()), starts(a.maybe()), most(a.integer()) {}
    bool fit() const { return all_dense({ctx, slots, lens, starts}) && all_typed(at::kInt, {ctx, slots, lens, starts}) && fits_int({ctx->numel(), most}); }
};
size_t bytes_of(const at::Tensor *t) { return t ? (size_t)t->numel() * t->element_size() : 0; }

// (kind, q, k, v, heads_per_group, gate a, gate b, three constants, cap, q_scale, den_eps, runs, state, its floats per head, heads, dim, vdim, out, workspace)
PyObject *whole_gated_linear(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 25 || !bound[k_pa_gated_linear]) Py_RETURN_NONE;
    Taken a{args};
    const int64_t kind = a.integer();
    const at::Tensor *q = a.tensor(), *k = a.tensor(), *v = a.tensor();
    const int64_t per = a.integer();
    const at::Tensor *ga = a.tensor(), *gb = a.maybe(), *ca = a.maybe(), *cb = a.maybe(), *cc = a.maybe();
    const float cap = a.number(), q_scale = a.number(), eps = a.number();
    const Runs r(a);
    const at::Tensor *state = a.tensor();
    const int64_t floats = a.integer(), heads = a.integer(), dim = a.integer(), vdim = a.integer();
    const at::Tensor *out = a.tensor(), *ws = a.maybe();
    void *stream;
    int64_t sq, sk, sv, so, sa, sb;
    if (!a.ok || !r.fit() || !fits_int({kind, per, heads, dim, vdim}) || per == 0 || !all_dense({state, out, ca, cb, cc}) || !all_typed(at::kFloat, {state, ca, cb, cc}) ||
        !all_typed(v->scalar_type(), {q, k, ga, gb, out}) || type_code(v) < 0 || !in_rows(v, -1, heads * vdim, sv))
        Py_RETURN_NONE;
    const int64_t rows = v->size(0), wide = heads / per * dim;
    if (!in_rows(q, rows, wide, sq) || !in_rows(k, rows, wide, sk) || !in_rows(out, rows, heads * vdim, so) || !in_rows(ga, rows, heads, sa)) Py_RETURN_NONE;
    if (gb && (!in_rows(gb, rows, heads, sb) || sb != sa)) Py_RETURN_NONE;
    for (const at::Tensor *c : {ca, cb, cc})
        if (c && c->numel() != heads) Py_RETURN_NONE;
    if (!sized(state, heads, floats) || !stream_of(v, stream)) Py_RETURN_NONE;
    return PyLong_FromLong(PA_UNLOCKED(pa_gated_linear, (int)kind, pointer(q), sq, pointer(k), sk, pointer(v), sv, (int)per, pointer(ga), pointer(gb), sa,
                                       pointer_of<float>(ca), pointer_of<float>(cb), pointer_of<float>(cc), cap, q_scale, eps, rows, pointer_of<float>(state),
                                       state->size(0), pointer_of<int32_t>(r.ctx), pointer_of<int32_t>(r.lens), pointer_of<int32_t>(r.starts),
                                       pointer_of<int32_t>(r.slots), (int)r.ctx->numel(), (int)r.most, pointer(out), (int)heads, (int)dim, (int)vdim, type_code(v),
                                       pointer(ws), bytes_of(ws), stream));
    END_HANDLE_TH_ERRORS
}

// (q, k, v, heads_per_group, decay logits, beta logits, decay bias, decay rate, q_scale, runs, state, heads, dim, vdim, out, workspace)
PyObject *whole_delta_rule(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 20 || !bound[k_pa_delta]) Py_RETURN_NONE;
    Taken a{args};
    const at::Tensor *q = a.tensor(), *k = a.tensor(), *v = a.tensor();
    const int64_t per = a.integer();
    const at::Tensor *decay = a.tensor(), *beta = a.tensor(), *bias = a.tensor(), *rate = a.tensor();
    const float q_scale = a.number();
    const Runs r(a);
    const at::Tensor *state = a.tensor();
    const int64_t heads = a.integer(), dim = a.integer(), vdim = a.integer();
    const at::Tensor *out = a.tensor(), *ws = a.maybe();
    void *stream;
    int64_t sq, sk, sv, so, sd, sb;
    if (!a.ok || !r.fit() || !fits_int({per, heads, dim, vdim}) || per == 0 || !all_dense({state, out, bias, rate}) || !all_typed(at::kFloat, {state, bias, rate}) ||
        !all_typed(v->scalar_type(), {q, k, decay, beta, out}) || type_code(v) < 0 || !in_rows(v, -1, heads * vdim, sv))
        Py_RETURN_NONE;
    const int64_t rows = v->size(0), wide = heads / per * dim;
    if (!in_rows(q, rows, wide, sq) || !in_rows(k, rows, wide, sk) || !in_rows(out, rows, heads * vdim, so) || !in_rows(decay, rows, heads, sd) ||
        !in_rows(beta, rows, heads, sb) || sd != sb || bias->numel() != heads || rate->numel() != heads || !sized(state, heads, pad16(dim), pad16(vdim)) ||
        !stream_of(v, stream))
        Py_RETURN_NONE;
    return PyLong_FromLong(PA_UNLOCKED(pa_delta, pointer(q), sq, pointer(k), sk, pointer(v), sv, (int)per, pointer(decay), pointer(beta), sd, pointer_of<float>(bias),
                                       pointer_of<float>(rate), q_scale, rows, pointer_of<float>(state), state->size(0), pointer_of<int32_t>(r.ctx),
                                       pointer_of<int32_t>(r.lens), pointer_of<int32_t>(r.starts), pointer_of<int32_t>(r.slots), (int)r.ctx->numel(), (int)r.most,
                                       pointer(out), (int)heads, (int)dim, (int)vdim, type_code(v), pointer(ws), bytes_of(ws), stream));
    END_HANDLE_TH_ERRORS
}

// (q, its activation, forget, f_bias, lower, v, runs, state, heads, dim, vdim, out, workspace)
PyObject *whole_channel_linear(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 17 || !bound[k_pa_channel_linear]) Py_RETURN_NONE;
    Taken a{args};
    const at::Tensor *q = a.tensor();
    const int64_t act = a.integer();
    const at::Tensor *forget = a.tensor(), *bias = a.maybe(), *lower = a.maybe(), *v = a.tensor();
    const Runs r(a);
    const at::Tensor *state = a.tensor();
    const int64_t heads = a.integer(), dim = a.integer(), vdim = a.integer();
    const at::Tensor *out = a.tensor(), *ws = a.maybe();
    void *stream;
    int64_t sq, sf, sv, so;
    if (!a.ok || !r.fit() || !fits_int({act, heads, dim, vdim}) || !all_dense({state, out, bias, lower}) || !all_typed(at::kFloat, {state, bias, lower}) ||
        !all_typed(v->scalar_type(), {q, forget, out}) || type_code(v) < 0 || !in_rows(v, -1, heads * vdim, sv))
        Py_RETURN_NONE;
    const int64_t rows = v->size(0), wide = heads * dim;
    if (!in_rows(q, rows, wide, sq) || !in_rows(forget, rows, wide, sf) || !in_rows(out, rows, heads * vdim, so) || (bias && bias->numel() != wide) ||
        (lower && lower->numel() != wide) || !sized(state, heads, pad16(dim), pad16(vdim)) || !stream_of(v, stream))
        Py_RETURN_NONE;
    return PyLong_FromLong(PA_UNLOCKED(pa_channel_linear, pointer(q), sq, (int)act, pointer(forget), sf, pointer_of<float>(bias), pointer_of<float>(lower), pointer(v), sv,
                                       rows, pointer_of<float>(state), state->size(0), pointer_of<int32_t>(r.ctx), pointer_of<int32_t>(r.lens),
                                       pointer_of<int32_t>(r.starts), pointer_of<int32_t>(r.slots), (int)r.ctx->numel(), (int)r.most, pointer(out), (int)heads,
                                       (int)dim, (int)vdim, type_code(v), pointer(ws), bytes_of(ws), stream));
    END_HANDLE_TH_ERRORS
}

// (u, runs, state, decay powers, heads, dim, vdim, out, workspace)
PyObject *whole_lightning(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 13 || !bound[k_pa_lightning_chunked] || !bound[k_pa_lightning_recurrent]) Py_RETURN_NONE;
    Taken a{args};
    const at::Tensor *u = a.tensor();
    const Runs r(a);
    const at::Tensor *state = a.tensor(), *powers = a.tensor();
    const int64_t heads = a.integer(), dim = a.integer(), vdim = a.integer();
    const at::Tensor *out = a.tensor(), *ws = a.maybe();
    void *stream;
    int64_t su, so;
    if (!a.ok || !r.fit() || !fits_int({heads, dim, vdim}) || !all_dense({state, powers, out}) || !all_typed(at::kFloat, {state, powers}) ||
        !all_typed(u->scalar_type(), {out}) || type_code(u) < 0 || !in_rows(u, -1, -1, su))
        Py_RETURN_NONE;
    const int64_t rows = u->size(0);
    if (powers->dim() != 2 || powers->size(0) != heads || powers->size(1) != 65 || !in_rows(out, rows, heads * vdim, so) ||
        !sized(state, heads, pad16(dim), pad16(vdim)) || !stream_of(u, stream))
        Py_RETURN_NONE;
    if (!r.lens || u->scalar_type() == at::kFloat)
        return PyLong_FromLong(PA_UNLOCKED(pa_lightning_recurrent, pointer(u), su, rows, pointer_of<float>(state), state->size(0), pointer_of<float>(powers),
                                           pointer_of<int32_t>(r.ctx), pointer_of<int32_t>(r.lens), pointer_of<int32_t>(r.starts), pointer_of<int32_t>(r.slots),
                                           (int)r.ctx->numel(), pointer(out), (int)heads, (int)dim, (int)vdim, type_code(u), stream));
    return PyLong_FromLong(PA_UNLOCKED(pa_lightning_chunked, pointer(u), su, rows, pointer_of<float>(state), state->size(0), pointer_of<float>(powers),
                                       pointer_of<int32_t>(r.ctx), pointer_of<int32_t>(r.lens), pointer_of<int32_t>(r.starts), pointer_of<int32_t>(r.slots),
                                       (int)r.ctx->numel(), (int)r.most, pointer(out), (int)heads, (int)dim, (int)vdim, type_code(u), pointer(ws), bytes_of(ws),
                                       stream));
    END_HANDLE_TH_ERRORS
}

// (x, w): the product
PyObject *whole_narrow_linear(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 2 || !bound[k_pa_narrow_linear]) Py_RETURN_NONE;
    Taken a{args};
    const at::Tensor *x = a.tensor(), *w = a.tensor();
    void *stream;
    int64_t sx;
    if (!a.ok || w->dim() != 2 || !all_dense({w}) || !all_typed(x->scalar_type(), {w}) || type_code(x) < 0 || !in_rows(x, -1, w->size(1), sx) ||
        !fits_int({w->size(0), w->size(1)}) || !stream_of(x, stream))
        Py_RETURN_NONE;
    at::Tensor out = at::empty({x->size(0), w->size(0)}, x->options().dtype(at::kFloat));
    if (const int status = PA_UNLOCKED(pa_narrow_linear, pointer(x), sx, pointer(w), pointer_of<float>(&out), x->size(0), (int)w->size(0), (int)w->size(1), type_code(x), stream))
        return PyLong_FromLong(status);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// (logits, correction, experts, identity, top, groups, keep, shared, columns of the shared expert, scores, group_top, renormalize): ids, weights, counts, lists
PyObject *whole_moe_choose(PyObject *, PyObject *const *args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 12 || !bound[k_pa_moe_choose] || !bound[k_pa_moe_workspace_bytes]) Py_RETURN_NONE;
    Taken a{args};
    const at::Tensor *logits = a.tensor(), *correction = a.maybe();
    const int64_t experts = a.integer(), identity = a.integer(), top = a.integer(), groups = a.integer(), keep = a.integer(), shared = a.integer(), gate = a.integer(),
                  scores = a.integer(), group_top = a.integer(), renormalize = a.integer(), all = experts + identity;
    void *stream;
    if (!a.ok || !fits_int({experts, identity, all, top, groups, keep, shared, scores, group_top}) || logits->dim() != 2 || !all_dense({logits, correction}) ||
        !all_typed(at::kFloat, {logits, correction}) || logits->size(1) != all + gate || (correction && correction->numel() != all) || !stream_of(logits, stream))
        Py_RETURN_NONE;
    const int64_t rows = logits->size(0);
    const auto ints = logits->options().dtype(at::kInt);
    at::Tensor ids = at::empty({rows, top}, ints), weights = at::empty({rows, top + (identity ? 2 : 1)}, logits->options()), counts = at::empty({all}, ints),
               lists = at::empty({all, rows}, ints);
    const int64_t need = (int64_t) reinterpret_cast<decltype(&pa_moe_workspace_bytes)>(bound[k_pa_moe_workspace_bytes])(rows, (int)all, (int)top);
    const at::Tensor ws = at::empty({need}, logits->options().dtype(at::kByte));
    if (const int status = PA_UNLOCKED(pa_moe_choose, pointer_of<float>(logits), logits->size(1), rows, (int)experts, (int)identity, (int)top, (int)groups, (int)keep, (int)shared,
                                       (int)scores, (int)group_top, renormalize != 0 ? 1 : 0, pointer_of<float>(correction), pointer_of<int32_t>(&ids),
                                       pointer_of<float>(&weights), pointer_of<int32_t>(&counts), pointer_of<int32_t>(&lists), pointer(&ws), (size_t)need, stream))
        return PyLong_FromLong(status);
    if (identity) {
        counts = counts.narrow(0, 0, experts);
        lists = lists.narrow(0, 0, experts);
    }
    PyObject *to = PyTuple_New(4);
    if (!to) return nullptr;
    at::Tensor *const results[] = {&ids, &weights, &counts, &lists};
    for (int i = 0; i < 4; ++i) {
        PyObject *t = THPVariable_Wrap(std::move(*results[i]));
        if (!t) {
            Py_DECREF(to);
            return nullptr;
        }
        PyTuple_SET_ITEM(to, i, t);
    }
    return to;
    END_HANDLE_TH_ERRORS
}

// (x, ids, weights, counts, lists, w, n, k, glu): the items' products
PyObject *whole_moe_product(PyObject *, PyObject *const *args, Py_ssize_t count) {
    HANDLE_TH_ERRORS
    if (count != 9 || !bound[k_pa_moe_product]) Py_RETURN_NONE;
    Taken a{args};
    const at::Tensor *x = a.tensor(), *ids = a.tensor(), *weights = a.tensor(), *counts = a.tensor(), *lists = a.tensor(), *w = a.tensor();
    const int64_t n = a.integer(), k = a.integer(), glu = a.integer();
    void *stream;
    int64_t sx;
    if (!a.ok || ids->dim() != 2 || w->dim() != 3 || !all_dense({w, ids, weights, counts, lists}) || !all_typed(x->scalar_type(), {w}) || type_code(x) < 0 ||
        !in_rows(x, -1, k, sx) || !fits_int({n, k, w->size(0), w->size(2), ids->size(1)}))
        Py_RETURN_NONE;
    const int64_t rows = ids->size(0), top = ids->size(1), mine = x->size(0);
    if ((mine != rows && mine != rows * top) || w->size(0) != counts->numel() || w->size(1) < n * (glu ? 2 : 1) || w->size(2) < k || !stream_of(x, stream)) Py_RETURN_NONE;
    at::Tensor out = at::empty({rows * top, n}, x->options());
    if (const int status = PA_UNLOCKED(pa_moe_product, pointer(x), sx, mine ? (int)(rows * top / mine) : 1, pointer(w), w->size(1), (int)w->size(2), (int)k,
                                       pointer_of<int32_t>(counts), pointer_of<int32_t>(lists), rows, (int)top, (int)w->size(0), glu ? 1 : 0, pointer(&out), (int)n,
                                       type_code(x), stream))
        return PyLong_FromLong(status);
    return THPVariable_Wrap(std::move(out));
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
    {"gated_linear", FAST(whole_gated_linear), METH_FASTCALL, nullptr},
    {"delta_rule", FAST(whole_delta_rule), METH_FASTCALL, nullptr},
    {"channel_linear", FAST(whole_channel_linear), METH_FASTCALL, nullptr},
    {"lightning", FAST(whole_lightning), METH_FASTCALL, nullptr},
    {"narrow_linear", FAST(whole_narrow_linear), METH_FASTCALL, nullptr},
    {"moe_choose", FAST(whole_moe_choose), METH_FASTCALL, nullptr},
    {"moe_product", FAST(whole_moe_product), METH_FASTCALL, nullptr},
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
