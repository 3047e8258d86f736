// Eager calls from Python.
//
// What torch.ops.macko_spmv.<name>.default(...) does on its way from Python to an operator's kernel (macko_torch.cpp; the arguments through
// the operator's schema onto a stack of values, the dispatcher, the stack again) takes longer than the rest of the call:
// 777 x 3333 at density 0.25, 5.8 us a call of `multiply`, of which the launch is 2.2 and the kernel, meanwhile, 4.0.  The
// functions below take the arguments from Python themselves, for calls that nothing but the CUDA kernel would see: plain
// tensors on one GPU, through which no gradient has to flow, and no mode, transform, recording, profiler or kernel of the
// program's own that is between Python and the kernel.  Anything else is answered with NotImplemented, and the caller goes
// through the operator.
//
// A library of its own: the operators' (libmacko_torch.so) is for programs without Python, too.

#include <Python.h>  // first, as its headers ask for

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>
#include <ATen/record_function.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "macko_torch.h"

namespace {

using namespace macko_torch;

// Nothing in this thread looks at operators: modes of Python, torch.func, tracing and whatever else adds dispatch keys
// of its own, autocasting (a program may have registered a rule); __torch_function__ modes; the profiler.
bool unobserved()
{
    const c10::impl::LocalDispatchKeySet tls = c10::impl::tls_local_dispatch_key_set();
    return (tls.included_ | c10::default_included_set) == c10::default_included_set &&
           tls.excluded_.has(c10::DispatchKey::AutocastCUDA) && !at::impl::torch_function_mode_enabled() && !at::hasCallbacks();
}

// A tensor whose operators only the CUDA kernel is registered for.
bool plain(const at::Tensor &t)
{
    constexpr c10::DispatchKeySet usual =
        c10::DispatchKeySet({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA});
    return t.defined() && t.is_cuda() && (t.key_set() | usual) == usual && !(t.requires_grad() && at::GradMode::is_enabled()) &&
           !t._fw_grad(0).defined();
}

// An operator and its kernel for the GPU.
template <typename F> class Operator;
template <typename R, typename... A> class Operator<R(A...)> {
    c10::OperatorHandle handle_;
    c10::TypedOperatorHandle<R(A...)> typed_;
    std::string registered_;

    std::string kernel_in_place() const { return handle_.getComputedKernelForDispatchKey(c10::DispatchKey::CUDA).debug(); }

public:
    explicit Operator(const char *name)
        : handle_(c10::Dispatcher::singleton().findSchemaOrThrow(name, "")), typed_(handle_.typed<R(A...)>()), registered_(kernel_in_place())
    {
    }
    // A program may have registered a kernel for what comes in front of the GPU's.
    bool first() const
    {
        for (const c10::DispatchKey key : {c10::DispatchKey::Autograd, c10::DispatchKey::AutogradCUDA, c10::DispatchKey::ADInplaceOrView,
                                           c10::DispatchKey::BackendSelect})
            if (handle_.hasKernelForDispatchKey(key)) return false;
        return true;
    }
    // ... or one in its place (asked only where the kernel is not called as the operator's)
    bool replaced() const { return kernel_in_place() != registered_; }
    R operator()(A... args) const { return typed_.redispatch(c10::DispatchKeySet(c10::DispatchKey::CUDA), std::forward<A>(args)...); }
};

#define MACKO_OPERATORS(X) \
    X(multiply) X(multiply_planned) X(multiply_axpby) X(multiply_axpby_planned) X(compress) X(plan)            \
    X(multiply_batched) X(multiply_int8) X(multiply_int8_axpby) X(multiply_rmsnorm) X(multiply_silu_mul_axpby) \
    X(multiply_attention_axpby) X(decode_rmsnorm) X(decode_norm_matvec) X(decode_rope_append)                  \
    X(decode_attention) X(decode_silu_mul) X(decode_rope_attention) X(decode_rope_attention_parts)             \
    X(pack_rmsnorm) X(rmsnorm_rows) X(pack_silu_mul) X(multiply_packed) X(multiply_packed_several)             \
    X(multiply_packed_silu) X(prefill_rope_append) X(prefill_attention)
#define MACKO_OPERATOR(NAME)                                                                  \
    struct NAME##_operator {                                                                   \
        typedef Operator<std::remove_pointer_t<decltype(&NAME##_hip)>> Type;                   \
        static const Type &get()                                                               \
        {                                                                                      \
            static const Type op("macko_spmv::" #NAME);                                        \
            return op;                                                                         \
        }                                                                                      \
    };
MACKO_OPERATORS(MACKO_OPERATOR)
#undef MACKO_OPERATOR

struct EagerCall {
    int device = -1;
    bool tensor(PyObject *o, const at::Tensor *&out)
    {
        if (!THPVariable_CheckExact(o)) return false;
        out = &THPVariable_Unpack(o);
        if (!plain(*out)) return false;
        const int index = out->get_device();
        if (device < 0) device = index;
        return index == device;
    }
    static bool integer(PyObject *o, int64_t &out)
    {
        if (!PyLong_CheckExact(o)) return false;
        int overflow = 0;
        out = PyLong_AsLongLongAndOverflow(o, &overflow);
        return overflow == 0;
    }
    static bool number(PyObject *o, double &out)
    {
        if (!PyFloat_CheckExact(o)) return false;
        out = PyFloat_AS_DOUBLE(o);
        return true;
    }
};

// An argument of an operator's kernel: what is kept of it while the call runs, and how it is handed over.
template <typename T> struct EagerArg;
template <> struct EagerArg<const at::Tensor &> {
    const at::Tensor *kept = nullptr;
    bool take(EagerCall &call, PyObject *o) { return call.tensor(o, kept); }
    const at::Tensor &give() const { return *kept; }
};
template <> struct EagerArg<at::Tensor> : EagerArg<const at::Tensor &> {};
template <> struct EagerArg<const std::optional<at::Tensor> &> {
    std::optional<at::Tensor> kept;
    bool take(EagerCall &call, PyObject *o)
    {
        if (o == Py_None) return true;
        const at::Tensor *t = nullptr;
        if (!call.tensor(o, t)) return false;
        kept = *t;
        return true;
    }
    const std::optional<at::Tensor> &give() const { return kept; }
};
template <> struct EagerArg<int64_t> {
    int64_t kept = 0;
    bool take(EagerCall &, PyObject *o) { return EagerCall::integer(o, kept); }
    int64_t give() const { return kept; }
};
template <> struct EagerArg<double> {
    double kept = 0.0;
    bool take(EagerCall &, PyObject *o) { return EagerCall::number(o, kept); }
    double give() const { return kept; }
};
template <> struct EagerArg<at::TensorList> {
    std::vector<at::Tensor> kept;
    bool take(EagerCall &call, PyObject *o)
    {
        if (!PyList_CheckExact(o)) return false;
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(o); ++i) {
            const at::Tensor *t = nullptr;
            if (!call.tensor(PyList_GET_ITEM(o, i), t)) return false;
            kept.push_back(*t);
        }
        return true;
    }
    at::TensorList give() const { return kept; }
};
template <> struct EagerArg<at::IntArrayRef> {
    std::vector<int64_t> kept;
    bool take(EagerCall &, PyObject *o)
    {
        if (!PyList_CheckExact(o)) return false;
        for (Py_ssize_t i = 0; i < PyList_GET_SIZE(o); ++i) {
            int64_t v = 0;
            if (!EagerCall::integer(PyList_GET_ITEM(o, i), v)) return false;
            kept.push_back(v);
        }
        return true;
    }
    at::IntArrayRef give() const { return kept; }
};

PyObject *to_python(at::Tensor &&t) { return THPVariable_Wrap(std::move(t)); }
PyObject *to_python(std::vector<at::Tensor> &&all)
{
    PyObject *list = PyList_New((Py_ssize_t)all.size());
    if (list == nullptr) return nullptr;
    for (size_t i = 0; i < all.size(); ++i) PyList_SET_ITEM(list, (Py_ssize_t)i, THPVariable_Wrap(std::move(all[i])));
    return list;
}

PyObject *not_implemented()
{
    Py_INCREF(Py_NotImplemented);
    return Py_NotImplemented;
}

struct WithoutGil {  // as around an operator's call: a launch may wait for room in the stream's queue
    PyThreadState *state = PyEval_SaveThread();
    ~WithoutGil() { PyEval_RestoreThread(state); }
};

template <typename R, typename... A, size_t... I>
PyObject *eager_call(const Operator<R(A...)> &op, std::index_sequence<I...>, PyObject *const *args, Py_ssize_t n)
{
    if (n != (Py_ssize_t)sizeof...(A) || !unobserved() || !op.first()) return not_implemented();
    EagerCall call;
    std::tuple<EagerArg<A>...> kept;
    if (!(std::get<I>(kept).take(call, args[I]) && ...)) return not_implemented();
    if constexpr (std::is_void_v<R>) {
        {
            WithoutGil released;
            op(std::get<I>(kept).give()...);
        }
        Py_RETURN_NONE;
    } else {
        std::optional<R> out;
        {
            WithoutGil released;
            out.emplace(op(std::get<I>(kept).give()...));
        }
        return to_python(std::move(*out));
    }
}

template <typename R, typename... A>
PyObject *eager_call(const Operator<R(A...)> &op, PyObject *const *args, Py_ssize_t n)
{
    return eager_call(op, std::index_sequence_for<A...>{}, args, n);
}

// The operator's own arguments, one by one.
template <typename OPERATOR> PyObject *eager(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    return eager_call(OPERATOR::get(), args, n);
    END_HANDLE_TH_ERRORS
}

// (compressed, V) and (compressed, V, C, alpha, beta) of a matrix that may carry its cuts as an attribute of row_indices
// (macko_spmv_amd/__init__.py).
PyObject *plan_attribute = nullptr;  // its name

struct Matrix {
    const at::Tensor *values = nullptr, *deltas = nullptr, *row_indices = nullptr, *plan = nullptr;
    at::Tensor plan_kept;
    int64_t rows = 0, cols = 0;
    bool take(EagerCall &call, PyObject *o)
    {
        PyObject *const *item;
        if (PyTuple_CheckExact(o) && PyTuple_GET_SIZE(o) >= 5)
            item = &PyTuple_GET_ITEM(o, 0);
        else
            return false;
        if (!call.tensor(item[0], values) || !call.tensor(item[1], deltas) || !call.tensor(item[2], row_indices) ||
            !EagerCall::integer(item[3], rows) || !EagerCall::integer(item[4], cols))
            return false;
        PyObject *found = nullptr;
        if (_PyObject_LookupAttr(item[2], plan_attribute, &found) < 0) {
            PyErr_Clear();
            return false;
        }
        if (found == nullptr) return true;
        bool fits = found == Py_None;
        if (!fits) {
            const at::Tensor *t = nullptr;
            fits = call.tensor(found, t);   // a plan of another device is the general path's to leave out
            if (fits) {
                plan_kept = *t;
                plan = &plan_kept;
            }
        }
        Py_DECREF(found);
        return fits;
    }
};

PyObject *eager_multiply(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    EagerCall call;
    Matrix m;
    const at::Tensor *v = nullptr;
    if (n != 2 || !unobserved() || !m.take(call, args[0]) || !call.tensor(args[1], v) || !v->is_contiguous()) return not_implemented();
    const auto &planned = multiply_planned_operator::get();
    const auto &bare = multiply_operator::get();
    if (!(m.plan != nullptr ? planned.first() : bare.first())) return not_implemented();
    at::Tensor out;
    {
        WithoutGil released;
        out = m.plan != nullptr ? planned(*m.values, *m.deltas, *m.row_indices, m.rows, m.cols, *v, *m.plan)
                                : bare(*m.values, *m.deltas, *m.row_indices, m.rows, m.cols, *v);
    }
    return to_python(std::move(out));
    END_HANDLE_TH_ERRORS
}

PyObject *eager_multiply_axpby(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    EagerCall call;
    Matrix m;
    const at::Tensor *v = nullptr, *c = nullptr;
    double alpha = 0.0, beta = 0.0;
    if (n != 5 || !unobserved() || !m.take(call, args[0]) || !call.tensor(args[1], v) || !call.tensor(args[2], c) ||
        !EagerCall::number(args[3], alpha) || !EagerCall::number(args[4], beta) || !v->is_contiguous() || !c->is_contiguous())
        return not_implemented();
    const auto &planned = multiply_axpby_planned_operator::get();
    const auto &bare = multiply_axpby_operator::get();
    if (!(m.plan != nullptr ? planned.first() : bare.first())) return not_implemented();
    {
        WithoutGil released;
        if (m.plan != nullptr)
            planned(*m.values, *m.deltas, *m.row_indices, m.rows, m.cols, *v, *c, alpha, beta, *m.plan);
        else
            bare(*m.values, *m.deltas, *m.row_indices, m.rows, m.cols, *v, *c, alpha, beta);
    }
    Py_INCREF(args[2]);
    return args[2];
    END_HANDLE_TH_ERRORS
}

// Whether compress and plan still have their own kernels.  The dispatcher answers with copies of strings, so it is asked while
// the count pass is running anyway.
bool compress_not_replaced() noexcept
{
    const PyGILState_STATE state = PyGILState_Ensure();  // kernels are registered with the lock held
    bool replaced = true;
    try {
        replaced = compress_operator::get().replaced() || plan_operator::get().replaced();
    } catch (...) {
    }
    PyGILState_Release(state);
    return !replaced;
}

// compress(M): the five of the operator and the plan (None: products of this shape take none), which the operator `plan` makes
// otherwise.
PyObject *eager_compress(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    EagerCall call;
    const at::Tensor *M = nullptr;
    if (n != 1 || !unobserved() || !call.tensor(args[0], M) || M->dtype() != at::kHalf || M->dim() != 2 || !M->is_contiguous())
        return not_implemented();
    if (!compress_operator::get().first() || !plan_operator::get().first()) return not_implemented();
    at::Tensor plan;
    std::optional<Compressed> out;
    {
        WithoutGil released;
        out.emplace(compress_on_device(*M, &plan, &compress_not_replaced));
    }
    if (!std::get<0>(*out).defined()) return not_implemented();
    PyObject *found = Py_None;
    if (plan.numel() > 0)
        found = THPVariable_Wrap(std::move(plan));
    else
        Py_INCREF(found);
    return Py_BuildValue("NNNLLN", THPVariable_Wrap(std::get<0>(*out)), THPVariable_Wrap(std::get<1>(*out)),
                         THPVariable_Wrap(std::get<2>(*out)), (long long)std::get<3>(*out), (long long)std::get<4>(*out), found);
    END_HANDLE_TH_ERRORS
}

// What Block.forward_fused (llm.py) does with the layer of a prompt, operator by operator, in one call: (x, cos, sin,
// positions, k_cache, v_cache, scale, norm weight, eps, norm weight, eps, then the five of q, k, v, o, gate, up and down each).
// A layer's nine launches take less time than Python takes between them where the layer is small: a prompt of 16 tokens,
// 4 layers of dim 512 391 -> 347 us, 100 tokens, 3 layers of dim 1024 323 -> 285; 128 tokens at dim 4096 the same (699).
PyObject *eager_prefill_layer(PyObject *, PyObject *const *args, Py_ssize_t n)
{
    HANDLE_TH_ERRORS
    struct Linear {
        const at::Tensor *values, *deltas, *row_indices;
        int64_t rows, cols;
    };
    constexpr int kLinears = 7, kOthers = 11;
    enum { Q, K, V, O, GATE, UP, DOWN };
    EagerCall call;
    const at::Tensor *x, *cos, *sin, *positions, *k_cache, *v_cache, *norm[2];
    double scale, eps[2];
    Linear m[kLinears];
    if (n != kOthers + 5 * kLinears || !unobserved() || !call.tensor(args[0], x) || !call.tensor(args[1], cos) || !call.tensor(args[2], sin) ||
        !call.tensor(args[3], positions) || !call.tensor(args[4], k_cache) || !call.tensor(args[5], v_cache) ||
        !EagerCall::number(args[6], scale) || !call.tensor(args[7], norm[0]) || !EagerCall::number(args[8], eps[0]) ||
        !call.tensor(args[9], norm[1]) || !EagerCall::number(args[10], eps[1]))
        return not_implemented();
    for (int i = 0; i < kLinears; ++i) {
        PyObject *const *five = args + kOthers + 5 * i;
        if (!call.tensor(five[0], m[i].values) || !call.tensor(five[1], m[i].deltas) || !call.tensor(five[2], m[i].row_indices) ||
            !EagerCall::integer(five[3], m[i].rows) || !EagerCall::integer(five[4], m[i].cols))
            return not_implemented();
    }
    const auto &normed = pack_rmsnorm_operator::get();
    const auto &several = multiply_packed_several_operator::get();
    const auto &rope = prefill_rope_append_operator::get();
    const auto &attention = prefill_attention_operator::get();
    const auto &product = multiply_packed_operator::get();
    const auto &gate = multiply_packed_silu_operator::get();
    if (x->dim() != 3 || x->size(0) != 1 || k_cache->dim() != 4 || v_cache->dim() != 4 || !normed.first() || !several.first() ||
        !rope.first() || !attention.first() || !product.first() || !gate.first())
        return not_implemented();
    at::Tensor out;
    {
        WithoutGil released;
        const int64_t tokens = x->size(1);
        const at::Tensor rows = x->reshape({tokens, -1}).contiguous(), at = positions->contiguous();
        const at::Tensor keys = k_cache->select(0, 0), values = v_cache->select(0, 0);
        at::Tensor packed = normed(rows, *norm[0], eps[0]);
        {
            const at::Tensor v[3] = {*m[Q].values, *m[K].values, *m[V].values}, d[3] = {*m[Q].deltas, *m[K].deltas, *m[V].deltas},
                             r[3] = {*m[Q].row_indices, *m[K].row_indices, *m[V].row_indices};
            const int64_t n_rows[3] = {m[Q].rows, m[K].rows, m[V].rows};
            const auto qkv = several(v, d, r, n_rows, m[Q].cols, packed, tokens);
            rope(qkv[0], qkv[1], qkv[2], cos->reshape({tokens, -1}), sin->reshape({tokens, -1}), at, keys, values);
            packed = attention(qkv[0], keys, values, at, scale);
        }
        const at::Tensor after = product(*m[O].values, *m[O].deltas, *m[O].row_indices, m[O].rows, m[O].cols, packed, tokens, rows);
        packed = normed(after, *norm[1], eps[1]);
        {
            const at::Tensor v[2] = {*m[GATE].values, *m[UP].values}, d[2] = {*m[GATE].deltas, *m[UP].deltas},
                             r[2] = {*m[GATE].row_indices, *m[UP].row_indices};
            packed = gate(v, d, r, m[GATE].rows, m[GATE].cols, packed, tokens);
        }
        out = product(*m[DOWN].values, *m[DOWN].deltas, *m[DOWN].row_indices, m[DOWN].rows, m[DOWN].cols, packed, tokens, after).view({1, tokens, -1});
    }
    return to_python(std::move(out));
    END_HANDLE_TH_ERRORS
}

#define MACKO_EAGER(NAME, ...) {#NAME, (PyCFunction)(void (*)(void))&__VA_ARGS__, METH_FASTCALL, nullptr}
PyMethodDef eager_functions[] = {
    MACKO_EAGER(compress, eager_compress),
    MACKO_EAGER(multiply, eager_multiply),
    MACKO_EAGER(multiply_axpby, eager_multiply_axpby),
    MACKO_EAGER(multiply_batched, eager<multiply_batched_operator>),
    MACKO_EAGER(multiply_int8, eager<multiply_int8_operator>),
    MACKO_EAGER(multiply_int8_axpby, eager<multiply_int8_axpby_operator>),
    MACKO_EAGER(multiply_rmsnorm, eager<multiply_rmsnorm_operator>),
    MACKO_EAGER(multiply_silu_mul_axpby, eager<multiply_silu_mul_axpby_operator>),
    MACKO_EAGER(multiply_attention_axpby, eager<multiply_attention_axpby_operator>),
    MACKO_EAGER(decode_rmsnorm, eager<decode_rmsnorm_operator>),
    MACKO_EAGER(decode_norm_matvec, eager<decode_norm_matvec_operator>),
    MACKO_EAGER(decode_rope_append, eager<decode_rope_append_operator>),
    MACKO_EAGER(decode_attention, eager<decode_attention_operator>),
    MACKO_EAGER(decode_silu_mul, eager<decode_silu_mul_operator>),
    MACKO_EAGER(decode_rope_attention, eager<decode_rope_attention_operator>),
    MACKO_EAGER(decode_rope_attention_parts, eager<decode_rope_attention_parts_operator>),
    MACKO_EAGER(pack_rmsnorm, eager<pack_rmsnorm_operator>),
    MACKO_EAGER(rmsnorm_rows, eager<rmsnorm_rows_operator>),
    MACKO_EAGER(pack_silu_mul, eager<pack_silu_mul_operator>),
    MACKO_EAGER(multiply_packed, eager<multiply_packed_operator>),
    MACKO_EAGER(multiply_packed_several, eager<multiply_packed_several_operator>),
    MACKO_EAGER(multiply_packed_silu, eager<multiply_packed_silu_operator>),
    MACKO_EAGER(prefill_rope_append, eager<prefill_rope_append_operator>),
    MACKO_EAGER(prefill_attention, eager<prefill_attention_operator>),
    MACKO_EAGER(prefill_layer, eager_prefill_layer),
    {nullptr, nullptr, 0, nullptr}};
#undef MACKO_EAGER
PyModuleDef eager_module = {PyModuleDef_HEAD_INIT, "libmacko_eager", nullptr, -1, eager_functions, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_libmacko_eager()
{
    HANDLE_TH_ERRORS
#define MACKO_OPERATOR(NAME) NAME##_operator::get();
    MACKO_OPERATORS(MACKO_OPERATOR)   // with the kernels that are registered now
#undef MACKO_OPERATOR
    plan_attribute = PyUnicode_InternFromString("_macko_spmv_plan");
    return plan_attribute == nullptr ? nullptr : PyModule_Create(&eager_module);
    END_HANDLE_TH_ERRORS
}
