// Python entry points of the operators that skip the interpretation of their schemas.
//
// torch.ops.gpuk.<op>(...) finds the overload, matches every Python argument against the schema and boxes it, which takes
// longer than everything else the host does for a small call but the launch: us per call that way / this way 4.79 / 3.42 for
// allreduce_rms of one row (nine arguments), 5.50 / 3.66 for fused_rope_rms_set_kv of 32 tokens (eighteen), of which the
// launch is 2.8 and what the operator itself does beside it 0.2.  The functions here take the same positional arguments,
// unpack them by the type the operator's C++ signature names and call the operator through the dispatcher, so that
// profiling, dispatch modes, functorch and the keys other code registers see the call as before.  Whatever is not plain --
// keywords, another number of arguments, tensor subclasses, symbolic or other numbers, a __torch_function__ mode, a trace
// being recorded -- goes to the callable that the function was made with, which is the packet's own.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/dispatch/Dispatcher.h>

#include <optional>
#include <string>
#include <tuple>
#include <type_traits>
#include <utility>

#include "ops/ops.h"

namespace {

// One argument: parse() says whether the object is the plain form of what the operator takes, and pass() hands it on.
template <typename A> struct Argument;

template <> struct Argument<at::Tensor &> {
    at::Tensor value;
    bool parse(PyObject *o) {
        if (!THPVariable_CheckExact(o)) return false;
        value = THPVariable_Unpack(o);
        return true;
    }
    at::Tensor &pass() { return value; }
};
template <> struct Argument<const at::Tensor &> : Argument<at::Tensor &> {};
template <> struct Argument<int64_t> {
    int64_t value;
    bool parse(PyObject *o) {
        if (!PyLong_CheckExact(o)) return false;
        int overflow = 0;
        value = PyLong_AsLongLongAndOverflow(o, &overflow);
        return overflow == 0;
    }
    int64_t pass() { return value; }
};
template <> struct Argument<double> {
    double value;
    bool parse(PyObject *o) {
        if (!PyFloat_CheckExact(o)) return false;
        value = PyFloat_AS_DOUBLE(o);
        return true;
    }
    double pass() { return value; }
};
template <> struct Argument<bool> {
    bool value;
    bool parse(PyObject *o) {
        value = o == Py_True;
        return o == Py_True || o == Py_False;
    }
    bool pass() { return value; }
};
template <> struct Argument<std::vector<int64_t>> {
    std::vector<int64_t> value;
    bool parse(PyObject *o) {
        if (!PyList_CheckExact(o) && !PyTuple_CheckExact(o)) return false;
        const Py_ssize_t n = PySequence_Fast_GET_SIZE(o);
        PyObject **items = PySequence_Fast_ITEMS(o);
        for (Py_ssize_t i = 0; i < n; ++i) {
            Argument<int64_t> one;
            if (!one.parse(items[i])) return false;
            value.push_back(one.value);
        }
        return true;
    }
    std::vector<int64_t> pass() { return std::move(value); }
};

template <typename... R, size_t... I>
PyObject *as_tuple(std::tuple<R...> &result, std::index_sequence<I...>) {
    PyObject *items[] = {THPVariable_Wrap(std::move(std::get<I>(result)))...};
    PyObject *tuple = PyTuple_New(sizeof...(R));
    bool ok = tuple != nullptr;
    for (PyObject *item : items) ok = ok && item != nullptr;
    if (!ok) {
        for (PyObject *item : items) Py_XDECREF(item);
        Py_XDECREF(tuple);
        return nullptr;
    }
    (PyTuple_SET_ITEM(tuple, I, items[I]), ...);
    return tuple;
}

template <auto F, auto G>
constexpr bool same_function = std::is_same_v<std::integral_constant<decltype(F), F>, std::integral_constant<decltype(G), G>>;

template <auto F> struct Call;
template <typename R, typename... A, R (*F)(A...)>
struct Call<F> {
    using Handle = c10::TypedOperatorHandle<R(A...)>;
    static inline std::optional<Handle> handle;  // set when the function is made, before it can be called
    static void find(const char *name, const char *overload) {
        if (!handle) handle = c10::Dispatcher::singleton().findSchemaOrThrow(name, overload).template typed<R(A...)>();
    }

    template <size_t... I>
    static PyObject *run(std::tuple<Argument<A>...> &args, std::index_sequence<I...>) {
        HANDLE_TH_ERRORS
        if constexpr (std::is_void_v<R>) {
            {
                pybind11::gil_scoped_release no_gil;
                handle->call(std::get<I>(args).pass()...);
            }
            Py_RETURN_NONE;
        } else {
            auto result = [&] {
                pybind11::gil_scoped_release no_gil;
                if constexpr (same_function<F, &gpuk_ops::add_rms_fused_static>) {
                    // (the scale comes back as a third output, in the shape the callers of
                    // GPUKDistEnv.allreduce_add_rms_fused expect; reshaped from Python it cost as much as an allocation)
                    auto [residual_out, norm_out] = handle->call(std::get<I>(args).pass()...);
                    return std::make_tuple(std::move(residual_out), std::move(norm_out), std::get<4>(args).value.reshape({1}));
                } else {
                    return handle->call(std::get<I>(args).pass()...);
                }
            }();
            return as_tuple(result, std::make_index_sequence<std::tuple_size_v<decltype(result)>>{});
        }
        END_HANDLE_TH_ERRORS
    }
    template <size_t... I>
    static bool parse(std::tuple<Argument<A>...> &args, PyObject *const *objects, std::index_sequence<I...>) {
        return (std::get<I>(args).parse(objects[I]) && ...);
    }
    // self: the general callable
    static PyObject *call(PyObject *self, PyObject *const *objects, Py_ssize_t count, PyObject *keywords) {
        constexpr auto each = std::index_sequence_for<A...>{};
        if (count == (Py_ssize_t)sizeof...(A) && (!keywords || PyTuple_GET_SIZE(keywords) == 0) &&
            !at::impl::torch_function_mode_enabled() && !torch::jit::tracer::isTracing()) {
            std::tuple<Argument<A>...> args;
            if (parse(args, objects, each)) return run(args, each);
        }
        return PyObject_Vectorcall(self, objects, (size_t)count, keywords);
    }
};

// direct(name, overload, general): a function that calls gpuk::name (overload) directly where it can, `general` elsewhere.
template <auto F>
PyObject *make(const char *name, const char *overload, PyObject *general) {
    static PyMethodDef method = {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Call<F>::call)), METH_FASTCALL | METH_KEYWORDS, nullptr};
    Call<F>::find((std::string("gpuk::") + name).c_str(), overload);
    return PyCFunction_NewEx(&method, general, nullptr);
}
struct Entry {
    const char *name, *overload;
    PyObject *(*make)(const char *, const char *, PyObject *);
};
const Entry kEntries[] = {
    {"allreduce_rms", "", &make<&gpuk_ops::allreduce_rms>},
    {"add_rms_fused", "", &make<&gpuk_ops::add_rms_fused>},
    {"add_rms_fused", "static", &make<&gpuk_ops::add_rms_fused_static>},
    {"fused_rope_rms", "", &make<&gpuk_ops::fused_rope_rms>},
    {"fused_mrope_3d_rms", "", &make<&gpuk_ops::fused_mrope_3d_rms>},
    {"fused_rope_rms_set_kv", "", &make<&gpuk_ops::fused_rope_rms_set_kv>},
    {"fused_mrope_3d_rms_set_kv", "", &make<&gpuk_ops::fused_mrope_3d_rms_set_kv>},
    {"fused_rope_rms_2way", "", &make<&gpuk_ops::fused_rope_rms_2way>},
};

PyObject *direct(PyObject *, PyObject *args) {
    HANDLE_TH_ERRORS
    const char *name = nullptr, *overload = nullptr;
    PyObject *general = nullptr;
    if (!PyArg_ParseTuple(args, "ssO:direct", &name, &overload, &general)) return nullptr;
    for (const Entry &e : kEntries)
        if (std::string(e.name) == name && std::string(e.overload) == overload) return e.make(e.name, e.overload, general);
    PyErr_Format(PyExc_ValueError, "no direct call of gpuk::%s.%s", name, overload);
    return nullptr;
    END_HANDLE_TH_ERRORS
}

PyObject *current_stream_is_capturing(PyObject *, PyObject *) {
    HANDLE_TH_ERRORS
    return PyBool_FromLong(gpuk_ops::current_stream_is_capturing());
    END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {{"current_stream_is_capturing", current_stream_is_capturing, METH_NOARGS, "as torch.cuda.is_current_stream_capturing()"},
                          {"direct", direct, METH_VARARGS, "direct(name, overload, general) -> function"}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "gpuk_direct", nullptr, -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit_gpuk_direct() { return PyModule_Create(&kModule); }
