// Calls of the C ABI with torch tensors as they come from Python: checking a tensor, taking its address and converting the
// arguments costs a few hundred nanoseconds here, and five to eight microseconds through ctypes, which is what a small
// layer's kernel takes.  An entry point's argument types come from its declaration.  A call with anything but plain
// tensors, None and numbers is not made here: it answers None, and the caller goes through ctypes and its checks.
#include <torch/csrc/autograd/python_variable.h>

#include "pixienn_hip.h"

#include <climits>
#include <exception>
#include <string_view>
#include <tuple>
#include <type_traits>
#include <utility>

namespace {

// Thrown for an argument that is left to the caller.
struct NotHere {};

template<typename A>
A argument(PyObject* o)
{
    if constexpr (std::is_same_v<A, float*> || std::is_same_v<A, const float*>) {
        // a tensor the kernels take: fp32, contiguous, on a HIP device
        if (o == Py_None) return nullptr;
        if (!THPVariable_CheckExact(o)) throw NotHere{};
        const at::Tensor& t = THPVariable_Unpack(o);
        if (t.scalar_type() != at::kFloat || !t.is_cuda() || !t.is_contiguous()) throw NotHere{};
        return static_cast<float*>(t.data_ptr());
    } else if constexpr (std::is_pointer_v<A>) {
        if (o == Py_None) return nullptr;
        if (!PyLong_CheckExact(o)) throw NotHere{};
        void* p = PyLong_AsVoidPtr(o);
        if (PyErr_Occurred()) { PyErr_Clear(); throw NotHere{}; }
        return reinterpret_cast<A>(p);
    } else if constexpr (std::is_same_v<A, float>) {
        if (!PyFloat_CheckExact(o)) throw NotHere{};
        return static_cast<float>(PyFloat_AS_DOUBLE(o));
    } else {
        static_assert(std::is_integral_v<A>, "a kind of argument of its own");
        if (!PyLong_CheckExact(o)) throw NotHere{};
        int overflow = 0;
        const long long v = PyLong_AsLongLongAndOverflow(o, &overflow);
        if (overflow || (std::is_same_v<A, int> && (v < INT_MIN || v > INT_MAX)) || (std::is_unsigned_v<A> && v < 0) ||
            (std::is_same_v<A, unsigned> && v > static_cast<long long>(UINT_MAX)))
            throw NotHere{};
        return static_cast<A>(v);
    }
}

template<typename F>
struct Entry;

// `self` holds the entry point's address in the loaded library.
template<typename... A>
struct Entry<int (*)(A...)> {
    using Function = int (*)(A...);

    template<size_t... I>
    static int call(Function f, PyObject* const* args, std::index_sequence<I...>)
    {
        const std::tuple<A...> values{ argument<A>(args[I])... };
        int rc;
        PyThreadState* const state = PyEval_SaveThread();
        rc = std::apply(f, values);
        PyEval_RestoreThread(state);
        return rc;
    }

    static PyObject* vectorcall(PyObject* self, PyObject* const* args, Py_ssize_t count)
    {
        if (count != static_cast<Py_ssize_t>(sizeof...(A))) Py_RETURN_NONE;
        const auto f = reinterpret_cast<Function>(PyLong_AsVoidPtr(self));
        try {
            return PyLong_FromLong(call(f, args, std::index_sequence_for<A...>{}));
        } catch (const NotHere&) {
        } catch (const std::exception&) {       // a tensor without storage, say: the caller's route reports it
        }
        Py_RETURN_NONE;
    }

    // which arguments are tensors
    static PyObject* tensors()
    {
        PyObject* t = PyTuple_New(sizeof...(A));
        Py_ssize_t i = 0;
        if (t) ((PyTuple_SET_ITEM(t, i++, PyBool_FromLong(std::is_same_v<A, float*> || std::is_same_v<A, const float*>))), ...);
        return t;
    }
};

struct Known {
    PyMethodDef def;
    PyObject* (*tensors)();
};

template<auto F>
Known known(const char* name)
{
    using E = Entry<decltype(F)>;
    return Known{ { name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&E::vectorcall)), METH_FASTCALL, nullptr },
                  &E::tensors };
}

#define ENTRY(name) known<&name>(#name)

Known entries[] = {
    ENTRY(pxh_bn_train_act_forward), ENTRY(pxh_bn_train_act_shortcut_forward), ENTRY(pxh_bn_folded_act_forward),
    ENTRY(pxh_bn_folded_act_shortcut_forward), ENTRY(pxh_bn_folded_act_maxpool_forward), ENTRY(pxh_bias_act_forward),
    ENTRY(pxh_bn_act_backward), ENTRY(pxh_bn_act_backward_clipped), ENTRY(pxh_bias_act_backward),
    ENTRY(pxh_bias_act_backward_clipped), ENTRY(pxh_axpy), ENTRY(pxh_fill_f32), ENTRY(pxh_route_forward),
    ENTRY(pxh_route_backward), ENTRY(pxh_maxpool_forward), ENTRY(pxh_maxpool_backward), ENTRY(pxh_shortcut_backward_clipped),
    ENTRY(pxh_yolo_activate), ENTRY(pxh_yolo_detections_append), ENTRY(pxh_rescale_clip), ENTRY(pxh_adam_update),
    ENTRY(pxh_sgd_update),
};

// bind(name, address) -> (callable, which arguments are tensors), or None for an entry point that is not made here
PyObject* bind(PyObject*, PyObject* args)
{
    const char* name;
    PyObject* address;
    if (!PyArg_ParseTuple(args, "sO!", &name, &PyLong_Type, &address)) return nullptr;
    for (Known& k: entries) {
        if (std::string_view(k.def.ml_name) != name) continue;
        PyObject* f = PyCFunction_New(&k.def, address);
        PyObject* t = f ? k.tensors() : nullptr;
        if (!t) { Py_XDECREF(f); return nullptr; }
        return Py_BuildValue("(NN)", f, t);
    }
    Py_RETURN_NONE;
}

// names() -> the entry points that are made here
PyObject* names(PyObject*, PyObject*)
{
    PyObject* list = PyList_New(0);
    for (const Known& k: entries) {
        PyObject* s = list ? PyUnicode_FromString(k.def.ml_name) : nullptr;
        if (!s || PyList_Append(list, s)) { Py_XDECREF(s); Py_XDECREF(list); return nullptr; }
        Py_DECREF(s);
    }
    return list;
}

PyMethodDef methods[] = { { "bind", bind, METH_VARARGS, nullptr }, { "names", names, METH_NOARGS, nullptr },
                          { nullptr, nullptr, 0, nullptr } };
PyModuleDef module = { PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr };

}  // namespace

PyMODINIT_FUNC PyInit__calls() { return PyModule_Create(&module); }
