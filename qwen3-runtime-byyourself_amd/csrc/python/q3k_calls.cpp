// The C entry points as Python callables, for the package's wrappers.
//
// A small launch costs the host more than the GPU: through ctypes a call's
// argument conversion took 0.7 us (rms_norm) to 5 us (gqa_attention with its
// stride arrays) beside 2 us in the HIP launch.  Here a vectorcall function per
// entry point converts the positional arguments from the C signature itself,
// in 0.1-0.3 us, and releases the interpreter lock around the call as ctypes
// does.  Conversions follow ctypes: integers wrap to the parameter's width,
// pointers are None, an int, or an object whose .ptr is one of these.  Any other
// argument makes the call return None without calling anything, and the wrapper
// goes through ctypes, with its conversions and its errors.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <stdint.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "q3k_abi.h"

namespace
{
    PyObject *g_ptr_name;

    bool to_address(PyObject *o, uintptr_t *out)
    {
        if (o == Py_None)
        {
            *out = 0;
            return true;
        }
        if (PyLong_CheckExact(o))
        {
            *out = static_cast<uintptr_t>(PyLong_AsUnsignedLongLongMask(o));
            return true;
        }
        return false;
    }

    // Four element strides, as the attention entry point takes them.
    struct Strides
    {
        int64_t v[4];
    };

    template <typename T>
    bool convert(PyObject *o, T *out)
    {
        if constexpr (std::is_pointer_v<T>)
        {
            uintptr_t a = 0;
            if (!to_address(o, &a))
            {
                PyObject *p = PyObject_GetAttr(o, g_ptr_name);
                if (p == nullptr)
                {
                    PyErr_Clear();
                    return false;
                }
                const bool ok = to_address(p, &a);
                Py_DECREF(p);
                if (!ok)
                    return false;
            }
            *out = reinterpret_cast<T>(a);
            return true;
        }
        else if constexpr (std::is_floating_point_v<T>)
        {
            if (!PyFloat_CheckExact(o))
                return false;
            *out = static_cast<T>(PyFloat_AS_DOUBLE(o));
            return true;
        }
        else
        {
            if (!PyLong_CheckExact(o))
                return false;
            *out = static_cast<T>(PyLong_AsUnsignedLongLongMask(o));
            return true;
        }
    }

    // A tuple of four ints.
    template <>
    bool convert<Strides>(PyObject *o, Strides *out)
    {
        if (!PyTuple_CheckExact(o) || PyTuple_GET_SIZE(o) != 4)
            return false;
        for (int i = 0; i < 4; ++i)
        {
            PyObject *e = PyTuple_GET_ITEM(o, i);
            if (!PyLong_CheckExact(e))
                return false;
            out->v[i] = static_cast<int64_t>(PyLong_AsUnsignedLongLongMask(e));
        }
        return true;
    }

    template <typename T>
    T pass(T v)
    {
        return v;
    }
    const int64_t *pass(const Strides &s) { return s.v; }

    template <auto Fn, typename... A, size_t... I>
    PyObject *call_with(PyObject *const *args, std::tuple<A...> &v, std::index_sequence<I...>)
    {
        if (!(convert(args[I], &std::get<I>(v)) && ...))
            Py_RETURN_NONE;
        long long result;
        Py_BEGIN_ALLOW_THREADS;
        result = static_cast<long long>(Fn(pass(std::get<I>(v))...));
        Py_END_ALLOW_THREADS;
        return PyLong_FromLongLong(result);
    }

    template <auto Fn, typename... A>
    PyObject *call_typed(PyObject *const *args, Py_ssize_t n)
    {
        if (n != static_cast<Py_ssize_t>(sizeof...(A)))
        {
            PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
            return nullptr;
        }
        std::tuple<A...> v;
        return call_with<Fn>(args, v, std::index_sequence_for<A...>{});
    }

    template <auto Fn, typename R, typename... A>
    PyObject *call_deduced(R (*)(A...), PyObject *const *args, Py_ssize_t n)
    {
        return call_typed<Fn, A...>(args, n);
    }

    template <auto Fn>
    PyObject *entry(PyObject *, PyObject *const *args, Py_ssize_t n)
    {
        return call_deduced<Fn>(Fn, args, n);
    }

    PyObject *attention(PyObject *, PyObject *const *args, Py_ssize_t n)
    {
        return call_typed<&q3k_gqa_attention_bf16, const uint16_t *, const uint16_t *, const uint16_t *, uint16_t *, int64_t,
                          int64_t, int32_t, int32_t, int32_t, int64_t, int64_t, Strides, Strides, void *, int64_t,
                          q3k_stream_t>(args, n);
    }

#define Q3K_ENTRY(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<&name>)), METH_FASTCALL, nullptr}
    PyMethodDef g_methods[] = {
        Q3K_ENTRY(q3k_embedding_bf16),
        Q3K_ENTRY(q3k_rms_norm_bf16),
        Q3K_ENTRY(q3k_add_rms_norm_bf16),
        Q3K_ENTRY(q3k_rms_norm_rows_bf16),
        Q3K_ENTRY(q3k_add_rms_norm_rows_bf16),
        Q3K_ENTRY(q3k_embedding_rms_norm_bf16),
        Q3K_ENTRY(q3k_add_inplace_bf16),
        Q3K_ENTRY(q3k_silu_mul_bf16),
        Q3K_ENTRY(q3k_rope_bf16),
        Q3K_ENTRY(q3k_rope_qk_bf16),
        Q3K_ENTRY(q3k_qk_norm_rope_bf16),
        {"q3k_gqa_attention_bf16", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&attention)), METH_FASTCALL,
         nullptr},
        Q3K_ENTRY(q3k_argmax_bf16),
        Q3K_ENTRY(q3k_argmax_bf16_noalloc),
        Q3K_ENTRY(q3k_topk_candidates_bf16),
        Q3K_ENTRY(q3k_kv_append),
        Q3K_ENTRY(q3k_qk_norm_rope_kv_append_bf16),
        {nullptr, nullptr, 0, nullptr},
    };

    PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "q3k_calls", "The C entry points as Python callables.", -1, g_methods,
                            nullptr, nullptr, nullptr, nullptr};
} // namespace

PyMODINIT_FUNC PyInit_q3k_calls()
{
    g_ptr_name = PyUnicode_InternFromString("ptr");
    if (g_ptr_name == nullptr)
        return nullptr;
    return PyModule_Create(&g_module);
}
