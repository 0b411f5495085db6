// The engine call of the Python mirror (acrotensor_amd/api.py), and the two that open and close a multi-kernel launch, as
// CPython functions over the C ABI.  A program that goes
// through ctypes pays for every argument's conversion; a solver on a small batch issues its kernels faster than that (a
// mass apply of seven recorded kernels takes 2 us on the device).  Per recorded kernel of a capture that is repeated, the C
// ABI's own 0.1 us included: 0.3 us, and 1.9 us through ctypes (both measured on one host).
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <vector>

#include "acrotensor_hip.h"

namespace
{
PyObject *g_address = nullptr;  // "_address": the attribute that holds a tensor's handle as an integer

bool handleOf(PyObject *tensor, acro_tensor **handle)
{
    PyObject *address = PyObject_GetAttr(tensor, g_address);
    if (address == nullptr) return false;
    *handle = static_cast<acro_tensor *>(PyLong_AsVoidPtr(address));
    Py_DECREF(address);
    return PyErr_Occurred() == nullptr;
}

// contract(engine address, kernel string, output tensor, tuple of input tensors) -> status of acro_engine_contract
PyObject *contract(PyObject *, PyObject *const *args, Py_ssize_t count)
{
    if (count != 4 || !PyUnicode_Check(args[1]) || !PyTuple_Check(args[3]))
    {
        PyErr_SetString(PyExc_TypeError, "contract(engine, kernel string, output, tuple of inputs)");
        return nullptr;
    }
    acro_engine *engine = static_cast<acro_engine *>(PyLong_AsVoidPtr(args[0]));
    if (engine == nullptr && PyErr_Occurred() != nullptr) return nullptr;
    const char *kernel = PyUnicode_AsUTF8(args[1]);
    if (kernel == nullptr) return nullptr;
    const Py_ssize_t n = PyTuple_GET_SIZE(args[3]);
    acro_tensor *out = nullptr, *few[8];
    std::vector<acro_tensor *> many;
    acro_tensor **inputs = few;
    if (n > 8)
    {
        many.resize(static_cast<size_t>(n));
        inputs = many.data();
    }
    if (!handleOf(args[2], &out)) return nullptr;
    for (Py_ssize_t i = 0; i < n; ++i)
    {
        if (!handleOf(PyTuple_GET_ITEM(args[3], i), &inputs[i])) return nullptr;
    }
    int status = 0;
    // (the arguments keep the tensors and the string alive; other threads run meanwhile, as under ctypes)
    Py_BEGIN_ALLOW_THREADS
    status = acro_engine_contract(engine, kernel, out, inputs, static_cast<int>(n));
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
}

// begin(engine address), end(engine address) -> status of acro_engine_begin_ / _end_multi_kernel_launch
template <int (*ENTRY)(acro_engine *)>
PyObject *capture(PyObject *, PyObject *address)
{
    acro_engine *engine = static_cast<acro_engine *>(PyLong_AsVoidPtr(address));
    if (engine == nullptr && PyErr_Occurred() != nullptr) return nullptr;
    int status = 0;
    Py_BEGIN_ALLOW_THREADS
    status = ENTRY(engine);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(status);
}

PyMethodDef methods[] = {
    {"begin", capture<acro_engine_begin_multi_kernel_launch>, METH_O, nullptr},
    {"end", capture<acro_engine_end_multi_kernel_launch>, METH_O, nullptr},
    {"contract", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(contract)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_acro_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};
}  // namespace

PyMODINIT_FUNC PyInit__acro_call(void)
{
    g_address = PyUnicode_InternFromString("_address");
    return g_address != nullptr ? PyModule_Create(&module) : nullptr;
}
