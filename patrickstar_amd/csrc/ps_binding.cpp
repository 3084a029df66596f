// adam_update of the operator module, from Python arguments to ps_adam_update without Python in between.
//
// A per-tensor loop calls the operator once for every tensor, 199 times for a BERT-base-sized module, and most of those
// tensors take the GPU less time than the call takes the host: 6.4 us a call, of which the checks of four tensors in
// Python were 1.3 and the conversion of seventeen arguments by ctypes 1.7 us.
//
// The function here takes calls of the ordinary form only: plain tensors and numbers, everything on the current device.
// Whatever else it is given it leaves alone and returns None; the caller then goes through its general path, which accepts or
// refuses it as always.  Nothing is kept between calls.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdio>
#include <exception>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "ps_adam.h"

namespace {

// A flat, contiguous tensor of the GPU `device` (-1: of any; then it is set) and of one of two types.
bool plain(PyObject* o, at::ScalarType a, at::ScalarType b, int& device, int64_t& numel, const at::Tensor*& out)
{
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || t.layout() != at::kStrided || !t.is_cuda() || t.dim() != 1 || !t.is_contiguous()) return false;
    if (t.scalar_type() != a && t.scalar_type() != b) return false;
    if (device >= 0 && (t.get_device() != device || t.numel() != numel)) return false;
    device = t.get_device();
    numel = t.numel();
    out = &t;
    return true;
}

bool number(PyObject* o, float& out)
{
    double d;
    if (PyFloat_Check(o)) {
        d = PyFloat_AS_DOUBLE(o);
    } else if (PyLong_CheckExact(o)) {
        d = PyLong_AsDouble(o);
        if (d == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
    } else {
        return false;
    }
    out = (float)d;
    return true;
}

bool integer(PyObject* o, long long lo, long long hi, long long& out)
{
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    out = PyLong_AsLongLongAndOverflow(o, &overflow);
    return !overflow && out >= lo && out <= hi;
}

// (address of ps_adam_update, then adam_update's own arguments) -> its return code, or None
PyObject* adam_update(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    long long address, id, step;
    float lr, beta1, beta2, eps, wd, scale;
    if (n != 14 || !integer(args[0], 1, INT64_MAX, address) || !integer(args[1], INT32_MIN, INT32_MAX, id) || !integer(args[2], 0, INT64_MAX, step) ||
        !number(args[3], lr) || !number(args[4], beta1) || !number(args[5], beta2) || !number(args[6], eps) || !number(args[7], wd) ||
        !number(args[13], scale) || (args[8] != Py_True && args[8] != Py_False))
        Py_RETURN_NONE;
    const at::Tensor *p, *g, *m, *v;
    void *pp, *gp, *mp, *vp, *stream;
    int64_t numel = 0;
    int half;
    try {
        int device = -1;
        if (!plain(args[9], at::kFloat, at::kFloat, device, numel, p) || !plain(args[10], at::kFloat, at::kHalf, device, numel, g) ||
            !plain(args[11], at::kFloat, at::kFloat, device, numel, m) || !plain(args[12], at::kFloat, at::kFloat, device, numel, v) ||
            device != c10::hip::current_device())
            Py_RETURN_NONE;
        pp = p->data_ptr(), gp = g->data_ptr(), mp = m->data_ptr(), vp = v->data_ptr();
        half = g->scalar_type() == at::kHalf;
        stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream();
    } catch (...) {  // a tensor without memory of its own (vmap, meta): the general path says so
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const auto call = reinterpret_cast<decltype(&ps_adam_update)>(address);
    const int bias = args[8] == Py_True;
    int rc = 0;
    char thrown[256];  // by a call that was begun: it is an error, and not made again by the general path
    thrown[0] = 0;
    Py_BEGIN_ALLOW_THREADS  // a launch waits where the queue is full; no exception passes this block's end
    try {
        rc = call((int)id, (size_t)step, lr, beta1, beta2, eps, wd, bias, static_cast<float*>(pp), gp, half, static_cast<float*>(mp),
                  static_cast<float*>(vp), (size_t)numel, scale, nullptr, stream);
    } catch (const std::exception& e) {
        std::snprintf(thrown, sizeof(thrown), "adam_update: %s", e.what());
    } catch (...) {
        std::snprintf(thrown, sizeof(thrown), "adam_update: unknown exception");
    }
    Py_END_ALLOW_THREADS
    if (thrown[0]) {
        PyErr_SetString(PyExc_RuntimeError, thrown);
        return nullptr;
    }
    return PyLong_FromLong(rc);
}

PyMethodDef methods[] = {
    {"adam_update", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(adam_update)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, 0, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// abi_version: of the library whose ps_adam_update it calls by its address; built_for: the Python and torch it was compiled with.
PyMODINIT_FUNC PyInit__binding()
{
    PyObject* m = PyModule_Create(&module);
    if (m && (PyModule_AddIntConstant(m, "abi_version", PS_ABI_VERSION) || PyModule_AddStringConstant(m, "built_for", PS_BUILT_FOR))) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
