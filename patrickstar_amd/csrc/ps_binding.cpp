// What the host does again and again for a step, compiled: adam_update of the operator module and FP16Adam's whole-list steps from
// Python arguments to the library without Python in between, and the look at every parameter's numbers.
//
// A per-tensor loop calls the operator once for every tensor, 199 times for a BERT-base-sized module, and most of those
// tensors take the GPU less time than the call takes the host: 6.4 us a call, of which the checks of four tensors in
// Python were 1.3 and the conversion of seventeen arguments by ctypes 1.7 us.
//
// The functions here take calls of the ordinary form only: plain tensors and numbers, everything on the current device.
// Whatever else they are given they leave alone and return None; the caller then goes through its general path, which accepts or
// refuses it as always.  Nothing is kept between calls.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdio>
#include <exception>

#include <ATen/core/Tensor.h>
#include <ATen/record_function.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
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

bool number(PyObject* o, double& out)
{
    if (PyFloat_Check(o)) {
        out = PyFloat_AS_DOUBLE(o);
    } else if (PyLong_CheckExact(o)) {
        out = PyLong_AsDouble(o);
        if (out == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            return false;
        }
    } else {
        return false;
    }
    return true;
}
bool number(PyObject* o, float& out)
{
    double d;
    if (!number(o, d)) return false;
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

// The return code of a call of the library.
template <typename F>
PyObject* called(const char* what, F call)
{
    int rc = 0;
    char thrown[256];  // by a call that was begun: it is an error, and not made again by the general path
    thrown[0] = 0;
    Py_BEGIN_ALLOW_THREADS  // a launch waits where the queue is full; no exception passes this block's end
    try {
        rc = call();
    } catch (const std::exception& e) {
        std::snprintf(thrown, sizeof(thrown), "%s: %s", what, e.what());
    } catch (...) {
        std::snprintf(thrown, sizeof(thrown), "%s: unknown exception", what);
    }
    Py_END_ALLOW_THREADS
    if (thrown[0]) {
        PyErr_SetString(PyExc_RuntimeError, thrown);
        return nullptr;
    }
    return PyLong_FromLong(rc);
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
    return called("adam_update", [&] {
        return call((int)id, (size_t)step, lr, beta1, beta2, eps, wd, bias, static_cast<float*>(pp), gp, half, static_cast<float*>(mp),
                    static_cast<float*>(vp), (size_t)numel, scale, nullptr, stream);
    });
}

// ------------------------------------------------------------------------------- steps over whole chunk lists
//
// FP16Adam.step() over a list of a few chunks is bound by the host: of 13.2 us for a device-decided step, one launch, 6.1 went into
// torch's wrapper of every optimizer's step (a profiler range and hooks, which mostly nobody asked for: quiet()), 1.2 into
// torch.no_grad(), 1.3 into the conversion of 16 arguments by ctypes.

// The stream to work on if the GPU with this number is the current one.
bool current_stream(PyObject* device, void*& stream)
{
    long long d;
    if (!integer(device, 0, INT8_MAX, d)) return false;
    try {
        if (c10::hip::current_device() != d) return false;
        stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)d).stream();
    } catch (...) {
        return false;
    }
    return true;
}

// A host address as an integer; None: NULL.
template <typename T>
bool host_address(PyObject* o, T*& out)
{
    long long a = 0;
    if (o != Py_None && !integer(o, 1, INT64_MAX, a)) return false;
    out = reinterpret_cast<T*>(a);
    return true;
}

// The bytes of a plain tensor on the GPU with this number; None: NULL.
bool device_bytes(PyObject* o, PyObject* device, void*& out)
{
    out = nullptr;
    if (o == Py_None) return true;
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    try {
        if (!t.defined() || t.layout() != at::kStrided || !t.is_cuda() || !t.is_contiguous() || t.get_device() != PyLong_AsLong(device)) return false;
        out = t.data_ptr();
    } catch (...) {
        return false;
    }
    return out != nullptr;
}

struct List {
    long long id, n, numel;
    const ps_chunk* chunks;
    const size_t* used;
    const ps_call_pattern* calls;
};
bool list_of(PyObject* const* args, List& l)  // optimizer, chunks, their number, length, used lengths, call pattern
{
    return integer(args[0], INT32_MIN, INT32_MAX, l.id) && host_address(args[1], l.chunks) && integer(args[2], 0, INT32_MAX, l.n) &&
           integer(args[3], 0, INT64_MAX, l.numel) && host_address(args[4], l.used) && host_address(args[5], l.calls);
}

// (address of ps_adam_step_chunks, device, list_of's, step, lr, beta1, beta2, eps, weight decay, loss scale) -> its return code, or None
PyObject* step_chunks(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    long long address, step;
    List l;
    double lr, beta1, beta2, eps, wd, scale;
    void* stream;
    if (n != 15 || !integer(args[0], 1, INT64_MAX, address) || !list_of(args + 2, l) || !integer(args[8], 0, INT64_MAX, step) || !number(args[9], lr) ||
        !number(args[10], beta1) || !number(args[11], beta2) || !number(args[12], eps) || !number(args[13], wd) || !number(args[14], scale) ||
        !current_stream(args[1], stream))
        Py_RETURN_NONE;
    const auto call = reinterpret_cast<decltype(&ps_adam_step_chunks)>(address);
    return called("step_chunks", [&] {
        return call((int)l.id, (size_t)step, lr, beta1, beta2, eps, wd, 1, l.chunks, (int)l.n, (size_t)l.numel, l.used, l.calls, scale, stream);
    });
}

// (address of ps_adam_step_chunks_dynamic_scratch, device, list_of's, lr, eps, weight decay, probe, state, log, its capacity, operator
// calls, scratch) -> its return code, or None
PyObject* step_dynamic(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    long long address, capacity, operator_calls;
    List l;
    double lr, eps, wd;
    void *state, *log, *scratch, *stream;
    if (n != 17 || !integer(args[0], 1, INT64_MAX, address) || !list_of(args + 2, l) || !number(args[8], lr) || !number(args[9], eps) ||
        !number(args[10], wd) || (args[11] != Py_True && args[11] != Py_False) || !integer(args[14], 0, INT64_MAX, capacity) ||
        !integer(args[15], 0, INT64_MAX, operator_calls) || !current_stream(args[1], stream) || !device_bytes(args[12], args[1], state) ||
        !device_bytes(args[13], args[1], log) || !state ||
        !device_bytes(args[16], args[1], scratch))
        Py_RETURN_NONE;
    const auto call = reinterpret_cast<decltype(&ps_adam_step_chunks_dynamic_scratch)>(address);
    const int probe = args[11] == Py_True;
    return called("step_dynamic", [&] {
        return call((int)l.id, lr, eps, wd, 1, l.chunks, (int)l.n, (size_t)l.numel, l.used, l.calls, probe, static_cast<ps_step_state*>(state),
                    static_cast<ps_scale_record*>(log), capacity, operator_calls, scratch, scratch ? PS_STEP_SCRATCH_BYTES : 0, stream);
    });
}

// Whether nobody watches what is called: no callbacks of a profiler or of any other observer, no dispatch mode.
PyObject* quiet(PyObject*, PyObject*)
{
    return PyBool_FromLong(!at::hasCallbacks() && !c10::impl::dispatch_mode_enabled());
}

// ----------------------------------------------------------------------------------- every parameter's numbers

// (parameters, their requires_grad as it was) -> whether it still is
PyObject* same_flags(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    if (n != 2 || !PyList_CheckExact(args[0]) || !PyTuple_CheckExact(args[1])) Py_RETURN_NONE;
    const Py_ssize_t k = PyList_GET_SIZE(args[0]);
    if (PyTuple_GET_SIZE(args[1]) != k) Py_RETURN_FALSE;
    for (Py_ssize_t i = 0; i < k; ++i) {
        PyObject* p = PyList_GET_ITEM(args[0], i);
        if (!THPVariable_Check(p)) Py_RETURN_NONE;
        if ((PyTuple_GET_ITEM(args[1], i) == Py_True) != THPVariable_Unpack(p).requires_grad()) Py_RETURN_FALSE;
    }
    Py_RETURN_TRUE;
}

PyObject *key_lr, *key_betas, *key_eps, *key_wd;

// A NaN is none: whether two of them are the same is a question of their objects in Python.
bool ordinary(PyObject* o, double& out) { return o != nullptr && number(o, out) && out == out; }
bool entry(PyObject* state, PyObject* key, double& out) { return ordinary(PyDict_GetItemWithError(state, key), out); }

// lr, betas, eps and weight_decay out of state[p] of the parameters that `wanted` holds a true byte for, in order, into records of
// ps_tensor_call; the rest of a record is left alone.
// (parameters, state, wanted, address of the records) -> True: all the same, False: they differ, None: not of the ordinary form (some
// records may have been written).  The optimizer's own dictionary has the parameters in their order, so nothing is looked up in it.
PyObject* read_numbers(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    ps_tensor_call* record;
    if (n != 4 || !PyList_CheckExact(args[0]) || !PyDict_Check(args[1]) || !PyBytes_CheckExact(args[2]) || !host_address(args[3], record) || !record)
        Py_RETURN_NONE;
    const Py_ssize_t k = PyList_GET_SIZE(args[0]);
    if (PyBytes_GET_SIZE(args[2]) != k || PyDict_GET_SIZE(args[1]) != k) Py_RETURN_NONE;
    const char* wanted = PyBytes_AS_STRING(args[2]);
    const ps_tensor_call* first = nullptr;
    bool same = true;
    Py_ssize_t at = 0;
    PyObject *p, *state;
    for (Py_ssize_t i = 0; i < k && PyDict_Next(args[1], &at, &p, &state); ++i) {
        if (p != PyList_GET_ITEM(args[0], i) || !PyDict_Check(state)) Py_RETURN_NONE;
        if (!wanted[i]) continue;
        PyObject* betas = PyDict_GetItemWithError(state, key_betas);
        const bool tuple = betas && PyTuple_CheckExact(betas), list = betas && PyList_CheckExact(betas);
        if ((!tuple && !list) || (tuple ? PyTuple_GET_SIZE(betas) : PyList_GET_SIZE(betas)) != 2 ||
            !ordinary(tuple ? PyTuple_GET_ITEM(betas, 0) : PyList_GET_ITEM(betas, 0), record->beta1) ||
            !ordinary(tuple ? PyTuple_GET_ITEM(betas, 1) : PyList_GET_ITEM(betas, 1), record->beta2) || !entry(state, key_lr, record->lr) ||
            !entry(state, key_eps, record->eps) || !entry(state, key_wd, record->weight_decay)) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
        if (first == nullptr) first = record;
        same = same && record->lr == first->lr && record->beta1 == first->beta1 && record->beta2 == first->beta2 && record->eps == first->eps &&
               record->weight_decay == first->weight_decay;
        ++record;
    }
    return PyBool_FromLong(same);
}

// (address of the records, how many, common counter, address of every tensor's distance from it): the step numbers of a step that the
// host decides.
PyObject* write_steps(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    ps_tensor_call* record;
    long long k, common;
    const int64_t* distance;
    if (n != 4 || !host_address(args[0], record) || !integer(args[1], 0, INT32_MAX, k) || !integer(args[2], 0, INT64_MAX, common) ||
        !host_address(args[3], distance) || ((!record || !distance) && k > 0)) {
        PyErr_SetString(PyExc_TypeError, "write_steps(records, n, common, distances)");
        return nullptr;
    }
    for (long long i = 0; i < k; ++i) record[i].step = common + distance[i];
    Py_RETURN_NONE;
}

PyCFunction fast(PyObject* (*f)(PyObject*, PyObject* const*, Py_ssize_t)) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }
PyMethodDef methods[] = {
    {"adam_update", fast(adam_update), METH_FASTCALL, nullptr},   {"step_chunks", fast(step_chunks), METH_FASTCALL, nullptr},
    {"step_dynamic", fast(step_dynamic), METH_FASTCALL, nullptr}, {"quiet", quiet, METH_NOARGS, nullptr},
    {"same_flags", fast(same_flags), METH_FASTCALL, nullptr},     {"read_numbers", fast(read_numbers), METH_FASTCALL, nullptr},
    {"write_steps", fast(write_steps), METH_FASTCALL, nullptr},   {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, 0, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// abi_version: of the library whose ps_adam_update it calls by its address; built_for: the Python and torch it was compiled with.
PyMODINIT_FUNC PyInit__binding()
{
    key_lr = PyUnicode_InternFromString("lr"), key_betas = PyUnicode_InternFromString("betas");
    key_eps = PyUnicode_InternFromString("eps"), key_wd = PyUnicode_InternFromString("weight_decay");
    if (!key_lr || !key_betas || !key_eps || !key_wd) return nullptr;
    PyObject* m = PyModule_Create(&module);
    if (m && (PyModule_AddIntConstant(m, "abi_version", PS_ABI_VERSION) || PyModule_AddStringConstant(m, "built_for", PS_BUILT_FOR))) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
