// _fo_hostscan: the per-step host work of the optimizers over tensor objects: the check of a cached multi-tensor launch
// plan as one C++ loop, the step counters, and the checks in front of a single-tensor launch.
//
// Before a cached plan may be launched again, step() has to see that every parameter still owns the storage the
// launch table points at and where its gradient lives now (torch frees and reallocates gradients every iteration).
// In Python that is four attribute reads or calls per parameter, 0.25 us each: 0.9 ms for a list of 4096 tensors,
// during which the device idles at the head of every burst of steps.  This module does the same walk over the
// at::Tensor objects directly (20 ns per parameter).  It is host-side bookkeeping only: no device code, no math; the
// package falls back to the Python loop when the module has not been built (flashoptim_amd/base.py).
//
// same_objects(a, b) -> bool
//   whether the two lists hold the very same objects in the same order (the group's parameter list against the one the
//   plan was built for).
// scan(params, table_address, table_entries) -> None | tuple of (index, new_gradient_address)
//   params         list of the bucket's parameters, in table order
//   table_address  address of the bucket's fo_tensor_desc array (host copy, include/flashoptim_hip.h)
//   table_entries  its length; a list of another length is an error (ValueError)
//   None: some parameter has no gradient, does not require one, moved to other storage, or its gradient changed
//         dtype, device, size or contiguity -- the caller takes the full planning path.  Otherwise the gradients
//         that now live at another address than the table says (empty tuple: the table is current).
//         A tensor object that libtorch cannot answer these questions for (a wrapper subclass without storage)
//         also gives None.
// counters(state, params, views, pool) -> None | float
//   whether state[p]["step"] still is views[i] for every parameter of the list, and all elements of `pool` (the CPU fp32
//   tensor the views look into) agree: their common value, else None.  (A Python loop over the lookups costs 75 ns per
//   parameter, more than the scan; this one 15.)
// advance(counter) -> None | float
//   counter += 1 on a CPU fp32 tensor and its new (first) value, without a dispatcher call (0.1 instead of 1.8 us); None,
//   and nothing changed, for any other kind of tensor.
// step_args(param, grad, errors, mom, mom_scales, var, var_scales, quantized) -> None | tuple
//   what a single-tensor step entry point takes: the addresses of mom, mom_scales, var, var_scales, param, grad, errors, then
//   elements, dtype code and bytes per error (flashoptim_amd/kernels.py: _step_args); None where one of the conditions its
//   Python checks raise for does not hold.  errors, and var with its scales, may be None.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>

namespace {

struct TensorDesc {  // fo_tensor_desc
    void* param;
    const void* grad;
    void* ecc;
    void* mom;
    void* mom_scales;
    void* var;
    void* var_scales;
    int64_t n;
};
static_assert(sizeof(TensorDesc) == 64, "layout of fo_tensor_desc");

PyObject* scan(PyObject*, PyObject* args) {
    PyObject* params = nullptr;
    unsigned long long address = 0;
    Py_ssize_t entries = 0;
    if (!PyArg_ParseTuple(args, "OKn", &params, &address, &entries)) return nullptr;
    if (!PyList_CheckExact(params)) {
        PyErr_SetString(PyExc_TypeError, "scan(params, table_address, table_entries): params must be a list");
        return nullptr;
    }
    const TensorDesc* table = reinterpret_cast<const TensorDesc*>(static_cast<uintptr_t>(address));
    const Py_ssize_t n = PyList_GET_SIZE(params);
    if (n != entries || (n > 0 && table == nullptr)) {
        PyErr_SetString(PyExc_ValueError, "scan: the parameter list and the launch table differ in length");
        return nullptr;
    }
    PyObject* moved = nullptr;
    try {
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* obj = PyList_GET_ITEM(params, i);
        bool ok = THPVariable_Check(obj);
        if (ok) {
            const at::Tensor& p = THPVariable_Unpack(obj);
            ok = p.defined() && p.requires_grad() && p.is_leaf();
            if (ok) {
                const at::Tensor& g = p.grad();
                ok = g.defined() && p.data_ptr() == table[i].param;
                if (ok) {
                    const void* ptr = g.data_ptr();
                    if (ptr != table[i].grad) {
                        ok = g.scalar_type() == p.scalar_type() && g.device() == p.device() && g.is_contiguous() &&
                             g.numel() == p.numel() && g.layout() == c10::kStrided;
                        if (ok) {
                            if (!moved) moved = PyList_New(0);
                            PyObject* item = moved ? Py_BuildValue("(nK)", i, (unsigned long long)(uintptr_t)ptr) : nullptr;
                            if (!item || PyList_Append(moved, item) != 0) {
                                Py_XDECREF(item);
                                Py_XDECREF(moved);
                                return nullptr;
                            }
                            Py_DECREF(item);
                        }
                    }
                }
            }
        }
        if (!ok) {
            Py_XDECREF(moved);
            Py_RETURN_NONE;
        }
    }
    } catch (...) {  // libtorch refused a query (e.g. data_ptr() of a tensor without storage): not a plan this walk can vouch for
        Py_XDECREF(moved);
        Py_RETURN_NONE;
    }
    if (!moved) return PyTuple_New(0);
    PyObject* out = PyList_AsTuple(moved);
    Py_DECREF(moved);
    return out;
}

PyObject* same_objects(PyObject*, PyObject* args) {
    PyObject *a = nullptr, *b = nullptr;
    if (!PyArg_ParseTuple(args, "OO", &a, &b)) return nullptr;
    if (!PyList_CheckExact(a) || !PyList_CheckExact(b)) {
        PyErr_SetString(PyExc_TypeError, "same_objects(a, b): both arguments must be lists");
        return nullptr;
    }
    const Py_ssize_t n = PyList_GET_SIZE(a);
    if (n != PyList_GET_SIZE(b)) Py_RETURN_FALSE;
    for (Py_ssize_t i = 0; i < n; ++i)
        if (PyList_GET_ITEM(a, i) != PyList_GET_ITEM(b, i)) Py_RETURN_FALSE;
    Py_RETURN_TRUE;
}

// dict[key] as a borrowed reference (nullptr: absent, or an error that is cleared).  A tensor's hash is its id(), evaluated
// by a Python function; `by_address` says that the caller has seen this hold for a key of the same type.  The lookup that
// takes a known hash is in CPython's headers up to 3.12.
PyObject* find(PyObject* dict, PyObject* key, bool by_address) {
#if PY_VERSION_HEX < 0x030d0000
    const Py_hash_t hash = by_address ? (Py_hash_t)(uintptr_t)key : PyObject_Hash(key);
    PyObject* value = hash == -1 ? nullptr : _PyDict_GetItem_KnownHash(dict, key, hash);
#else
    (void)by_address;
    PyObject* value = PyDict_GetItemWithError(dict, key);
#endif
    if (!value) PyErr_Clear();
    return value;
}

bool is_cpu_float(PyObject* obj) {
    if (!THPVariable_CheckExact(obj)) return false;
    const at::Tensor& t = THPVariable_Unpack(obj);
    return t.defined() && t.layout() == c10::kStrided && t.device().is_cpu() && t.scalar_type() == at::kFloat &&
           t.is_contiguous() && !t.requires_grad();
}

PyObject* counters(PyObject*, PyObject* args) {
    PyObject *state, *params, *views, *pool;
    if (!PyArg_ParseTuple(args, "OOOO", &state, &params, &views, &pool)) return nullptr;
    // a dict whose lookup is the built-in one (collections.defaultdict among them)
    const bool plain_lookup = PyDict_Check(state) && Py_TYPE(state)->tp_as_mapping->mp_subscript == PyDict_Type.tp_as_mapping->mp_subscript;
    if (!plain_lookup || !PyList_CheckExact(params) || !PyList_CheckExact(views)) Py_RETURN_NONE;
    const Py_ssize_t n = PyList_GET_SIZE(params);
    if (n == 0 || PyList_GET_SIZE(views) != n) Py_RETURN_NONE;
    static PyObject* const step = PyUnicode_InternFromString("step");
    PyObject* const first = PyList_GET_ITEM(params, 0);
    const Py_hash_t hash = PyObject_Hash(first);
    if (hash == -1) PyErr_Clear();
    const bool by_address = hash == (Py_hash_t)(uintptr_t)first;
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject* key = PyList_GET_ITEM(params, i);
        PyObject* entry = find(state, key, by_address && Py_TYPE(key) == Py_TYPE(first));
        if (!entry || !PyDict_CheckExact(entry)) Py_RETURN_NONE;
        PyObject* counter = PyDict_GetItemWithError(entry, step);
        if (!counter) PyErr_Clear();
        if (counter != PyList_GET_ITEM(views, i)) Py_RETURN_NONE;
    }
    try {
        if (!is_cpu_float(pool)) Py_RETURN_NONE;
        const at::Tensor& t = THPVariable_Unpack(pool);
        if (t.numel() != n) Py_RETURN_NONE;
        const float* v = t.const_data_ptr<float>();
        for (Py_ssize_t i = 0; i < n; ++i)
            if (!(v[i] == v[0])) Py_RETURN_NONE;
        return PyFloat_FromDouble(v[0]);
    } catch (...) {
        Py_RETURN_NONE;
    }
}

PyObject* advance(PyObject*, PyObject* obj) {
    try {
        if (!is_cpu_float(obj)) Py_RETURN_NONE;
        const at::Tensor& t = THPVariable_Unpack(obj);
        const int64_t n = t.numel();
        if (n == 0 || t.is_inference()) Py_RETURN_NONE;
        float* v = t.mutable_data_ptr<float>();
        t.unsafeGetTensorImpl()->bump_version();
        for (int64_t i = 0; i < n; ++i) v[i] += 1.0f;
        return PyFloat_FromDouble(v[0]);
    } catch (...) {
        Py_RETURN_NONE;
    }
}

// The state's tensor as the kernels take it: `n` elements, contiguous, on `device`.
bool flat_on(const at::Tensor& t, int64_t n, c10::Device device) {
    return t.defined() && t.layout() == c10::kStrided && t.numel() == n && t.is_contiguous() && t.device() == device;
}

PyObject* step_args(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 8) {
        PyErr_SetString(PyExc_TypeError, "step_args takes 8 arguments");
        return nullptr;
    }
    const at::Tensor* t[7];
    for (int i = 0; i < 7; ++i) {
        t[i] = nullptr;
        if (args[i] == Py_None) continue;
        if (!THPVariable_CheckExact(args[i])) Py_RETURN_NONE;
        t[i] = &THPVariable_Unpack(args[i]);
    }
    const int quantized = PyObject_IsTrue(args[7]);
    if (quantized < 0) return nullptr;
    const at::Tensor *param = t[0], *grad = t[1], *errors = t[2];
    if (!param || !grad) Py_RETURN_NONE;
    try {
        const int64_t n = param->numel();
        const c10::Device device = param->device();
        const at::ScalarType type = param->scalar_type();
        const int dtype = type == at::kFloat ? 0 : type == at::kBFloat16 ? 1 : type == at::kHalf ? 2 : -1;  // fo_dtype
        if (dtype < 0 || !device.is_cuda() || !flat_on(*param, n, device) || !flat_on(*grad, n, device) || grad->scalar_type() != type)
            Py_RETURN_NONE;
        int ecc_bytes = 0;
        if (errors) {
            ecc_bytes = (int)errors->element_size();
            if ((ecc_bytes != 1 && ecc_bytes != 2) || !flat_on(*errors, n, device)) Py_RETURN_NONE;
        }
        unsigned long long address[7] = {0, 0, 0, 0, 0, 0, 0};
        for (int i = 0; i < 2; ++i) {  // mom, var
            const at::Tensor *state = t[3 + 2 * i], *scales = t[4 + 2 * i];
            if (!state) continue;
            if (!flat_on(*state, n, device) || state->scalar_type() != (!quantized ? type : i == 0 ? at::kChar : at::kByte)) Py_RETURN_NONE;
            address[2 * i] = (unsigned long long)(uintptr_t)state->data_ptr();
            if (!quantized) continue;
            if (!scales || scales->scalar_type() != at::kHalf || scales->numel() < (n + 31) / 32 ||
                !flat_on(*scales, scales->numel(), device))
                Py_RETURN_NONE;
            address[2 * i + 1] = (unsigned long long)(uintptr_t)scales->data_ptr();
        }
        address[4] = (unsigned long long)(uintptr_t)param->data_ptr();
        address[5] = (unsigned long long)(uintptr_t)grad->data_ptr();
        if (errors) address[6] = (unsigned long long)(uintptr_t)errors->data_ptr();
        return Py_BuildValue("(KKKKKKKLii)", address[0], address[1], address[2], address[3], address[4], address[5], address[6],
                             (long long)n, dtype, ecc_bytes);
    } catch (...) {  // libtorch refused a query: the Python checks say what is wrong
        Py_RETURN_NONE;
    }
}

PyMethodDef methods[] = {
    {"counters", counters, METH_VARARGS, "counters(state, params, views, pool) -> None | float"},
    {"advance", advance, METH_O, "advance(counter) -> None | float"},
    {"step_args", (PyCFunction)(void (*)(void))step_args, METH_FASTCALL,
     "step_args(param, grad, errors, mom, mom_scales, var, var_scales, quantized) -> None | tuple"},
    {"same_objects", same_objects, METH_VARARGS, "same_objects(a, b) -> bool: the same objects in the same order"},
    {"scan", scan, METH_VARARGS, "scan(params, table_address, table_entries) -> None | tuple of (index, gradient address)"},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_fo_hostscan", "per-step validation of cached launch plans", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fo_hostscan(void) { return PyModule_Create(&module); }
