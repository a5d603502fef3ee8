// Segment tables from lists of tensors, as a CPython module.
//
// A unit's gradients or views are many small tensors, and their checks in
// Python (type, device, layout, address, size) took 0.7 us each: 61 tensors
// cost 49 us a call, the kernel that moves them 9.5.  Here they are read from
// the tensors directly.
//
// Only what needs no further thought is taken: plain torch.Tensor or
// Parameter objects on a GPU, strided, contiguous, of the types expected.
// For anything else the functions return None and the caller's own checks
// decide, so what is refused, and with which error, is written in one place.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <stdint.h>
#include <string.h>

#include "../../include/slidefsdp.h"

namespace {

enum Kind { kB16 = 0, kF32 = 1, kBf16 = 2 };

bool type_ok(at::ScalarType t, Kind kind) {
    switch (kind) {
        case kF32: return t == at::kFloat;
        case kBf16: return t == at::kBFloat16;
        default: return t == at::kBFloat16 || t == at::kHalf || t == at::kShort || t == at::kUInt16;
    }
}

// Address and size of a plain tensor; false if it is anything else.
bool plain(PyObject* o, Kind kind, uint64_t* ptr, uint64_t* n) {
    if (!THPVariable_CheckExact(o)) return false;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || !type_ok(t.scalar_type(), kind)) return false;
    // transforms (vmap, functionalisation) wrap tensors without an address of their own
    if (!t.has_storage() || t.unsafeGetTensorImpl()->key_set().has_any(c10::DispatchKeySet(
            {c10::DispatchKey::Python, c10::DispatchKey::Functionalize, c10::DispatchKey::FuncTorchBatched,
             c10::DispatchKey::FuncTorchGradWrapper})))
        return false;
    if (!t.is_contiguous()) return false;
    *ptr = reinterpret_cast<uint64_t>(t.data_ptr());
    *n = uint64_t(t.numel());
    return true;
}

void put(PyObject* table, Py_ssize_t i, uint64_t src, uint64_t dst, uint64_t n) {
    const sf_seg s = {src, dst, n};
    memcpy(PyBytes_AS_STRING(table) + i * Py_ssize_t(sizeof(s)), &s, sizeof(s));
}

// list_table(tensors, as_dst): (table, count, elements) of 16-bit tensors,
// their addresses as the segments' destinations or sources, or None.
PyObject* list_table(PyObject*, PyObject* args) {
    PyObject* arg;
    int as_dst;
    if (!PyArg_ParseTuple(args, "Op", &arg, &as_dst)) return nullptr;
    if (!PyList_CheckExact(arg) && !PyTuple_CheckExact(arg)) Py_RETURN_NONE;
    const Py_ssize_t k = PySequence_Fast_GET_SIZE(arg);
    PyObject* table = PyBytes_FromStringAndSize(nullptr, k * Py_ssize_t(sizeof(sf_seg)));
    if (table == nullptr) return nullptr;
    uint64_t total = 0;
    try {
        for (Py_ssize_t i = 0; i < k; ++i) {
            uint64_t ptr, n;
            if (!plain(PySequence_Fast_GET_ITEM(arg, i), kB16, &ptr, &n)) {
                Py_DECREF(table);
                Py_RETURN_NONE;
            }
            put(table, i, as_dst ? 0 : ptr, as_dst ? ptr : 0, n);
            total += n;
        }
    } catch (...) {   // a tensor without an address: the caller reports it
        Py_DECREF(table);
        Py_RETURN_NONE;
    }
    return Py_BuildValue("NnK", table, k, static_cast<unsigned long long>(total));
}

// pair_table(pairs, cast): (table, count) of (src, dst) tensors of equal size,
// float32 to bfloat16 or both 16-bit, or None.
PyObject* pair_table(PyObject*, PyObject* args) {
    PyObject* arg;
    int cast;
    if (!PyArg_ParseTuple(args, "Op", &arg, &cast)) return nullptr;
    if (!PyList_CheckExact(arg) && !PyTuple_CheckExact(arg)) Py_RETURN_NONE;
    const Py_ssize_t k = PySequence_Fast_GET_SIZE(arg);
    PyObject* table = PyBytes_FromStringAndSize(nullptr, k * Py_ssize_t(sizeof(sf_seg)));
    if (table == nullptr) return nullptr;
    try {
        for (Py_ssize_t i = 0; i < k; ++i) {
            PyObject* pair = PySequence_Fast_GET_ITEM(arg, i);
            uint64_t src, dst, n, m;
            if ((!PyTuple_CheckExact(pair) && !PyList_CheckExact(pair)) || PySequence_Fast_GET_SIZE(pair) != 2 ||
                !plain(PySequence_Fast_GET_ITEM(pair, 0), cast ? kF32 : kB16, &src, &n) ||
                !plain(PySequence_Fast_GET_ITEM(pair, 1), cast ? kBf16 : kB16, &dst, &m) || n != m) {
                Py_DECREF(table);
                Py_RETURN_NONE;
            }
            put(table, i, src, dst, n);
        }
    } catch (...) {   // a tensor without an address: the caller reports it
        Py_DECREF(table);
        Py_RETURN_NONE;
    }
    return Py_BuildValue("Nn", table, k);
}

PyMethodDef methods[] = {
    {"list_table", list_table, METH_VARARGS, "Segment table of 16-bit GPU tensors, or None."},
    {"pair_table", pair_table, METH_VARARGS, "Segment table of (src, dst) GPU tensors, or None."},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_sf_segs", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__sf_segs(void) {
    PyObject* m = PyModule_Create(&module);
    // the layout of the tensors read here is this torch's alone
    if (m != nullptr && PyModule_AddStringConstant(m, "TORCH_VERSION", SF_TORCH_VERSION) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
