// The calls of the Python binding that a serving loop makes for every layer, as a CPython extension: phase 1 of the matmuls and the
// quantizers from Tensor objects, and phase 2.  Bound to the entry points' addresses in the library that ctypes has loaded, so that
// there is one copy of the library in the process; the GIL is released around the library, as ctypes does.
//
// Why: ctypes converts every argument through a Python-level protocol, which took longer than the launches.  Quantizer and
// matmul of 8 rows: host time 12.2 us a pass with ctypes, 8.5 here, of which two launches take 4.8.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>

#include "acl/acl.h"
#include "aclnnop/aclnn_dynamic_block_quant.h"
#include "aclnnop/aclnn_dynamic_mx_quant.h"
#include "aclnnop/aclnn_dynamic_quant.h"
#include "aclnnop/aclnn_quant_matmul_v5.h"
#include "aclnnop/aclnn_quant_matmul_weight_nz.h"
#include "aclnnop/aclnn_weight_quant_batch_matmul_v2.h"

namespace {

PyObject* g_handle;   // interned attribute name

// Of every argument only the plain form is taken here -- None, an int, a float, bytes, a Tensor whose handle is one of the first two --, with
// the value that ctypes makes of it.  Anything else is left to ctypes, which knows what each parameter accepts: a phase 1 function then
// returns NotImplemented, phase 2 calls the ctypes function itself.  The readers below return false for that, without a Python error.

// None or an int, of which the low bits count.
bool as_pointer(PyObject* o, void** out)
{
    if (o == Py_None) { *out = nullptr; return true; }
    if (!PyLong_Check(o)) return false;
    *out = (void*)(uintptr_t)PyLong_AsUnsignedLongLongMask(o);
    return true;
}
bool as_int64(PyObject* o, int64_t* out)
{
    if (!PyLong_Check(o)) return false;
    *out = (int64_t)PyLong_AsUnsignedLongLongMask(o);
    return true;
}
bool as_double(PyObject* o, double* out)
{
    if (!PyFloat_Check(o)) return false;
    *out = PyFloat_AS_DOUBLE(o);
    return true;
}
bool as_flag(PyObject* o, bool* out)
{
    *out = o == Py_True;
    return PyBool_Check(o);
}
// (lives as long as the argument)
bool as_text(PyObject* o, const char** out)
{
    if (o == Py_None) { *out = nullptr; return true; }
    if (!PyBytes_Check(o)) return false;
    *out = PyBytes_AS_STRING(o);
    return true;
}
bool tensors(PyObject* const* args, int n, const aclTensor** t)
{
    for (int i = 0; i < n; i++) {
        t[i] = nullptr;
        if (args[i] == Py_None) continue;
        PyObject* h = PyObject_GetAttr(args[i], g_handle);
        if (!h) { PyErr_Clear(); return false; }
        void* p = nullptr;
        const bool ok = as_pointer(h, &p);
        Py_DECREF(h);
        if (!ok) return false;
        t[i] = (const aclTensor*)p;
    }
    return true;
}
PyObject* phase1_result(aclnnStatus rc, uint64_t ws, const aclOpExecutor* ex)
{
    PyObject *r = PyLong_FromLong((long)rc), *w = PyLong_FromUnsignedLongLong(ws), *e = ex ? PyLong_FromVoidPtr((void*)ex) : Py_None;
    if (e == Py_None) Py_INCREF(e);
    PyObject* t = r && w && e ? PyTuple_New(3) : nullptr;
    if (!t) { Py_XDECREF(r); Py_XDECREF(w); Py_XDECREF(e); return nullptr; }
    PyTuple_SET_ITEM(t, 0, r); PyTuple_SET_ITEM(t, 1, w); PyTuple_SET_ITEM(t, 2, e);
    return t;
}

// The entry points, by address (bind).
struct Entry {
    decltype(&aclnnQuantMatmulV5GetWorkspaceSize) qmm;
    decltype(&aclnnQuantMatmulWeightNzGetWorkspaceSize) qmm_nz;
    decltype(&aclnnWeightQuantBatchMatmulV2GetWorkspaceSize) wqmm;
    decltype(&aclnnDynamicQuantGetWorkspaceSize) dynamic_quant;
    decltype(&aclnnDynamicBlockQuantGetWorkspaceSize) block_quant;
    decltype(&aclnnDynamicMxQuantGetWorkspaceSize) mx_quant;
} g_entry;

// bind(six addresses in the order of Entry)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    void* p[6];
    bool ok = n == 6;
    for (int i = 0; ok && i < 6; i++) ok = as_pointer(args[i], &p[i]) && p[i];
    if (!ok) {
        PyErr_SetString(PyExc_TypeError, "six addresses are wanted");
        return nullptr;
    }
    g_entry.qmm = (decltype(g_entry.qmm))p[0];
    g_entry.qmm_nz = (decltype(g_entry.qmm_nz))p[1];
    g_entry.wqmm = (decltype(g_entry.wqmm))p[2];
    g_entry.dynamic_quant = (decltype(g_entry.dynamic_quant))p[3];
    g_entry.block_quant = (decltype(g_entry.block_quant))p[4];
    g_entry.mx_quant = (decltype(g_entry.mx_quant))p[5];
    Py_RETURN_NONE;
}

// qmm(x1, x2, x1_scale, x2_scale, y_scale, x1_offset, x2_offset, y_offset, bias, out, transpose_x1, transpose_x2, group_size, ws, ex, nz)
PyObject* qmm(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    const aclTensor* t[10];
    bool ta, tb, want_ws, want_ex, nz;
    int64_t group;
    if (n != 16 || !tensors(args, 10, t) || !as_flag(args[10], &ta) || !as_flag(args[11], &tb) || !as_int64(args[12], &group) ||
        !as_flag(args[13], &want_ws) || !as_flag(args[14], &want_ex) || !as_flag(args[15], &nz)) Py_RETURN_NOTIMPLEMENTED;
    uint64_t ws = 0;
    aclOpExecutor* ex = nullptr;
    aclnnStatus rc;
    Py_BEGIN_ALLOW_THREADS
    rc = (nz ? g_entry.qmm_nz : g_entry.qmm)(t[0], t[1], t[2], t[3], t[4], t[5], t[6], t[7], t[8], ta, tb, group, const_cast<aclTensor*>(t[9]),
                                             want_ws ? &ws : nullptr, want_ex ? &ex : nullptr);
    Py_END_ALLOW_THREADS
    return phase1_result(rc, ws, ex);
}
// wqmm(x, weight, scale, offset, quant_scale, quant_offset, bias, y, group_size)
PyObject* wqmm(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    const aclTensor* t[8];
    int64_t group;
    if (n != 9 || !tensors(args, 8, t) || !as_int64(args[8], &group)) Py_RETURN_NOTIMPLEMENTED;
    uint64_t ws = 0;
    aclOpExecutor* ex = nullptr;
    aclnnStatus rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_entry.wqmm(t[0], t[1], t[2], t[3], t[4], t[5], t[6], (int)group, t[7], &ws, &ex);
    Py_END_ALLOW_THREADS
    return phase1_result(rc, ws, ex);
}
// dynamic_quant(x, smooth, y, scale)
PyObject* dynamic_quant(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    const aclTensor* t[4];
    if (n != 4 || !tensors(args, 4, t)) Py_RETURN_NOTIMPLEMENTED;
    uint64_t ws = 0;
    aclOpExecutor* ex = nullptr;
    aclnnStatus rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_entry.dynamic_quant(t[0], t[1], t[2], t[3], &ws, &ex);
    Py_END_ALLOW_THREADS
    return phase1_result(rc, ws, ex);
}
// block_quant(x, y, scale, min_scale, round_mode, dst_type, row_block, col_block)
PyObject* block_quant(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    const aclTensor* t[3];
    const char* mode;
    double min_scale;
    int64_t v[3];
    if (n != 8 || !tensors(args, 3, t) || !as_double(args[3], &min_scale) || !as_text(args[4], &mode)) Py_RETURN_NOTIMPLEMENTED;
    for (int i = 0; i < 3; i++)
        if (!as_int64(args[5 + i], &v[i])) Py_RETURN_NOTIMPLEMENTED;
    uint64_t ws = 0;
    aclOpExecutor* ex = nullptr;
    aclnnStatus rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_entry.block_quant(t[0], min_scale, const_cast<char*>(mode), v[0], v[1], v[2], t[1], t[2], &ws, &ex);
    Py_END_ALLOW_THREADS
    return phase1_result(rc, ws, ex);
}
// mx_quant(x, y, scale, axis, round_mode, dst_type, blocksize, scale_alg)
PyObject* mx_quant(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    const aclTensor* t[3];
    const char* mode;
    int64_t axis, v[3];
    if (n != 8 || !tensors(args, 3, t) || !as_int64(args[3], &axis) || !as_text(args[4], &mode)) Py_RETURN_NOTIMPLEMENTED;
    for (int i = 0; i < 3; i++)
        if (!as_int64(args[5 + i], &v[i])) Py_RETURN_NOTIMPLEMENTED;
    uint64_t ws = 0;
    aclOpExecutor* ex = nullptr;
    aclnnStatus rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_entry.mx_quant(t[0], axis, const_cast<char*>(mode), v[0], v[1], v[2], t[1], t[2], &ws, &ex);
    Py_END_ALLOW_THREADS
    return phase1_result(rc, ws, ex);
}

// phase2(address, function of ctypes) -> f(workspace, size, executor, stream), the status.
typedef aclnnStatus (*Phase2)(void*, uint64_t, aclOpExecutor*, aclrtStream);
PyObject* run_phase2(PyObject* self, PyObject* const* args, Py_ssize_t n)
{
    void *address, *ws, *ex, *stream;
    int64_t size = 0;
    if (n != 4 || !as_pointer(PyTuple_GET_ITEM(self, 0), &address) || !as_pointer(args[0], &ws) || !as_int64(args[1], &size) ||
        !as_pointer(args[2], &ex) || !as_pointer(args[3], &stream)) return PyObject_Vectorcall(PyTuple_GET_ITEM(self, 1), args, (size_t)n, nullptr);
    aclnnStatus rc;
    Py_BEGIN_ALLOW_THREADS
    rc = ((Phase2)address)(ws, (uint64_t)size, (aclOpExecutor*)ex, (aclrtStream)stream);
    Py_END_ALLOW_THREADS
    return PyLong_FromLong((long)rc);
}
PyMethodDef g_phase2 = {"phase2", (PyCFunction)(void (*)(void))run_phase2, METH_FASTCALL, "(workspace, size, executor, stream) -> status"};
PyObject* phase2(PyObject*, PyObject* const* args, Py_ssize_t n)
{
    if (n != 2) {
        PyErr_SetString(PyExc_TypeError, "an address and a function are wanted");
        return nullptr;
    }
    PyObject* self = PyTuple_Pack(2, args[0], args[1]);
    PyObject* f = self ? PyCFunction_New(&g_phase2, self) : nullptr;
    Py_XDECREF(self);
    return f;
}

#define FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {FAST(bind), FAST(qmm), FAST(wqmm), FAST(dynamic_quant), FAST(block_quant), FAST(mx_quant), FAST(phase2), {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "opsnn_calls", "per-call entry points of the binding", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_opsnn_calls()
{
    g_handle = PyUnicode_InternFromString("handle");
    return g_handle ? PyModule_Create(&g_module) : nullptr;
}
