// Host side of the Python ops, natively: the calls that a program makes once per product
// (rode_sddmm, rode_spmm), and the pass over the row offsets that a new matrix needs.
//
// A small matrix takes a few microseconds on the GPU, so its calls are bound by what the host
// does around the launch: argument checks, an allocation and the launch itself cost 10-11 us
// through ctypes, 3-4 us here.  The functions take the ordinary case only - plain float32 or
// float16 tensors on the current GPU, contiguous, nothing to differentiate - and return None
// for every other one, which the Python layer then handles (or refuses with its own message).
//
// (The kernels' boundary stays the C ABI of include/rode_hip.h: no torch type crosses it.)
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/GradMode.h>
#include <torch/csrc/autograd/python_variable.h>

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdint>

#include "../../include/rode_hip.h"

namespace {

// The tensor behind a Python object, or null for anything but a plain tensor or parameter.
const at::Tensor* tensor_of(PyObject* o)
{
    return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr;
}

bool int_of(PyObject* o, long long& v)
{
    v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

struct Matrix {
    const at::Tensor *block, *residue, *start, *row_ptr, *col, *val;
    long long m1, m2, m, n;
    int device;
};

// args: block_indices, residue_indices, st_offsets, m1, m2, row_offsets, column_indices, values, m, n
bool matrix_of(PyObject* const* args, Matrix& a)
{
    a.block = tensor_of(args[0]), a.residue = tensor_of(args[1]), a.start = tensor_of(args[2]);
    a.row_ptr = tensor_of(args[5]), a.col = tensor_of(args[6]), a.val = tensor_of(args[7]);
    if (!a.block || !a.residue || !a.start || !a.row_ptr || !a.col || !a.val) return false;
    if (!int_of(args[3], a.m1) || !int_of(args[4], a.m2) || !int_of(args[8], a.m) || !int_of(args[9], a.n)) return false;
    if (a.m1 + a.m2 <= 0 || !a.val->is_cuda() || a.val->scalar_type() != at::kFloat || !a.val->is_contiguous()) return false;
    a.device = a.val->device().index();
    int current = -1;
    return hipGetDevice(&current) == hipSuccess && current == a.device;
}

// A dense operand as the kernels read it; 0 / 1: RODE_DENSE_F32 / _F16, -1: not one of the ordinary ones.
int dense_kind(const Matrix& a, const at::Tensor* t, long long rows)
{
    if (!t || !t->is_cuda() || t->device().index() != a.device || t->dim() != 2 || t->size(0) != rows || !t->is_contiguous()) return -1;
    return t->scalar_type() == at::kFloat ? RODE_DENSE_F32 : t->scalar_type() == at::kHalf ? RODE_DENSE_F16 : -1;
}

bool wants_grad(const at::Tensor& t) { return t.requires_grad(); }

PyObject* failed(const char* what, int code)
{
    return PyErr_Format(PyExc_RuntimeError, "%s failed: %s (hipError %d)", what, rode_hip_error_string(code), code);
}

// sddmm(<matrix>, k, lhs, rhs, plans address, stream) -> out or None
PyObject* sddmm(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    Matrix a;
    long long k, plans, stream;
    if (count != 15 || !matrix_of(args, a) || !int_of(args[10], k) || !int_of(args[13], plans) || !int_of(args[14], stream)) Py_RETURN_NONE;
    const at::Tensor *lhs = tensor_of(args[11]), *rhs = tensor_of(args[12]);
    const int kind = dense_kind(a, lhs, a.m);
    if (kind < 0 || dense_kind(a, rhs, a.n) != kind || lhs->size(1) != k || rhs->size(1) != k) Py_RETURN_NONE;
    if (k <= 0 || k > 512 || k % (kind == RODE_DENSE_F16 ? 8 : 4) != 0) Py_RETURN_NONE;
    if (c10::GradMode::is_enabled() && (wants_grad(*lhs) || wants_grad(*rhs) || wants_grad(*a.val))) Py_RETURN_NONE;
    at::Tensor out;
    try {
        out = at::empty({a.val->size(0)}, a.val->options().requires_grad(false));
    } catch (const std::exception& e) {
        return PyErr_Format(PyExc_RuntimeError, "%s", e.what());
    }
    int code;
    void* s = reinterpret_cast<void*>(stream);
    Py_BEGIN_ALLOW_THREADS
    code = rode_hip_sddmm_planned(kind, 0, (int)a.m1, (int)a.m2, (int)a.n, (int)k, static_cast<const int*>(a.block->data_ptr()),
                                  static_cast<const int*>(a.residue->data_ptr()), static_cast<const int*>(a.start->data_ptr()),
                                  static_cast<const int*>(a.row_ptr->data_ptr()), static_cast<const int*>(a.col->data_ptr()),
                                  static_cast<const float*>(a.val->data_ptr()), lhs->data_ptr(), rhs->data_ptr(),
                                  static_cast<float*>(out.data_ptr()), reinterpret_cast<const rode_hip_plans*>(plans), s, s);
    Py_END_ALLOW_THREADS
    if (code != 0) return failed("rode_hip_sddmm_planned", code);
    return THPVariable_Wrap(std::move(out));
}

// spmm(<matrix>, dense, plans address, every row stored, stream) -> C or None
PyObject* spmm(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    Matrix a;
    long long plans, stored, stream;
    if (count != 14 || !matrix_of(args, a) || !int_of(args[11], plans) || !int_of(args[12], stored) || !int_of(args[13], stream)) Py_RETURN_NONE;
    const at::Tensor* dense = tensor_of(args[10]);
    const int kind = dense_kind(a, dense, a.n);
    if (kind < 0) Py_RETURN_NONE;
    const long long width = dense->size(1);
    if (width <= 0 || width > 0x7fffffff || width % (kind == RODE_DENSE_F16 ? 8 : 4) != 0) Py_RETURN_NONE;
    if (c10::GradMode::is_enabled() && (wants_grad(*dense) || wants_grad(*a.val))) Py_RETURN_NONE;
    at::Tensor out;
    try {
        out = at::empty({(int64_t)a.m, (int64_t)width}, a.val->options().requires_grad(false));
    } catch (const std::exception& e) {
        return PyErr_Format(PyExc_RuntimeError, "%s", e.what());
    }
    int code = 0;
    const char* what = "rode_hip_spmm_clear_rows";
    void* s = reinterpret_cast<void*>(stream);
    Py_BEGIN_ALLOW_THREADS
    const int* row_ptr = static_cast<const int*>(a.row_ptr->data_ptr());
    // (only the rows that the kernels add to, or skip, need clearing)
    if (!stored) code = rode_hip_spmm_clear_rows((int)a.m, (int)width, 4, row_ptr, out.data_ptr(), s);
    if (code == 0) {
        what = "rode_hip_spmm_planned";
        code = rode_hip_spmm_planned(kind, RODE_SPMM_WHOLE_LISTS | (stored ? RODE_SPMM_OVERWRITE : 0), (int)a.m1, (int)a.m2, (int)a.n,
                                     (int)width, a.val->data_ptr(), static_cast<const int*>(a.col->data_ptr()), row_ptr,
                                     static_cast<const int*>(a.block->data_ptr()), static_cast<const int*>(a.residue->data_ptr()),
                                     static_cast<const int*>(a.start->data_ptr()), dense->data_ptr(), out.data_ptr(),
                                     reinterpret_cast<const rode_hip_plans*>(plans), s, s);
    }
    Py_END_ALLOW_THREADS
    if (code != 0) return failed(what, code);
    return THPVariable_Wrap(std::move(out));
}

PyMethodDef methods[] = {
    {"sddmm", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(sddmm)), METH_FASTCALL,
     "sddmm(block, residue, start, m1, m2, row_offsets, columns, values, m, n, k, lhs, rhs, plans, stream) -> tensor or None"},
    {"spmm", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(spmm)), METH_FASTCALL,
     "spmm(block, residue, start, m1, m2, row_offsets, columns, values, m, n, dense, plans, stored, stream) -> tensor or None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__host_call() { return PyModule_Create(&module); }
