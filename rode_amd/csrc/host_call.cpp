// Host side of the Python ops, natively: the calls that a program makes once per product
// (rode_sddmm, rode_spmm, attention and its gradient), and what a new matrix needs (row statistics, decomposition).
//
// A small matrix takes a few microseconds on the GPU, so its calls are bound by what the host
// does around the launch: argument checks, an allocation and the launch itself cost 10-11 us
// through ctypes, 5 us here.  The functions take the ordinary case only - plain float32 or
// float16 tensors on the current GPU, contiguous, nothing to differentiate - and return None
// for every other one, which the Python layer then handles (or refuses with its own message).
//
// (The kernels' boundary stays the C ABI of include/rode_hip.h: no torch type crosses it.)
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <ATen/ops/zeros.h>
#include <c10/core/GradMode.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <cstdint>
#include <string>

#include "../../include/rode_hip.h"

namespace {

// Every function's body is in a try: what torch throws - no memory, no data behind a tensor, a Python error of a dispatch
// mode - becomes the Python exception it stands for.  (Not HANDLE_TH_ERRORS, which also collects warnings: 0.1 us a call.)
PyObject* raised()
{
    torch::translate_exception_to_python(std::current_exception());
    return nullptr;
}

// Without the interpreter's lock, until the end of the scope however it is left.
struct NoGil {
    PyThreadState* state = PyEval_SaveThread();
    NoGil() = default;
    NoGil(const NoGil&) = delete;
    ~NoGil() { PyEval_RestoreThread(state); }
};

// The tensor behind a Python object if its elements are in memory as its sizes and strides say, else null: not one of
// another layout (sparse), not a wrapper (vmap, jvp, functionalization), not one with a dispatch of its own (fake
// tensors) and no lazy negation or zero.
const at::Tensor* strided_of(PyObject* o)
{
    using K = c10::DispatchKey;
    static const c10::DispatchKeySet wrapped({K::Python, K::Functionalize, K::FuncTorchBatched, K::FuncTorchGradWrapper, K::Batched, K::Negative,
                                              K::Conjugate, K::ZeroTensor});
    if (!THPVariable_Check(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || t.layout() != at::kStrided || !t.has_storage() || t.unsafeGetTensorImpl()->key_set().has_any(wrapped)) return nullptr;
    return &t;
}

// The same, or null for anything but a tensor or parameter itself: a subclass may mean something else by the call.
const at::Tensor* tensor_of(PyObject* o) { return THPVariable_CheckExact(o) ? strided_of(o) : nullptr; }

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

// The memory of a tensor.  (What a dispatch mode made of an allocation of ours may have none.)
void* data(const at::Tensor& t)
{
    void* p = t.data_ptr();
    TORCH_CHECK(p != nullptr || t.numel() == 0, "a tensor without data");
    return p;
}
const int* ints(const at::Tensor* t) { return static_cast<const int*>(data(*t)); }
const float* floats(const at::Tensor* t) { return static_cast<const float*>(data(*t)); }
float* floats(const at::Tensor& t) { return static_cast<float*>(data(t)); }

bool wants_grad(const at::Tensor& t) { return t.requires_grad(); }

PyObject* failed(const char* what, int code)
{
    return PyErr_Format(PyExc_RuntimeError, "%s failed: %s (hipError %d)", what, rode_hip_error_string(code), code);
}

// sddmm(<matrix>, k, lhs, rhs, plans address, stream) -> out or None
PyObject* sddmm(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    try {
    Matrix a;
    long long k, plans, stream;
    if (count != 15 || !matrix_of(args, a) || !int_of(args[10], k) || !int_of(args[13], plans) || !int_of(args[14], stream)) Py_RETURN_NONE;
    const at::Tensor *lhs = tensor_of(args[11]), *rhs = tensor_of(args[12]);
    const int kind = dense_kind(a, lhs, a.m);
    if (kind < 0 || dense_kind(a, rhs, a.n) != kind || lhs->size(1) != k || rhs->size(1) != k) Py_RETURN_NONE;
    if (k <= 0 || k > 512 || k % (kind == RODE_DENSE_F16 ? 8 : 4) != 0) Py_RETURN_NONE;
    if (c10::GradMode::is_enabled() && (wants_grad(*lhs) || wants_grad(*rhs) || wants_grad(*a.val))) Py_RETURN_NONE;
    const at::Tensor out = at::empty({a.val->size(0)}, a.val->options().requires_grad(false));
    const int *block = ints(a.block), *residue = ints(a.residue), *start = ints(a.start), *row_ptr = ints(a.row_ptr), *col = ints(a.col);
    const float* val = floats(a.val);
    float* o = floats(out);
    const void *l = data(*lhs), *r = data(*rhs);
    int code;
    {
        NoGil no_gil;
        void* s = reinterpret_cast<void*>(stream);
        code = rode_hip_sddmm_planned(kind, 0, (int)a.m1, (int)a.m2, (int)a.n, (int)k, block, residue, start, row_ptr, col, val, l, r, o,
                                      reinterpret_cast<const rode_hip_plans*>(plans), s, s);
    }
    if (code != 0) return failed("rode_hip_sddmm_planned", code);
    return THPVariable_Wrap(out);
    } catch (...) {
        return raised();
    }
}

// spmm(<matrix>, dense, plans address, every row stored, stream[, longest row in aligned slots]) -> C or None
PyObject* spmm(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    try {
    Matrix a;
    long long plans, stored, stream, longest = 0;
    if ((count != 14 && count != 15) || !matrix_of(args, a) || !int_of(args[11], plans) || !int_of(args[12], stored) || !int_of(args[13], stream) ||
        (count == 15 && (!int_of(args[14], longest) || longest < 0 || longest > INT32_MAX)))
        Py_RETURN_NONE;
    const at::Tensor* dense = tensor_of(args[10]);
    const int kind = dense_kind(a, dense, a.n);
    if (kind < 0) Py_RETURN_NONE;
    const long long width = dense->size(1);
    if (width <= 0 || width > 0x7fffffff || width % (kind == RODE_DENSE_F16 ? 8 : 4) != 0) Py_RETURN_NONE;
    if (c10::GradMode::is_enabled() && (wants_grad(*dense) || wants_grad(*a.val))) Py_RETURN_NONE;
    const at::Tensor out = at::empty({(int64_t)a.m, (int64_t)width}, a.val->options().requires_grad(false));
    const int *block = ints(a.block), *residue = ints(a.residue), *start = ints(a.start), *row_ptr = ints(a.row_ptr), *col = ints(a.col);
    const float* val = floats(a.val);
    const void* b = data(*dense);
    float* c = floats(out);
    const rode_hip_plans* p = reinterpret_cast<const rode_hip_plans*>(plans);
    // A hub plan's partial rows are this call's own (the allocator orders their next use on the stream): calls on one matrix
    // may overlap on other streams, and those of other threads come between two kernels of this one.
    rode_hip_plans own;
    at::Tensor scratch;
    if (p && p->hub && !p->hub_workspace) {
        own = *p, p = &own;
        own.hub_workspace_bytes = rode_hip_hub_workspace_bytes(own.hub_counts, (int)width, 4);
        scratch = at::empty({(int64_t)own.hub_workspace_bytes}, a.val->options().dtype(at::kByte).requires_grad(false));
        own.hub_workspace = data(scratch);
    }
    int code = 0;
    const char* what = stored ? "rode_hip_spmm_planned" : "rode_hip_spmm_new";
    {
        NoGil no_gil;
        void* s = reinterpret_cast<void*>(stream);
        if (stored)
            code = rode_hip_spmm_planned(kind, RODE_SPMM_WHOLE_LISTS | RODE_SPMM_OVERWRITE, (int)a.m1, (int)a.m2, (int)a.n, (int)width, val, col,
                                         row_ptr, block, residue, start, b, c, p, s, s);
        else // (some rows are added to, or in no list)
            code = rode_hip_spmm_new(kind, (int)a.m, (int)longest, (int)a.m1, (int)a.m2, (int)a.n, (int)width,
                                     val, col, row_ptr, block, residue, start, b, c, p, s);
    }
    if (code != 0) return failed(what, code);
    return THPVariable_Wrap(out);
    } catch (...) {
        return raised();
    }
}

// ---- attention -----------------------------------------------------------------------------
struct Pattern {
    const at::Tensor *row_ptr, *col, *val;
    int device;
};

// args: row_offsets, column_indices, values
bool pattern_of(PyObject* const* args, Pattern& a)
{
    a.row_ptr = tensor_of(args[0]), a.col = tensor_of(args[1]), a.val = tensor_of(args[2]);
    if (!a.row_ptr || !a.col || !a.val || !a.val->is_cuda() || a.val->scalar_type() != at::kFloat || !a.val->is_contiguous()) return false;
    if (a.val->numel() == 0) return false;
    a.device = a.val->device().index();
    int current = -1;
    return hipGetDevice(&current) == hipSuccess && current == a.device;
}

bool dense_like(const Pattern& a, const at::Tensor* t, at::ScalarType type, long long heads, int dims, long long rows, long long d)
{
    return t && t->is_cuda() && t->device().index() == a.device && t->scalar_type() == type && t->is_contiguous() && t->dim() == dims &&
           (dims == 2 || t->size(0) == heads) && t->size(dims - 2) == rows && t->size(dims - 1) == d;
}

// What q, k and v have in common, if they are ordinary.
struct Heads {
    int kind = -1, dims = 0;
    long long heads = 1, m = 0, n = 0, d = 0;
};
bool heads_of(const Pattern& a, const at::Tensor* q, const at::Tensor* k, const at::Tensor* v, Heads& h)
{
    if (!q || !k || !v || (q->dim() != 2 && q->dim() != 3) || k->dim() != q->dim()) return false;
    h.dims = (int)q->dim();
    h.heads = h.dims == 3 ? q->size(0) : 1;
    h.m = q->size(h.dims - 2), h.n = k->size(h.dims - 2), h.d = q->size(h.dims - 1);
    h.kind = q->scalar_type() == at::kFloat ? RODE_DENSE_F32 : q->scalar_type() == at::kHalf ? RODE_DENSE_F16 : -1;
    const at::ScalarType type = q->scalar_type();
    return h.kind >= 0 && h.m == a.row_ptr->numel() - 1 && h.heads > 0 && dense_like(a, q, type, h.heads, h.dims, h.m, h.d) &&
           dense_like(a, k, type, h.heads, h.dims, h.n, h.d) && dense_like(a, v, type, h.heads, h.dims, h.n, h.d);
}

bool float_of(PyObject* o, double& v)
{
    v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

// attention(<pattern>, q, k, v, scale, keep scores, plans address, stream) -> (out, scores or None, stats or None), or None
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    try {
    Pattern a;
    Heads h;
    long long keep, plans, stream;
    double scale;
    if (count != 10 || !pattern_of(args, a) || !float_of(args[6], scale) || !int_of(args[7], keep) || !int_of(args[8], plans) ||
        !int_of(args[9], stream))
        Py_RETURN_NONE;
    const at::Tensor *q = tensor_of(args[3]), *k = tensor_of(args[4]), *v = tensor_of(args[5]);
    if (!heads_of(a, q, k, v, h)) Py_RETURN_NONE;
    at::Tensor out, scores, stats;
    const long long nnz = a.val->numel();
    const auto f32 = a.val->options().requires_grad(false);
    out = at::empty(q->sizes(), f32);
    if (keep) {
        scores = h.dims == 3 ? at::empty({h.heads, nnz}, f32) : at::empty({nnz}, f32);
        stats = h.dims == 3 ? at::empty({h.heads, h.m, 2}, f32) : at::empty({h.m, 2}, f32);
    }
    const int *row_ptr = ints(a.row_ptr), *col = ints(a.col);
    const float* val = floats(a.val);
    const void *qp = data(*q), *kp = data(*k), *vp = data(*v);
    float *o = floats(out), *kept = keep ? floats(scores) : nullptr, *row_stats = keep ? floats(stats) : nullptr;
    int code;
    {
        NoGil no_gil;
        code = rode_hip_attention_forward_batched(h.kind, (int)h.heads, (int)h.m, (int)h.n, (int)nnz, (int)h.d, row_ptr, col, val, qp, kp, vp,
                                                  (float)scale, o, kept, row_stats, reinterpret_cast<const rode_hip_plans*>(plans),
                                                  reinterpret_cast<void*>(stream));
    }
    if (code != 0) return failed("rode_hip_attention_forward_batched", code);
    if (!keep) return Py_BuildValue("(NOO)", THPVariable_Wrap(std::move(out)), Py_None, Py_None);
    return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(out)), THPVariable_Wrap(std::move(scores)), THPVariable_Wrap(std::move(stats)));
    } catch (...) {
        return raised();
    }
}

// attention_backward(<pattern>, row_offsets_t, column_indices_t, slots_t, scores, stats or None, grad, out, q, k, v, scale, plans address,
// plans address of the transposed pattern, stream) -> (dq, dk, dv) in float32, or None
PyObject* attention_backward(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    try {
    Pattern a;
    Heads h;
    long long plans, plans_t, stream;
    double scale;
    if (count != 17 || !pattern_of(args, a) || !float_of(args[13], scale) || !int_of(args[14], plans) || !int_of(args[15], plans_t) ||
        !int_of(args[16], stream))
        Py_RETURN_NONE;
    const at::Tensor *t_row_ptr = tensor_of(args[3]), *t_col = tensor_of(args[4]), *t_slot = tensor_of(args[5]), *scores = tensor_of(args[6]);
    const at::Tensor *stats = args[7] == Py_None ? nullptr : tensor_of(args[7]), *g = tensor_of(args[8]), *out = tensor_of(args[9]);
    const at::Tensor *q = tensor_of(args[10]), *k = tensor_of(args[11]), *v = tensor_of(args[12]);
    if (!t_row_ptr || !t_col || !t_slot || !scores || (args[7] != Py_None && !stats) || !heads_of(a, q, k, v, h)) Py_RETURN_NONE;
    if (!dense_like(a, g, at::kFloat, h.heads, h.dims, h.m, h.d) || !dense_like(a, out, at::kFloat, h.heads, h.dims, h.m, h.d)) Py_RETURN_NONE;
    const long long nnz = a.val->numel();
    if (t_slot->numel() != nnz || t_row_ptr->numel() != h.n + 1 || scores->numel() != h.heads * nnz) Py_RETURN_NONE;
    const auto f32 = a.val->options().requires_grad(false);
    at::Tensor dq = at::empty(q->sizes(), f32), dk = at::empty(k->sizes(), f32), dv = at::empty(v->sizes(), f32);
    const at::Tensor pairs = at::empty({2 * h.heads * nnz}, f32);
    const int *row_ptr = ints(a.row_ptr), *col = ints(a.col), *rows_t = ints(t_row_ptr), *col_t = ints(t_col), *slot = ints(t_slot);
    const float *val = floats(a.val), *kept = floats(scores), *row_stats = stats ? floats(stats) : nullptr, *grad = floats(g), *o = floats(out);
    const void *qp = data(*q), *kp = data(*k), *vp = data(*v);
    float *pz = floats(pairs), *dqp = floats(dq), *dkp = floats(dk), *dvp = floats(dv);
    int code;
    const char* what = "rode_hip_attention_backward_rows";
    {
        NoGil no_gil;
        void* s = reinterpret_cast<void*>(stream);
        code = rode_hip_attention_backward_rows(h.kind, (int)h.heads, (int)h.m, (int)h.n, (int)nnz, (int)h.d, row_ptr, col, val, kept, row_stats, grad,
                                                o, kp, vp, (float)scale, slot, dqp, pz, reinterpret_cast<const rode_hip_plans*>(plans), s);
        if (code == 0) {
            what = "rode_hip_attention_backward_cols";
            code = rode_hip_attention_backward_cols(h.kind, (int)h.heads, (int)h.m, (int)h.n, (int)nnz, (int)h.d, rows_t, col_t, pz, grad, qp, dkp, dvp,
                                                    reinterpret_cast<const rode_hip_plans*>(plans_t), s);
        }
    }
    if (code != 0) return failed(what, code);
    return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(dq)), THPVariable_Wrap(std::move(dk)), THPVariable_Wrap(std::move(dv)));
    } catch (...) {
        return raised();
    }
}

// ---- a new matrix ------------------------------------------------------------------------
// What RoDeCSR asks of the row offsets, in one pass (a dozen vector instructions per eight
// rows; as a chain of tensor operations it takes 0.3 - 1 ms for 65 K rows, mostly waking threads).
struct RowStats {
    long long max_len = 0;                             // longest row
    long long shortest = INT64_MAX, longest = INT64_MIN; // ... counted in aligned slots (a row from its start & ~3)
    long long blocked = 0;                             // rows with block segments (32 aligned slots or more)
    long long segments_512 = 0;                        // segments of 512 slots that those rows have
    long long up_to_512 = 0, up_to_1024 = 0;           // those of at most that many slots
    long long hub_nonzeros = 0;                        // nonzeros of the rows of hub_min_len aligned slots or more
};

// (sums of a block in the offsets' own type: they cannot pass the last offset)
template <typename T>
__attribute__((target_clones("avx512f", "avx2", "default"))) void row_stats_block(const T* ro, long long rows, T hub_min_len, RowStats& r)
{
    T max_len = 0, shortest = r.shortest > INT32_MAX ? (T)INT32_MAX : (T)r.shortest, longest = INT32_MIN;
    T blocked = 0, segments = 0, up_to_512 = 0, up_to_1024 = 0, hub = 0;
    for (long long i = 0; i < rows; ++i) {
        const T len = ro[i + 1] - ro[i], aligned = len + (ro[i] & 3);
        const T is_blocked = aligned >= 32 ? 1 : 0, is_hub = aligned >= hub_min_len ? -1 : 0; // (a mask)
        max_len = len > max_len ? len : max_len;
        shortest = aligned < shortest ? aligned : shortest;
        longest = aligned > longest ? aligned : longest;
        blocked += is_blocked;
        segments += is_blocked * ((aligned + 511) >> 9);
        up_to_512 += is_blocked & (aligned <= 512 ? 1 : 0);
        up_to_1024 += is_blocked & (aligned <= 1024 ? 1 : 0);
        hub += len & is_hub;
    }
    r.max_len = std::max<long long>(r.max_len, max_len);
    r.shortest = std::min<long long>(r.shortest, shortest);
    r.longest = std::max<long long>(r.longest, longest);
    r.blocked += blocked, r.segments_512 += segments, r.up_to_512 += up_to_512, r.up_to_1024 += up_to_1024;
    r.hub_nonzeros += hub;
}

RowStats stats_of(const at::Tensor& ro, long long hub_min_len)
{
    const long long rows = ro.size(0) - 1;
    const void* offsets = data(ro);
    const bool is_int = ro.scalar_type() == at::kInt;
    RowStats r;
    constexpr long long kBlock = 1 << 16; // (a block's sums are added up in 64 bits)
    for (long long at = 0; at < rows; at += kBlock) {
        const long long n = std::min(kBlock, rows - at);
        if (is_int)
            row_stats_block<int32_t>(static_cast<const int32_t*>(offsets) + at, n, (int32_t)std::min<long long>(hub_min_len, INT32_MAX), r);
        else
            row_stats_block<int64_t>(static_cast<const int64_t*>(offsets) + at, n, hub_min_len, r);
    }
    if (rows <= 0) r.shortest = r.longest = 0;
    return r;
}

PyObject* built(const RowStats& r)
{
    return Py_BuildValue("(LLLLLLLL)", r.max_len, r.shortest, r.longest, r.blocked, r.segments_512, r.up_to_512, r.up_to_1024, r.hub_nonzeros);
}

// row_stats(row offsets on the CPU, int32 or int64; hub_min_len) -> the fields of RowStats
PyObject* row_stats(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    try {
    const at::Tensor* ro = count == 2 ? strided_of(args[0]) : nullptr;
    long long hub_min_len;
    if (!ro || !int_of(args[1], hub_min_len) || !ro->is_cpu() || ro->dim() != 1 || !ro->is_contiguous() ||
        (ro->scalar_type() != at::kInt && ro->scalar_type() != at::kLong))
        return PyErr_Format(PyExc_ValueError, "row_stats takes a contiguous int32 or int64 vector on the CPU and an int");
    RowStats r;
    {
        NoGil no_gil;
        r = stats_of(*ro, hub_min_len);
    }
    return built(r);
    } catch (...) {
        return raised();
    }
}

// How many block segments and residue rows the decomposition has (k_block 32, vec_len 4): the
// closed form per row that the GPU's decompose_kernel uses (rode_preprocess.hip, row_counts).
__attribute__((target_clones("avx512f", "avx2", "default"))) void list_sizes_shift(const int32_t* ro, long long rows, int shift, long long& n_blk, long long& n_res)
{
    int32_t blk = 0, res = 0; // (both totals are below 2^31)
    for (long long i = 0; i < rows; ++i) {
        const int32_t n = ro[i + 1] - ro[i] + (ro[i] & 3);
        const int32_t some = n > 0 ? 1 : 0;
        const int32_t t = (n - some) >> shift, rest = n - (int32_t)((uint32_t)t << shift);
        blk += some * (t + (rest >= 32 ? 1 : 0));
        res += some & ((rest & 31) != 0 ? 1 : 0);
    }
    n_blk = blk, n_res = res;
}

void list_sizes(const int32_t* ro, long long rows, int seg, long long& n_blk, long long& n_res)
{
    if ((seg & (seg - 1)) == 0) return list_sizes_shift(ro, rows, __builtin_ctz(seg), n_blk, n_res);
    n_blk = n_res = 0;
    for (long long i = 0; i < rows; ++i) {
        const int32_t n = ro[i + 1] - ro[i] + (ro[i] & 3);
        if (n <= 0) continue;
        const int32_t t = (n - 1) / seg, rest = n - t * seg;
        n_blk += t + (rest >= 32 ? 1 : 0);
        n_res += (rest & 31) != 0 ? 1 : 0;
    }
}

// A stream that memory of the scope is in use on: waited for at its end, however it is left.
struct Waited {
    hipStream_t stream;
    bool used = false;
    int wait()
    {
        used = false;
        return hipStreamSynchronize(stream);
    }
    ~Waited()
    {
        if (used) (void)hipStreamSynchronize(stream);
    }
};

// send_offsets(row offsets on the CPU, memory for them on the GPU, hub_min_len, stream) -> what row_stats says of them: the copy is queued
// first and runs while they are counted here and by decompose (65 K rows: 17 us on its own).  The caller keeps both until the stream has
// been waited for, as decompose does.
PyObject* send_offsets(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    try {
    const at::Tensor *host = count == 4 ? strided_of(args[0]) : nullptr, *dev = host ? strided_of(args[1]) : nullptr;
    long long hub_min_len, stream;
    if (!dev || !int_of(args[2], hub_min_len) || !int_of(args[3], stream) || !host->is_cpu() || !dev->is_cuda() || host->scalar_type() != at::kInt ||
        dev->scalar_type() != at::kInt || host->dim() != 1 || dev->dim() != 1 || host->size(0) < 1 || host->size(0) != dev->size(0) ||
        !host->is_contiguous() || !dev->is_contiguous())
        return PyErr_Format(PyExc_ValueError, "send_offsets takes int32 row offsets on the CPU and memory for them on the GPU");
    RowStats r;
    int code;
    {
        NoGil no_gil;
        code = hipMemcpyAsync(data(*dev), data(*host), (size_t)host->size(0) * sizeof(int), hipMemcpyHostToDevice, reinterpret_cast<hipStream_t>(stream));
        r = stats_of(*host, hub_min_len);
    }
    return code != 0 ? failed("hipMemcpyAsync", code) : built(r);
    } catch (...) {
        return raised();
    }
}

// decompose(row offsets on the CPU, the same on the GPU, columns or None, dense rows, segment
// length, stream[, upload]) -> (block_indices, st_offsets, residue_indices, m1, m2, plan, counts): the row
// decomposition and, with the columns given, the descriptors of a locality plan (tensor and its
// four counts; else None, None).  The list lengths are counted here, so that the lists are
// allocated at their size and everything is queued at once: one wait for the whole of it
// instead of one for the counts, one for the plan and a copy of every list.  With `upload`, the offsets on the GPU are still to be
// filled: their copy runs while the lists are counted here (65 K rows: 17 us on its own, hidden but for the 5 us of starting it); `upload`
// None: send_offsets has queued it.  Either way the GPU's offsets are the host's, and the lists are placed by what is counted here, tile by tile.
PyObject* decompose(PyObject*, PyObject* const* args, Py_ssize_t count)
{
    try {
    long long dense_rows, seg, stream;
    if ((count != 6 && count != 7) || !int_of(args[3], dense_rows) || !int_of(args[4], seg) || !int_of(args[5], stream))
        return PyErr_Format(PyExc_ValueError, "decompose takes 6 or 7 arguments");
    const bool upload = count == 7 && args[6] == Py_True, same = upload || (count == 7 && args[6] == Py_None);
    const at::Tensor *host = strided_of(args[0]), *dev = strided_of(args[1]), *col = args[2] == Py_None ? nullptr : strided_of(args[2]);
    if (!host || !dev || !host->is_cpu() || !dev->is_cuda() || host->scalar_type() != at::kInt || dev->scalar_type() != at::kInt ||
        host->dim() != 1 || dev->dim() != 1 || host->size(0) < 1 || host->size(0) != dev->size(0) || !host->is_contiguous() ||
        !dev->is_contiguous() || seg <= 0 || seg > INT32_MAX || (args[2] != Py_None && (!col || !col->is_cuda() || col->scalar_type() != at::kInt)))
        return PyErr_Format(PyExc_ValueError, "decompose takes int32 row offsets on the CPU and on the GPU");
    const long long m = dev->size(0) - 1;
    at::Tensor blk, start, res, plan, scratch, counts;
    long long m1 = 0, m2 = 0;
    int code = 0;
    const char* what = "rode_hip_preprocess";
    std::string error;
    {
        NoGil no_gil;
        hipStream_t s = reinterpret_cast<hipStream_t>(stream);
        Waited queued{s}; // (also when an allocation below fails)
        queued.used = same;
        if (upload) {
            what = "hipMemcpyAsync";
            code = hipMemcpyAsync(data(*dev), data(*host), (size_t)(m + 1) * sizeof(int), hipMemcpyHostToDevice, s);
        }
        const int32_t* offsets = static_cast<const int32_t*>(data(*host));
        const long long tile = same && m > 0 ? rode_hip_preprocess_tile_rows((int)m) : 0, tiles = tile > 0 ? (m + tile - 1) / tile : 0;
        // (pinned: the kernels read what lies before every tile and write the counts where the host reads them)
        const long long chunks_most = tiles > 0 && col && rode_hip_preprocess_plan_too((int)m) ? (m + 127) / 128 : 0;
        counts = at::empty({8 + 2 * tiles + 3 * chunks_most}, at::TensorOptions().dtype(at::kInt).pinned_memory(true));
        int* h = static_cast<int*>(data(counts));
        unsigned long long* before = reinterpret_cast<unsigned long long*>(h + 8);
        unsigned long long* places = before + tiles;
        int* has_window = reinterpret_cast<int*>(places + chunks_most);
        long long most_tiles = 0; // that the residue rows of a chunk lie in, with those between
        if (tiles > 0) {
            long long chunk = 0, begins = 0, last = 0; // (tiles: of the chunk before, the last one with a residue row)
            for (long long t = 0; t < tiles; ++t) {
                long long b, r;
                before[t] = (unsigned long long)m1 << 32 | (unsigned long long)m2;
                list_sizes(offsets + t * tile, std::min(tile, m - t * tile), (int)seg, b, r);
                for (; chunk < chunks_most && 128 * chunk < m2 + r; ++chunk) {
                    places[chunk] = (unsigned long long)t << 32 | (unsigned long long)(128 * chunk - m2);
                    if (chunk > 0) most_tiles = std::max(most_tiles, (128 * chunk > m2 ? t : last) - begins + 1);
                    begins = t;
                }
                if (r > 0) last = t;
                m1 += b, m2 += r;
            }
            most_tiles = std::max(most_tiles, last - begins + 1);
        } else {
            list_sizes(offsets, m, (int)seg, m1, m2);
        }
        blk = m1 > 0 ? at::empty({m1}, dev->options()) : at::zeros({1}, dev->options()); // (an empty list has one place that is never read)
        start = at::empty({m1 + 1}, dev->options());
        res = m2 > 0 ? at::empty({m2}, dev->options()) : at::zeros({1}, dev->options());
        const size_t ws_bytes = tiles > 0 ? 0 : rode_hip_preprocess_workspace_bytes((int)m);
        if (tiles == 0) scratch = at::empty({(int64_t)((ws_bytes + 7) / 8)}, dev->options().dtype(at::kLong));
        size_t plan_bytes = 0;
        if (col && m2 > 0) {
            plan_bytes = rode_hip_window_plan_bytes((int)m2);
            plan = at::empty({(int64_t)(plan_bytes / 4)}, dev->options());
        }
        int *segments = static_cast<int*>(data(blk)), *starts = static_cast<int*>(data(start));
        int* rows = static_cast<int*>(data(res));
        h[0] = h[1] = -1;
        const int *rp = static_cast<const int*>(data(*dev)), *columns = plan_bytes ? static_cast<const int*>(data(*col)) : nullptr;
        void *work = tiles > 0 ? nullptr : data(scratch), *windows = plan_bytes ? data(plan) : nullptr;
        // From here to the end of the wait nothing throws: what is queued uses the memory above.
        queued.used = true;
        // List and plan at once: where at least every second row is a residue row, and no chunk's workgroup - it goes through the rows from its
        // first residue row to its last, 2 us for 1024 - has so many to go through that the two launches are sooner done: a sixteenth of all.
        // (us of a build, so many empty rows in the middle: at once / two launches, 65 K rows of 21: 2048 61, 4096 64 / 68, 8192 73 / 67, 32 768 120 / 65;
        // 131 K: 8192 91 / 93, 16 384 107 / 92; 262 K: 16 384 141 / 147, 32 768 173 / 145; 400 K: 16 384 185 / 193, 32 768 214 / 192, 200 000 515 / 173.)
        const long long walk_rows = std::min(std::max(m / 16, 1024ll), 16384ll);
        const bool at_once = chunks_most > 0 && plan_bytes > 0 && 2 * m2 >= m && most_tiles * tile <= walk_rows;
        if (code == 0 && tiles > 0) {
            what = "rode_hip_preprocess_placed";
            code = rode_hip_preprocess_placed((int)seg, (int)m, rp, segments, starts, rows, h, (int)m1, (int)m2, before, (int)dense_rows, columns, windows,
                                              plan_bytes, at_once ? places : nullptr, has_window, s);
        } else if (code == 0 && plan_bytes) {
            what = "rode_hip_preprocess_with_plan";
            code = rode_hip_preprocess_with_plan((int)seg, (int)m, rp, segments, starts, rows, h, (int)m1, work, ws_bytes, (int)m2, (int)dense_rows, columns,
                                                 windows, plan_bytes, s);
        } else if (code == 0) {
            what = "rode_hip_preprocess";
            code = rode_hip_preprocess((int)seg, 32, 4, (int)m, rp, segments, starts, rows, h, h + 1, (int)m1, work, ws_bytes, s);
        }
        const int waited = queued.wait(); // (also after an error: the scratch is in use until then)
        if (code == 0) code = waited;
        if (code == 0 && at_once) {
            h[4] = (int)((m2 + 127) / 128), h[5] = h[6] = h[7] = 0;
            for (int c = 0; c < h[4]; ++c) h[5] += has_window[c] != 0;
            if (h[5] > 0) {
                what = "rode_hip_window_plan_count";
                code = rode_hip_window_plan_count((int)m2, h[5], windows, plan_bytes, s);
            }
        }
        if (code == 0 && (h[0] != m1 || h[1] != m2)) error = "the row decomposition on the GPU does not have the expected size";
    }
    if (!error.empty()) return PyErr_Format(PyExc_RuntimeError, "%s", error.c_str());
    if (code != 0) return failed(what, code);
    const int* h = static_cast<const int*>(data(counts));
    PyObject* plan_counts = plan.defined() ? Py_BuildValue("[iiii]", h[4], h[5], h[6], h[7]) : Py_BuildValue("");
    PyObject* plan_data = plan.defined() ? THPVariable_Wrap(std::move(plan)) : Py_BuildValue("");
    return Py_BuildValue("(NNNLLNN)", THPVariable_Wrap(std::move(blk)), THPVariable_Wrap(std::move(start)), THPVariable_Wrap(std::move(res)),
                         m1, m2, plan_data, plan_counts);
    } catch (...) {
        return raised();
    }
}

PyMethodDef methods[] = {
    {"row_stats", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(row_stats)), METH_FASTCALL,
     "row_stats(row_offsets, hub_min_len) -> (max_len, shortest, longest, blocked, segments_512, up_to_512, up_to_1024, hub_nonzeros)"},
    {"send_offsets", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(send_offsets)), METH_FASTCALL,
     "send_offsets(row_offsets_cpu, row_offsets, hub_min_len, stream) -> row_stats(row_offsets_cpu, hub_min_len), the copy to the GPU queued"},
    {"decompose", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(decompose)), METH_FASTCALL,
     "decompose(row_offsets_cpu, row_offsets, columns or None, dense_rows, seg_length, stream[, upload]) -> (block, start, residue, m1, m2, plan, counts)"},
    {"sddmm", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(sddmm)), METH_FASTCALL,
     "sddmm(block, residue, start, m1, m2, row_offsets, columns, values, m, n, k, lhs, rhs, plans, stream) -> tensor or None"},
    {"spmm", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(spmm)), METH_FASTCALL,
     "spmm(block, residue, start, m1, m2, row_offsets, columns, values, m, n, dense, plans, stored, stream[, longest]) -> tensor or None"},
    {"attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(attention)), METH_FASTCALL,
     "attention(row_offsets, columns, values, q, k, v, scale, keep, plans, stream) -> (out, scores, stats) or None"},
    {"attention_backward", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(attention_backward)), METH_FASTCALL,
     "attention_backward(row_offsets, columns, values, row_offsets_t, columns_t, slots_t, scores, stats, grad, out, q, k, v, scale, plans, "
     "plans_t, stream) -> (dq, dk, dv) or None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__host_call() { return PyModule_Create(&module); }
