// The calls a program makes every step, from Python to the C ABI without ctypes: checks the tensors, takes their
// addresses and the current stream, calls the library.  Every function returns the library's status, or -1 when an
// argument is not the ordinary one (a raw address, a tensor of another type, a layout or placement the operator does not
// take, no tensor at all): ops.py then goes its own way, which takes the unusual arguments and words the errors.
//
// What it is for: a small SpMM takes 2.4 us on the GPU and 3.3 us of launch in the HIP runtime; the same call took 6.0 us
// on the host with ctypes (a Python check per operand, 0.24 us each, the current stream 0.34 us, the conversion of eleven
// arguments 0.6 us), and 15 to 29 us for the attention layer, whose checks index every operand.
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/vsparse.h"

namespace {

constexpr long kUnusual = -1;

// Reads positional arguments in order; the first unusual one clears `ok` and everything after it reads as zero.
struct Reader {
    PyObject *const *args;
    Py_ssize_t left;
    bool ok = true;

    Reader(PyObject *const *a, Py_ssize_t n) : args(a), left(n) {}

    PyObject *next()
    {
        if (!ok || left <= 0) {
            ok = false;
            return nullptr;
        }
        --left;
        return *args++;
    }
    const at::Tensor *tensor()
    {
        PyObject *o = next();
        if (!o || !THPVariable_Check(o)) {
            ok = false;
            return nullptr;
        }
        const at::Tensor &t = THPVariable_Unpack(o);
        if (!t.is_cuda() || t.layout() != at::kStrided) {
            ok = false;
            return nullptr;
        }
        return &t;
    }
    int integer()
    {
        PyObject *o = next();
        if (!o || !PyLong_CheckExact(o)) {
            ok = false;
            return 0;
        }
        int overflow = 0;
        const long v = PyLong_AsLongAndOverflow(o, &overflow);
        if (overflow || v < INT32_MIN || v > INT32_MAX) ok = false;
        return (int)v;
    }
    bool flag()
    {
        PyObject *o = next();
        if (!o || !PyBool_Check(o)) ok = false;
        return o == Py_True;
    }
    // a tuple of three integers; None: false
    bool counts(int (&to)[3])
    {
        PyObject *o = next();
        if (o == Py_None) return false;
        if (!o || !PyTuple_CheckExact(o) || PyTuple_GET_SIZE(o) != 3) {
            ok = false;
            return false;
        }
        Reader each(&PyTuple_GET_ITEM(o, 0), 3);
        for (int &count : to) count = each.integer();
        ok &= each.ok;
        return ok;
    }
    float number()
    {
        PyObject *o = next();
        if (!o || !PyFloat_CheckExact(o)) {
            ok = false;
            return 0.f;
        }
        return (float)PyFloat_AS_DOUBLE(o);
    }
    void *stream()  // None: torch's current stream of the current device
    {
        PyObject *o = next();
        if (o == Py_None) return (void *)c10::hip::getCurrentHIPStream().stream();
        if (o && PyLong_CheckExact(o)) {
            void *const handle = PyLong_AsVoidPtr(o);
            if (handle || !PyErr_Occurred()) return handle;
            PyErr_Clear();
        }
        ok = false;
        return nullptr;
    }
    // a contiguous tensor of one type
    void *operand(at::ScalarType type)
    {
        const at::Tensor *t = tensor();
        if (!t || t->scalar_type() != type || !t->is_contiguous()) {
            ok = false;
            return nullptr;
        }
        return t->data_ptr();
    }
    void *indices() { return operand(at::kInt); }
    void *halves() { return operand(at::kHalf); }
    // halves or floats
    void *output(bool &f32)
    {
        const at::Tensor *t = tensor();
        if (!t || (t->scalar_type() != at::kHalf && t->scalar_type() != at::kFloat) || !t->is_contiguous()) {
            ok = false;
            return nullptr;
        }
        f32 = t->scalar_type() == at::kFloat;
        return t->data_ptr();
    }
    // [batch, rows, columns] (or two-dimensional: shared), contiguous behind the first dimension; `batch` of one or a
    // shared operand has no stride
    void *batched(int batch, long long &stride)
    {
        const at::Tensor *t = tensor();
        stride = 0;
        if (!t || t->scalar_type() != at::kHalf) {
            ok = false;
            return nullptr;
        }
        if (t->dim() == 3) {
            const auto sizes = t->sizes(), strides = t->strides();
            const bool whole = sizes[1] == 0 || sizes[2] == 0 ||
                               ((sizes[2] == 1 || strides[2] == 1) && (sizes[1] == 1 || strides[1] == sizes[2]));
            if (!whole || sizes[0] == 0) ok = false;
            if (batch != 1) stride = strides[0];
        } else if (!t->is_contiguous()) {
            ok = false;
        }
        return t->data_ptr();
    }
    // batched, of an operand that is written: no two problems may share an element
    void *batched_output(int batch, long long &stride)
    {
        const at::Tensor *t = ok && left > 0 && THPVariable_Check(*args) ? &THPVariable_Unpack(*args) : nullptr;
        void *const p = batched(batch, stride);
        if (ok && batch != 1 && t->dim() == 3 && stride < (long long)t->size(1) * t->size(2)) ok = false;
        return p;
    }
    // batched_output, of an operand that is read first: every problem has one
    void *batched_in_place(int batch, long long &stride)
    {
        const at::Tensor *t = ok && left > 0 && THPVariable_Check(*args) ? &THPVariable_Unpack(*args) : nullptr;
        void *const p = batched_output(batch, stride);
        if (ok && batch > 1 && (t->dim() != 3 || t->size(0) < batch)) ok = false;
        return p;
    }
    // bytes of a caller's buffer, or None
    void *buffer(long long &bytes)
    {
        bytes = 0;
        if (ok && left > 0 && *args == Py_None) {
            next();
            return nullptr;
        }
        const at::Tensor *t = tensor();
        if (!t) return nullptr;
        bytes = (long long)t->numel() * (long long)t->element_size();
        return t->data_ptr();
    }
    bool done() const { return ok && left == 0; }
};

template <typename Call>
PyObject *status_of(const Reader &r, Call &&call)
{
    if (!r.done()) return PyLong_FromLong(kUnusual);
    int status;
    Py_BEGIN_ALLOW_THREADS;
    status = call();
    Py_END_ALLOW_THREADS;
    return PyLong_FromLong(status);
}

typedef int (*SpmmEntry)(int, int, int, int, const int *, const int *, const int *, const void *, const void *, void *, void *);
typedef int (*SpmmEntryF32)(int, int, int, int, const int *, const int *, const int *, const void *, const void *, float *, void *);

// (m_vec, vec_length, k, n, row_indices, row_offsets, column_indices, values, rhs, out, stream)
template <SpmmEntry F16, SpmmEntryF32 F32>
PyObject *spmm(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int m_vec = r.integer(), v = r.integer(), k = r.integer(), n = r.integer();
    const int *ri = (const int *)r.indices(), *ro = (const int *)r.indices(), *ci = (const int *)r.indices();
    const void *values = r.halves(), *rhs = r.halves();
    bool f32 = false;
    void *out = r.output(f32), *stream = r.stream();
    return status_of(r, [&] {
        return f32 ? F32(m_vec, v, k, n, ri, ro, ci, values, rhs, (float *)out, stream)
                   : F16(m_vec, v, k, n, ri, ro, ci, values, rhs, out, stream);
    });
}

// (fine_grained, m_vec, vec_length, k, n, nonzeros_vec, longest_row_vec, long_rows, row_length_hints, row_indices, row_offsets,
// column_indices, values, rhs, out, stream, lists), fp16 outputs; lists: the three counts of vs_spmm_packed_lists where the caller may
// make a workspace, else None; -2 - with nothing launched - where spmm_packed is expected to be faster
PyObject *spmm_ascending(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const bool fine_grained = r.flag();
    const int m_vec = r.integer(), v = r.integer(), k = r.integer(), n = r.integer(), nnz = r.integer(), longest = r.integer();
    const int long_rows = r.integer();
    const bool hints = r.flag();
    const int *ri = (const int *)r.indices(), *ro = (const int *)r.indices(), *ci = (const int *)r.indices();
    const void *values = r.halves(), *rhs = r.halves();
    void *out = r.halves(), *stream = r.stream();
    int lists[3];
    if (r.counts(lists) && r.done() && vs_spmm_packed_workspace_bytes_lists(fine_grained, m_vec, v, k, n, nnz, longest, lists) > 0) return PyLong_FromLong(-2);
    return status_of(r, [&] {
        return fine_grained ? vs_cuda_spmm_f16_ascending(m_vec, v, k, n, nnz, longest, hints, ri, ro, ci, values, rhs, out, stream)
                            : vs_wmma_spmm_f16_ascending(m_vec, v, k, n, nnz, longest, long_rows, hints, ri, ro, ci, values, rhs, out, stream);
    });
}

// (fine_grained, m_vec, vec_length, k, n, nonzeros_vec, longest_row_vec, row_offsets, column_indices, values, rhs, out, workspace, stream)
PyObject *spmm_packed(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const bool fine_grained = r.flag();
    const int m_vec = r.integer(), v = r.integer(), k = r.integer(), n = r.integer(), nnz = r.integer(), longest = r.integer();
    const int *ro = (const int *)r.indices(), *ci = (const int *)r.indices();
    const void *values = r.halves(), *rhs = r.halves();
    void *out = r.halves();
    long long bytes;
    void *workspace = r.buffer(bytes), *stream = r.stream();
    return status_of(r, [&] {
        return vs_spmm_f16_packed(fine_grained, m_vec, v, k, n, nnz, longest, ro, ci, values, rhs, out, workspace, bytes, stream);
    });
}

// (m_vec, k, n, nonzeros_vec, row_indices, row_offsets, col_indices, lhs, rhs, out, vec_length, stream, algorithm, columns_sorted)
PyObject *wmma_sddmm(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int m_vec = r.integer(), k = r.integer(), n = r.integer(), nnz = r.integer();
    const int *ri = (const int *)r.indices(), *ro = (const int *)r.indices(), *ci = (const int *)r.indices();
    const void *lhs = r.halves(), *rhs = r.halves();
    bool f32 = false;
    void *out = r.output(f32);
    const int v = r.integer();
    void *stream = r.stream();
    const int algorithm = r.integer();
    const bool sorted = r.flag();
    return status_of(r, [&] {
        if (sorted) return vs_wmma_sddmm_f16_sorted(1, m_vec, k, n, nnz, ri, ro, ci, lhs, 0, rhs, 0, out, 0, f32, v, stream, algorithm);
        return f32 ? vs_wmma_sddmm_f16_f32out(m_vec, k, n, nnz, ri, ro, ci, lhs, rhs, (float *)out, v, stream, algorithm)
                   : vs_wmma_sddmm_f16(m_vec, k, n, nnz, ri, ro, ci, lhs, rhs, out, v, stream, algorithm);
    });
}

// (m_vec, k, n, nonzeros_vec, row_indices, row_offsets, col_indices, lhs, rhs, out, vec_length, stream, columns_sorted)
PyObject *cuda_sddmm(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int m_vec = r.integer(), k = r.integer(), n = r.integer(), nnz = r.integer();
    const int *ri = (const int *)r.indices(), *ro = (const int *)r.indices(), *ci = (const int *)r.indices();
    const void *lhs = r.halves(), *rhs = r.halves();
    bool f32 = false;
    void *out = r.output(f32);
    const int v = r.integer();
    void *stream = r.stream();
    const bool sorted = r.flag();
    return status_of(r, [&] {
        if (sorted) return vs_cuda_sddmm_f16_sorted(1, m_vec, k, n, nnz, ri, ro, ci, lhs, 0, rhs, 0, out, 0, f32, v, stream);
        return f32 ? vs_cuda_sddmm_f16_f32out(m_vec, k, n, nnz, ri, ro, ci, lhs, rhs, (float *)out, v, stream)
                   : vs_cuda_sddmm_f16(m_vec, k, n, nnz, ri, ro, ci, lhs, rhs, out, v, stream);
    });
}

// (batch, m_vec, vec_length, k, n, nonzeros_vec, longest_row_vec, long_rows, row_indices, row_offsets, column_indices, values,
// rhs, out, stream); MFMA path, long_rows < 0: not known
PyObject *wmma_spmm_batched(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int batch = r.integer(), m_vec = r.integer(), v = r.integer(), k = r.integer(), n = r.integer();
    const int nnz = r.integer(), longest = r.integer(), long_rows = r.integer();
    const int *ri = (const int *)r.indices(), *ro = (const int *)r.indices(), *ci = (const int *)r.indices();
    long long sa, sb, so;
    const void *values = r.batched(batch, sa), *rhs = r.batched(batch, sb);
    void *out = r.batched(batch, so), *stream = r.stream();
    return status_of(r, [&] {
        return long_rows >= 0
                   ? vs_wmma_spmm_f16_batched_sorted(batch, m_vec, v, k, n, nnz, longest, long_rows, ri, ro, ci, values, sa, rhs, sb, out, so, stream)
                   : vs_wmma_spmm_f16_batched(batch, m_vec, v, k, n, nnz, longest, ri, ro, ci, values, sa, rhs, sb, out, so, stream);
    });
}

// (batch, m_vec, vec_length, k, n, nonzeros_vec, longest_row_vec, row_indices, row_offsets, column_indices, values, rhs, out,
// stream); fine-grained path
PyObject *cuda_spmm_batched(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int batch = r.integer(), m_vec = r.integer(), v = r.integer(), k = r.integer(), n = r.integer();
    const int nnz = r.integer(), longest = r.integer();
    const int *ri = (const int *)r.indices(), *ro = (const int *)r.indices(), *ci = (const int *)r.indices();
    long long sa, sb, so;
    const void *values = r.batched(batch, sa), *rhs = r.batched(batch, sb);
    void *out = r.batched(batch, so), *stream = r.stream();
    return status_of(r, [&] {
        return vs_cuda_spmm_f16_batched(batch, m_vec, v, k, n, nnz, longest, ri, ro, ci, values, sa, rhs, sb, out, so, stream);
    });
}

// (batch, m_vec, vec_length, k, n, nonzeros_vec, longest_row_vec, row_indices, row_offsets, column_indices, scores, rhs, out,
// scale, stream); KEPT: the scores become the probabilities
template <bool KEPT>
PyObject *spmm_softmax_batched(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int batch = r.integer(), m_vec = r.integer(), v = r.integer(), k = r.integer(), n = r.integer();
    const int nnz = r.integer(), longest = r.integer();
    const int *ri = (const int *)r.indices(), *ro = (const int *)r.indices(), *ci = (const int *)r.indices();
    long long sa, sb, so;
    void *scores = KEPT ? r.batched_in_place(batch, sa) : r.batched(batch, sa);
    const void *rhs = r.batched(batch, sb);
    void *out = r.batched(batch, so);
    const float scale = r.number();
    void *stream = r.stream();
    return status_of(r, [&] {
        if constexpr (KEPT)
            return vs_wmma_softmax_spmm_f16_batched(batch, m_vec, v, k, n, nnz, longest, ri, ro, ci, scores, sa, rhs, sb, out, so, scale, stream);
        else
            return vs_wmma_spmm_softmax_f16_batched(batch, m_vec, v, k, n, nnz, longest, ri, ro, ci, scores, sa, rhs, sb, out, so, scale, stream);
    });
}

// (batch, m_vec, vec_length, n, d_qk, d_v, nonzeros_vec, longest_row_vec, row_indices, row_offsets, col_indices, q, k, v, out,
// probabilities or None, scale, stream)
PyObject *sparse_attention_rows(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int batch = r.integer(), m_vec = r.integer(), vec = r.integer(), n = r.integer(), d_qk = r.integer(), d_v = r.integer();
    const int nnz = r.integer(), longest = r.integer();
    const int *ri = (const int *)r.indices(), *ro = (const int *)r.indices(), *ci = (const int *)r.indices();
    long long sq, sk, sv, so, sp = 0;
    const void *q = r.batched(batch, sq), *k = r.batched(batch, sk), *v = r.batched(batch, sv);
    void *out = r.batched_output(batch, so), *probabilities = nullptr;
    if (r.ok && r.left > 0 && *r.args == Py_None) r.next();
    else probabilities = r.batched_in_place(batch, sp);
    const float scale = r.number();
    void *stream = r.stream();
    return status_of(r, [&] {
        return vs_sparse_attention_rows_f16(batch, m_vec, vec, n, d_qk, d_v, nnz, longest, ri, ro, ci, q, sq, k, sk, v, sv, out, so,
                                            probabilities, sp, scale, stream);
    });
}

// (batch, m_vec, k, n, nonzeros_vec, row_indices, row_offsets, col_indices, lhs, rhs, out, vec_length, stream, columns_sorted)
// and, MFMA path, (..., algorithm)
template <bool MFMA>
PyObject *sddmm_batched(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int batch = r.integer(), m_vec = r.integer(), k = r.integer(), n = r.integer(), nnz = r.integer();
    const int *ri = (const int *)r.indices(), *ro = (const int *)r.indices(), *ci = (const int *)r.indices();
    long long sa, sb, so;
    const void *lhs = r.batched(batch, sa), *rhs = r.batched(batch, sb);
    void *out = r.batched(batch, so);
    const int v = r.integer();
    void *stream = r.stream();
    const bool sorted = r.flag();
    const int algorithm = MFMA ? r.integer() : 0;
    return status_of(r, [&] {
        if constexpr (MFMA)
            return sorted ? vs_wmma_sddmm_f16_sorted(batch, m_vec, k, n, nnz, ri, ro, ci, lhs, sa, rhs, sb, out, so, 0, v, stream, algorithm)
                          : vs_wmma_sddmm_f16_batched(batch, m_vec, k, n, nnz, ri, ro, ci, lhs, sa, rhs, sb, out, so, v, stream, algorithm);
        else
            return sorted ? vs_cuda_sddmm_f16_sorted(batch, m_vec, k, n, nnz, ri, ro, ci, lhs, sa, rhs, sb, out, so, 0, v, stream)
                          : vs_cuda_sddmm_f16_batched(batch, m_vec, k, n, nnz, ri, ro, ci, lhs, sa, rhs, sb, out, so, v, stream);
    });
}

// (batch, m_vec, vec_length, row_indices, row_offsets, values_in, values_out, scale, stream)
PyObject *sparse_softmax(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int batch = r.integer(), m_vec = r.integer(), v = r.integer();
    const int *ri = (const int *)r.indices(), *ro = (const int *)r.indices();
    long long si, so;
    const void *in = r.batched(batch, si);
    void *out = r.batched(batch, so);
    const float scale = r.number();
    void *stream = r.stream();
    return status_of(r, [&] { return vs_sparse_softmax_f16(batch, m_vec, v, ri, ro, in, si, out, so, scale, stream); });
}

// (batch, m_vec, vec_length, n, d_qk, d_v, row_indices, row_offsets, col_indices, q, k, v, out, scale, rows_per_workgroup, plan,
// stream)
PyObject *sparse_attention(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int batch = r.integer(), m_vec = r.integer(), vec = r.integer(), n = r.integer(), d_qk = r.integer(), d_v = r.integer();
    const int *ri = (const int *)r.indices(), *ro = (const int *)r.indices(), *ci = (const int *)r.indices();
    long long sq, sk, sv, so, plan_bytes;
    const void *q = r.batched(batch, sq), *k = r.batched(batch, sk), *v = r.batched(batch, sv);
    void *out = r.batched(batch, so);
    const float scale = r.number();
    const int rows = r.integer();
    const void *plan = r.buffer(plan_bytes);
    void *stream = r.stream();
    return status_of(r, [&] {
        return vs_sparse_attention_f16(batch, m_vec, vec, n, d_qk, d_v, ri, ro, ci, q, sq, k, sk, v, sv, out, so, scale, rows, plan,
                                       plan_bytes, stream);
    });
}

// (batch, m_vec, vec_length, n, d_qk, d_v, row_offsets, col_indices, q, k, v, out, scale, plan, slots, n_slots, n_merges,
// n_partials, workspace, stream)
PyObject *sparse_attention_split(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int batch = r.integer(), m_vec = r.integer(), vec = r.integer(), n = r.integer(), d_qk = r.integer(), d_v = r.integer();
    const int *ro = (const int *)r.indices(), *ci = (const int *)r.indices();
    long long sq, sk, sv, so, plan_bytes, bytes;
    const void *q = r.batched(batch, sq), *k = r.batched(batch, sk), *v = r.batched(batch, sv);
    void *out = r.batched(batch, so);
    const float scale = r.number();
    const void *plan = r.buffer(plan_bytes);
    const int *slots = (const int *)r.indices();
    const int n_slots = r.integer(), n_merges = r.integer(), n_partials = r.integer();
    void *workspace = r.buffer(bytes), *stream = r.stream();
    return status_of(r, [&] {
        return vs_sparse_attention_f16_split(batch, m_vec, vec, n, d_qk, d_v, ro, ci, q, sq, k, sk, v, sv, out, so, scale, plan,
                                             plan_bytes, slots, n_slots, n_merges, n_partials, workspace, bytes, stream);
    });
}

// (batch, vec_length, k, n, n_slots, slots, n_split, parts_max, nonzeros_vec, longest_part_vec, column_indices, values, rhs, out,
// workspace, stream)
PyObject *spmm_row_parts(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int batch = r.integer(), vec = r.integer(), k = r.integer(), n = r.integer(), n_slots = r.integer();
    const int *slots = (const int *)r.indices();
    const int n_split = r.integer(), parts_max = r.integer(), nnz = r.integer(), longest = r.integer();
    const int *ci = (const int *)r.indices();
    long long sa, sb, so, ws_bytes;
    const void *values = r.batched(batch, sa), *rhs = r.batched(batch, sb);
    void *out = r.batched_output(batch, so), *ws = r.buffer(ws_bytes), *stream = r.stream();
    return status_of(r, [&] {
        return vs_wmma_spmm_f16_row_parts(batch, vec, k, n, n_slots, slots, n_split, parts_max, nnz, longest, ci, values, sa, rhs, sb,
                                          out, so, ws, ws_bytes, stream);
    });
}

// (batch, k, n, n_slots, slots, nonzeros_vec, col_indices, lhs, rhs, out, vec_length, stream)
PyObject *sddmm_row_parts(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int batch = r.integer(), k = r.integer(), n = r.integer(), n_slots = r.integer();
    const int *slots = (const int *)r.indices();
    const int nnz = r.integer();
    const int *ci = (const int *)r.indices();
    long long sa, sb, so;
    const void *lhs = r.batched(batch, sa), *rhs = r.batched(batch, sb);
    void *out = r.batched_output(batch, so);
    const int vec = r.integer();
    void *stream = r.stream();
    return status_of(r, [&] {
        return vs_wmma_sddmm_f16_row_parts(batch, k, n, n_slots, slots, nnz, ci, lhs, sa, rhs, sb, out, so, vec, stream);
    });
}

// (batch, vec_length, n_slots, slots, n_split, parts_max, values_in, values_out, scale, workspace, stream)
PyObject *softmax_row_parts(PyObject *, PyObject *const *args, Py_ssize_t n_args)
{
    Reader r(args, n_args);
    const int batch = r.integer(), vec = r.integer(), n_slots = r.integer();
    const int *slots = (const int *)r.indices();
    const int n_split = r.integer(), parts_max = r.integer();
    long long si, so, ws_bytes;
    const void *in = r.batched(batch, si);
    void *out = r.batched_output(batch, so);
    const float scale = r.number();
    void *ws = r.buffer(ws_bytes), *stream = r.stream();
    return status_of(r, [&] {
        return vs_sparse_softmax_f16_row_parts(batch, vec, n_slots, slots, n_split, parts_max, in, si, out, so, scale, ws, ws_bytes, stream);
    });
}

// Tensors without storage (fake and functional ones, those inside vmap) throw when they are asked for an address, a
// process without a device when it is asked for a stream; an exception must not leave a C function.  Both are unusual
// arguments: ops.py meets the same refusal as a Python exception.
typedef PyObject *(*Method)(PyObject *, PyObject *const *, Py_ssize_t);
template <Method F>
PyObject *guarded(PyObject *self, PyObject *const *args, Py_ssize_t n_args) noexcept
{
    try {
        return F(self, args, n_args);
    } catch (...) {
        return PyLong_FromLong(kUnusual);
    }
}

#define VS_METHOD(name, fn) {name, (PyCFunction)(void (*)(void))(guarded<fn>), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    VS_METHOD("wmma_spmm", (spmm<vs_wmma_spmm_f16, vs_wmma_spmm_f16_f32out>)),
    VS_METHOD("cuda_spmm", (spmm<vs_cuda_spmm_f16, vs_cuda_spmm_f16_f32out>)),
    VS_METHOD("spmm_ascending", spmm_ascending),
    VS_METHOD("spmm_packed", spmm_packed),
    VS_METHOD("wmma_sddmm", wmma_sddmm),
    VS_METHOD("cuda_sddmm", cuda_sddmm),
    VS_METHOD("wmma_spmm_batched", wmma_spmm_batched),
    VS_METHOD("cuda_spmm_batched", cuda_spmm_batched),
    VS_METHOD("spmm_softmax_batched", spmm_softmax_batched<false>),
    VS_METHOD("softmax_spmm_batched", spmm_softmax_batched<true>),
    VS_METHOD("wmma_sddmm_batched", sddmm_batched<true>),
    VS_METHOD("cuda_sddmm_batched", sddmm_batched<false>),
    VS_METHOD("sparse_softmax", sparse_softmax),
    VS_METHOD("sparse_attention", sparse_attention),
    VS_METHOD("sparse_attention_rows", sparse_attention_rows),
    VS_METHOD("sparse_attention_split", sparse_attention_split),
    VS_METHOD("spmm_row_parts", spmm_row_parts),
    VS_METHOD("sddmm_row_parts", sddmm_row_parts),
    VS_METHOD("softmax_row_parts", softmax_row_parts),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding() { return PyModule_Create(&module); }
