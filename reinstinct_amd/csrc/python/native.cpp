// The launch calls of reinstinct_amd.runtime as a CPython extension over librein's C ABI: a decode step makes hundreds of
// them, a few microseconds each on the GPU, and a ctypes call with eight arguments costs 0.7-1.1 us of conversions, the
// four tables of matvec_multi_xq8 2.4 (hipModuleLaunchKernel itself: 2.4).  Here a call is a walk over its
// arguments, about 0.1 us.  The GIL is released around the C call, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <array>
#include <cstring>
#include <tuple>
#include <utility>

#include "../../../include/rein.h"

namespace {

PyObject* g_check;        // reinstinct_amd._lib.check: raises ReinError with rein_last_error()
PyObject* g_shape;        // reinstinct_amd._lib.MoeShape
PyObject* g_as_parameter;
PyObject* g_value;
PyObject* g_raw;
PyObject *g_cast, *g_void_p, *g_int, *g_uint, *g_size, *g_float;        // of ctypes

// ---- one argument.  What ctypes takes for a parameter of its C type is taken, and nothing else: the quick ways are a test of the
// type, the others go through ctypes' own types.  Whole numbers are cut to their C type as ctypes does.
bool to_c(PyObject* o, void** out);
bool to_c(PyObject* o, unsigned* out);
bool to_c(PyObject* o, int* out);
bool to_c(PyObject* o, size_t* out);
bool to_c(PyObject* o, float* out);

// the attribute of o called name, converted; -1: there is none
template <class T> int from_attribute(PyObject* o, PyObject* name, T* out)
{
    PyObject* v = PyObject_GetAttr(o, name);
    if (!v) {
        PyErr_Clear();
        return -1;
    }
    bool ok = false;
    if (Py_EnterRecursiveCall(" in an argument") == 0) {
        ok = to_c(v, out);
        Py_LeaveRecursiveCall();
    }
    Py_DECREF(v);
    return ok;
}
bool wrong(const char* want, PyObject* o)
{
    PyErr_Format(PyExc_TypeError, "%s is wanted, not %.80s", want, Py_TYPE(o)->tp_name);
    return false;
}
// a pointer: an int, None, an object that stands for one (DeviceBuf), or what ctypes turns into a void pointer
bool to_c(PyObject* o, void** out)
{
    if (PyLong_Check(o)) {
        *out = PyLong_AsVoidPtr(o);
        return *out || !PyErr_Occurred();
    }
    if (o == Py_None) {
        *out = nullptr;
        return true;
    }
    const int got = from_attribute(o, g_as_parameter, out);
    if (got >= 0) return got;
    PyObject* p = PyObject_CallFunctionObjArgs(g_cast, o, g_void_p, nullptr);
    if (!p) {
        PyErr_Clear();
        return wrong("a device pointer (an int, None or a DeviceBuf)", o);
    }
    const int ok = from_attribute(p, g_value, out);          // the memory it points to is o's, which the caller holds
    Py_DECREF(p);
    return ok > 0;
}
// a stream: None or a hip.Stream, an object whose `raw` is the handle.  Nothing else: a number here is a count or a pointer that
// slipped by one parameter
struct Stream { void* raw; operator void*() const { return raw; } };
bool to_c(PyObject* o, Stream* out)
{
    out->raw = nullptr;
    if (o == Py_None) return true;
    const int got = from_attribute(o, g_raw, &out->raw);
    return got < 0 ? wrong("a stream (a hip.Stream or None)", o) : got;
}
template <class T> bool to_c(PyObject* o, T** out) { return to_c(o, reinterpret_cast<void**>(const_cast<std::remove_const_t<T>**>(out))); }
template <class T> bool whole(PyObject* o, PyObject* ctype, T* out)
{
    if (PyLong_Check(o) || PyIndex_Check(o)) {
        const unsigned long long v = PyLong_AsUnsignedLongLongMask(o);
        *out = (T)v;
        return v != (unsigned long long)-1 || !PyErr_Occurred();
    }
    const int is = PyObject_IsInstance(o, ctype);
    if (is < 0) return false;
    const int got = from_attribute(o, is ? g_value : g_as_parameter, out);
    return got < 0 ? wrong("a whole number", o) : got;
}
bool to_c(PyObject* o, unsigned* out) { return whole(o, g_uint, out); }
bool to_c(PyObject* o, int* out) { return whole(o, g_int, out); }
bool to_c(PyObject* o, size_t* out) { return whole(o, g_size, out); }
bool to_c(PyObject* o, float* out)
{
    const double v = PyFloat_AsDouble(o);
    *out = (float)v;
    if (v != -1.0 || !PyErr_Occurred()) return true;
    PyErr_Clear();
    const int is = PyObject_IsInstance(o, g_float);
    if (is < 0) return false;
    const int got = from_attribute(o, is ? g_value : g_as_parameter, out);
    return got < 0 ? wrong("a number", o) : got;
}

// ---- the arguments of a call in the order of the parameters, keywords and defaults filled in.  `names` ends with NULL;
// the last `n_dflt` parameters have a default.
template <size_t N>
bool gather(const char* who, const char* const* names, PyObject* const* dflt, size_t n_dflt, PyObject* const* args, Py_ssize_t n,
            PyObject* kwnames, std::array<PyObject*, N>& got)
{
    const size_t n_pos = (size_t)n;
    if (n_pos > N) {
        PyErr_Format(PyExc_TypeError, "%s() takes %zu arguments, %zu given", who, N, n_pos);
        return false;
    }
    for (size_t i = 0; i < N; i++) got[i] = i < n_pos ? args[i] : nullptr;
    const Py_ssize_t n_kw = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
    for (Py_ssize_t k = 0; k < n_kw; k++) {
        PyObject* name = PyTuple_GET_ITEM(kwnames, k);
        size_t i = 0;
        while (i < N && PyUnicode_CompareWithASCIIString(name, names[i]) != 0) i++;
        if (i == N || got[i]) {
            PyErr_Format(PyExc_TypeError, "%s() got %s '%U'", who, i == N ? "an unexpected keyword argument" : "more than one value for", name);
            return false;
        }
        got[i] = args[n + k];
    }
    for (size_t i = 0; i < N; i++) {
        if (got[i]) continue;
        if (i + n_dflt < N) {
            PyErr_Format(PyExc_TypeError, "%s() is missing the argument '%s'", who, names[i]);
            return false;
        }
        got[i] = dflt[i + n_dflt - N];
    }
    return true;
}

PyObject* result(int rc)
{
    if (rc == 0) Py_RETURN_NONE;
    return PyObject_CallFunction(g_check, "i", rc);      // raises
}

template <class... A, size_t... I>
PyObject* call(int (*fn)(A...), const std::array<PyObject*, sizeof...(A)>& got, std::index_sequence<I...>)
{
    // (the last parameter of every one of them is the stream)
    std::tuple<std::conditional_t<I + 1 == sizeof...(A), Stream, A>...> c;
    if (!(to_c(got[I], &std::get<I>(c)) && ...)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = fn(std::get<I>(c)...);
    Py_END_ALLOW_THREADS
    return result(rc);
}
template <class... A>
PyObject* run(int (*fn)(A...), const char* who, const char* const* names, PyObject* const* dflt, size_t n_dflt, PyObject* const* args,
              Py_ssize_t n, PyObject* kw)
{
    std::array<PyObject*, sizeof...(A)> got;
    if (!gather(who, names, dflt, n_dflt, args, n, kw, got)) return nullptr;
    return call(fn, got, std::index_sequence_for<A...>{});
}

PyObject* g_none[1];                     // defaults: stream
PyObject* g_one_none[2];                 // a count, stream
PyObject* g_one_eps_none[3];             // a count, eps, stream
PyObject* g_eps_none[2];                 // eps, stream

// A function whose Python parameters are those of the C function, in its order
#define REIN_FN(name, dflt, n_dflt, ...)                                                               \
    PyObject* py_##name(PyObject*, PyObject* const* a, Py_ssize_t n, PyObject* kw)                     \
    {                                                                                                  \
        static const char* const names[] = {__VA_ARGS__, nullptr};                                    \
        return run(rein_##name, #name, names, dflt, n_dflt, a, n, kw);                                 \
    }
REIN_FN(quantize_q8, g_one_none, 2, "x", "xq", "in_dim", "n_vec", "stream")
REIN_FN(rmsnorm_q8, g_one_eps_none, 3, "x", "w", "xq", "n", "n_vec", "eps", "stream")
REIN_FN(add_rmsnorm_q8, g_one_eps_none, 3, "hidden", "add", "w", "y", "xq", "n", "n_vec", "eps", "stream")
REIN_FN(swiglu_q8, g_none, 1, "gate", "up", "out", "xq", "n", "stream")
REIN_FN(sigmoid_mul_q8, g_none, 1, "x", "gate", "xq", "n", "stream")
REIN_FN(rmsnorm_gated_q8, g_eps_none, 2, "x", "z", "w", "y", "xq", "n_heads", "head_dim", "eps", "stream")
REIN_FN(moe_geglu_q8, g_none, 1, "gu", "xq", "ff_exp", "n_slot", "stream")
REIN_FN(matvec_xq8, g_none, 1, "fmt", "w", "xq", "y", "in_dim", "out_dim", "stream")
REIN_FN(matvec_batched_xq8, g_none, 1, "fmt", "w", "xq", "y", "in_dim", "out_dim", "n_rows", "stream")
REIN_FN(matvec_ondisk_xq8, g_none, 1, "fmt", "w_blocks", "xq", "y", "in_dim", "out_dim", "stream")
REIN_FN(matvec_q8_0_splitk, g_none, 1, "w", "xq", "y_partials", "in_dim", "out_dim", "n_split", "stream")
REIN_FN(mmq_xq8, g_none, 1, "fmt", "w", "xq", "y", "in_dim", "out_dim", "p_rows", "stream")
REIN_FN(mmq_xq8_ws, g_none, 1, "fmt", "w", "xq", "y", "in_dim", "out_dim", "p_rows", "workspace", "workspace_bytes", "stream")
REIN_FN(mmq_xq8_noalloc, g_none, 1, "fmt", "w", "xq", "y", "in_dim", "out_dim", "p_rows", "stream")
REIN_FN(matmul, g_none, 1, "fmt", "w", "x", "y", "in_dim", "out_dim", "n_rows", "xq_scratch", "stream")
REIN_FN(matmul_ws, g_none, 1, "fmt", "w", "x", "y", "in_dim", "out_dim", "n_rows", "scratch", "scratch_bytes", "stream")
REIN_FN(moe_topk, g_none, 1, "logits", "n_tok", "n_expert", "n_used", "out_ids", "out_weights", "stream")
REIN_FN(moe_sort, g_none, 1, "ids", "n_entries", "n_expert", "bn", "count", "cursor", "perm", "expert_off", "tile_off", "stream")
REIN_FN(moe_gather_xq, g_none, 1, "xq_src", "perm", "xq_dst", "nsub", "n_used", "n_entries", "stream")
REIN_FN(moe_quantize_scatter, g_none, 1, "x", "inv", "xq_dst", "in_dim", "n_used", "n_tok", "stream")
REIN_FN(moe_scatter_rows, g_none, 1, "src", "perm", "dst", "dim", "n_entries", "stream")
REIN_FN(moe_grouped_gemm, g_none, 1, "fmt", "slab", "bytes_per_expert", "expert_off", "tile_off", "n_expert", "xq", "y", "in_dim", "out_dim",
        "n_entries", "stream")
REIN_FN(moe_grouped_swiglu_q8, g_none, 1, "fmt", "gate_slab", "up_slab", "bytes_per_expert", "expert_off", "tile_off", "n_expert", "xq",
        "xq_out", "in_dim", "out_dim", "n_entries", "stream")
REIN_FN(moe_expert_matvec, g_one_none, 2, "fmt", "slab", "ids", "xq", "y", "in_dim", "out_dim", "bytes_per_expert", "xq_tok_stride",
        "xq_slot_stride", "n_used", "n_tok", "stream")
REIN_FN(moe_down, g_one_none, 2, "fmt", "slab", "ids", "xq", "y", "in_dim", "out_dim", "bytes_per_expert", "xq_tok_stride",
        "xq_slot_stride", "n_used", "n_tok", "stream")
REIN_FN(moe_gate_up_swiglu, g_one_none, 2, "fmt", "gate_slab", "up_slab", "ids", "xq", "y", "in_dim", "out_dim", "bytes_per_expert",
        "xq_tok_stride", "xq_slot_stride", "n_used", "n_tok", "stream")
REIN_FN(moe_gate_up_swiglu_q8, g_one_none, 2, "fmt", "gate_slab", "up_slab", "ids", "xq", "xq_out", "in_dim", "out_dim", "bytes_per_expert",
        "xq_tok_stride", "xq_slot_stride", "n_used", "n_tok", "stream")
REIN_FN(moe_down_combine, g_one_none, 2, "fmt", "slab", "ids", "weights", "down_exps_s", "xq", "out", "in_dim", "out_dim", "bytes_per_expert",
        "xq_tok_stride", "xq_slot_stride", "n_used", "n_tok", "stream")
REIN_FN(swiglu_mul, g_none, 1, "gate", "up", "out", "n", "stream")
REIN_FN(moe_combine, g_none, 1, "experts", "ids", "weights", "down_exps_s", "out", "n_tok", "hidden", "n_used", "stream")

// the tables of matvec_multi_xq8: sequences of as many elements; the library takes four at most and says so itself
template <class T>
bool table(PyObject* o, const char* what, Py_ssize_t n, T* out)
{
    PyObject* s = PySequence_Fast(o, what);
    if (!s) return false;
    bool ok = PySequence_Fast_GET_SIZE(s) == n;
    if (!ok) PyErr_Format(PyExc_ValueError, "matvec_multi_xq8: %s holds %zd elements, fmts %zd", what, PySequence_Fast_GET_SIZE(s), n);
    for (Py_ssize_t i = 0; ok && i < n && i < 4; i++) ok = to_c(PySequence_Fast_GET_ITEM(s, i), &out[i]);
    Py_DECREF(s);
    return ok;
}
PyObject* py_matvec_multi_xq8(PyObject*, PyObject* const* a, Py_ssize_t nargs, PyObject* kw)
{
    static const char* const names[] = {"fmts", "ws", "ys", "out_dims", "xq", "in_dim", "n_rows", "stream", nullptr};
    std::array<PyObject*, 8> got;
    if (!gather("matvec_multi_xq8", names, g_one_none, 2, a, nargs, kw, got)) return nullptr;
    const Py_ssize_t n = PySequence_Size(got[0]);
    if (n < 0) return nullptr;
    int fmts[4] = {};
    const void* ws[4] = {};
    float* ys[4] = {};
    unsigned dims[4] = {}, in_dim, n_rows;
    const void* xq;
    Stream stream;
    if (!table(got[0], "fmts", n, fmts) || !table(got[1], "ws", n, ws) || !table(got[2], "ys", n, ys) || !table(got[3], "out_dims", n, dims) ||
        !to_c(got[4], &xq) || !to_c(got[5], &in_dim) || !to_c(got[6], &n_rows) || !to_c(got[7], &stream))
        return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = rein_matvec_multi_xq8((unsigned)n, fmts, ws, ys, dims, xq, in_dim, n_rows, stream);
    Py_END_ALLOW_THREADS
    return result(rc);
}

// the shape of moe_ffn is a ctypes structure (runtime.moe_shape), read through the buffer protocol
PyObject* py_moe_ffn(PyObject*, PyObject* const* a, Py_ssize_t nargs, PyObject* kw)
{
    static const char* const names[] = {"shape", "x", "logits", "gate_exps", "up_exps", "down_exps", "down_exps_s", "workspace", "out",
                                        "stream", nullptr};
    std::array<PyObject*, 10> got;
    if (!gather("moe_ffn", names, g_none, 1, a, nargs, kw, got)) return nullptr;
    const int is = PyObject_IsInstance(got[0], g_shape);
    if (is <= 0) {
        if (is == 0) PyErr_SetString(PyExc_TypeError, "moe_ffn: shape is what moe_shape() returns");
        return nullptr;
    }
    Py_buffer b;
    if (PyObject_GetBuffer(got[0], &b, PyBUF_SIMPLE) != 0) return nullptr;
    rein_moe_shape shape;
    std::memcpy(&shape, b.buf, sizeof shape);
    PyBuffer_Release(&b);
    void* p[8];
    Stream stream;
    for (int i = 0; i < 8; i++)
        if (!to_c(got[1 + i], &p[i])) return nullptr;
    if (!to_c(got[9], &stream)) return nullptr;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = rein_moe_ffn(&shape, (const float*)p[0], (const float*)p[1], p[2], p[3], p[4], (const float*)p[5], p[6], (float*)p[7], stream);
    Py_END_ALLOW_THREADS
    return result(rc);
}

#define REIN_DEF(name, args, doc) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL | METH_KEYWORDS, #name "(" args ")\n--\n\n" doc}
PyMethodDef g_methods[] = {
    REIN_DEF(quantize_q8, "x, xq, in_dim, n_vec=1, stream=None", "launch_quantize_q8 (src/runtime/qwen35.rs:3202-3211)"),
    REIN_DEF(rmsnorm_q8, "x, w, xq, n, n_vec=1, eps=1e-06, stream=None", "rmsnorm_q8_f32 (kernels/rmsnorm_q8.cpp:38-103): xq = q8(rmsnorm(x) * w)"),
    REIN_DEF(add_rmsnorm_q8, "hidden, add, w, y, xq, n, n_vec=1, eps=1e-06, stream=None",
             "add_rmsnorm_q8_f32 (kernels/qwen35_fused.cpp:66-121): hidden += add; y, xq = rmsnorm(hidden) * w"),
    REIN_DEF(swiglu_q8, "gate, up, out, xq, n, stream=None", "swiglu_q8_f32 (kernels/qwen35_fused.cpp:132-146): out, xq = silu(gate) * up"),
    REIN_DEF(sigmoid_mul_q8, "x, gate, xq, n, stream=None", "sigmoid_mul_q8_f32 (kernels/qwen35_fused.cpp:149-162): x *= sigmoid(gate); xq = q8(x)"),
    REIN_DEF(rmsnorm_gated_q8, "x, z, w, y, xq, n_heads, head_dim, eps=1e-06, stream=None",
             "rmsnorm_gated_q8_f32 (kernels/qwen35_fused.cpp:195-217)"),
    REIN_DEF(moe_geglu_q8, "gu, xq, ff_exp, n_slot, stream=None", "moe_geglu_q8_f32 (kernels/moe_geglu_q8.cpp:31-66): xq = q8(gelu(gate) * up)"),
    REIN_DEF(matvec_xq8, "fmt, w, xq, y, in_dim, out_dim, stream=None", "launch_matvec_repacked_xq8 (src/runtime/qwen35.rs:2232-2280)"),
    REIN_DEF(matvec_batched_xq8, "fmt, w, xq, y, in_dim, out_dim, n_rows, stream=None",
             "matmul_kquant_batched_into minus its quantize (src/runtime/prefill.rs:448-508)"),
    REIN_DEF(matvec_multi_xq8, "fmts, ws, ys, out_dims, xq, in_dim, n_rows=1, stream=None",
             "the decode step's consecutive matvecs on the same activations (Q / K / V, gate / up; src/runtime/qwen35.rs:2670-2672,\n"
             "2702-2703) as one launch: ys[i][n_rows][out_dims[i]] = xq . ws[i]^T, up to four matrices and four rows"),
    REIN_DEF(matvec_ondisk_xq8, "fmt, w_blocks, xq, y, in_dim, out_dim, stream=None", "the on-disk-layout dp4a matvec (src/runtime/qwen35.rs:2209-2229)"),
    REIN_DEF(matvec_q8_0_splitk, "w, xq, y_partials, in_dim, out_dim, n_split, stream=None",
             "matvec_q8_0_repacked_splitk_f32 (kernels/matvec_q8_0_repacked.cpp:117-176)"),
    REIN_DEF(mmq_xq8, "fmt, w, xq, y, in_dim, out_dim, p_rows, stream=None", "matmul_mmq_into minus its quantize (src/runtime/prefill.rs:512-567)"),
    REIN_DEF(mmq_xq8_ws, "fmt, w, xq, y, in_dim, out_dim, p_rows, workspace, workspace_bytes, stream=None",
             "mmq_xq8 with the caller's workspace (the scratch PrefillGemm keeps, prefill.rs:479-495)"),
    REIN_DEF(mmq_xq8_noalloc, "fmt, w, xq, y, in_dim, out_dim, p_rows, stream=None",
             "mmq_xq8_ws on the library's fixed 48 MiB device array: allocates nothing"),
    REIN_DEF(matmul, "fmt, w, x, y, in_dim, out_dim, n_rows, xq_scratch, stream=None", "PrefillGemm::matmul_into_raw (src/runtime/prefill.rs:343-384)"),
    REIN_DEF(matmul_ws, "fmt, w, x, y, in_dim, out_dim, n_rows, scratch, scratch_bytes, stream=None",
             "matmul with one scratch buffer for the quantized activations and the MMQ workspace"),
    REIN_DEF(moe_topk, "logits, n_tok, n_expert, n_used, out_ids, out_weights, stream=None", "launch of moe_topk_f32 (src/runtime/qwen35.rs:2873-2886)"),
    REIN_DEF(moe_sort, "ids, n_entries, n_expert, bn, count, cursor, perm, expert_off, tile_off, stream=None",
             "launch_moe_sort (src/runtime/qwen35.rs:2892-2938)"),
    REIN_DEF(moe_gather_xq, "xq_src, perm, xq_dst, nsub, n_used, n_entries, stream=None", "moe_gather_xq (kernels/moe_expert_sort.cpp:81-95)"),
    REIN_DEF(moe_quantize_scatter, "x, inv, xq_dst, in_dim, n_used, n_tok, stream=None",
             "quantize_q8 + moe_gather_xq in one launch (inv = inverse of the sort's perm)"),
    REIN_DEF(moe_scatter_rows, "src, perm, dst, dim, n_entries, stream=None", "moe_scatter_rows (kernels/moe_expert_sort.cpp:96-110)"),
    REIN_DEF(moe_grouped_gemm, "fmt, slab, bytes_per_expert, expert_off, tile_off, n_expert, xq, y, in_dim, out_dim, n_entries, stream=None",
             "launch_moe_grouped_gemm (src/runtime/qwen35.rs:3036-3064)"),
    REIN_DEF(moe_grouped_swiglu_q8,
             "fmt, gate_slab, up_slab, bytes_per_expert, expert_off, tile_off, n_expert, xq, xq_out, in_dim, out_dim, n_entries, stream=None",
             "gate + up grouped GEMM with SwiGLU and the BlockQ8 quantizer in the epilogue"),
    REIN_DEF(moe_expert_matvec,
             "fmt, slab, ids, xq, y, in_dim, out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok=1, stream=None",
             "launch_moe_expert_matvec (src/runtime/qwen35.rs:3071-3100)"),
    REIN_DEF(moe_down, "fmt, slab, ids, xq, y, in_dim, out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok=1, stream=None",
             "launch_moe_down (src/runtime/qwen35.rs:3102-3139)"),
    REIN_DEF(moe_gate_up_swiglu,
             "fmt, gate_slab, up_slab, ids, xq, y, in_dim, out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok=1, stream=None",
             "launch_moe_gate_up_swiglu (src/runtime/qwen35.rs:3141-3167)"),
    REIN_DEF(moe_gate_up_swiglu_q8,
             "fmt, gate_slab, up_slab, ids, xq, xq_out, in_dim, out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok=1, stream=None",
             "moe_gate_up_swiglu followed by quantize_q8 in one launch (BlockQ8 rows of the down projection's input)"),
    REIN_DEF(moe_down_combine,
             "fmt, slab, ids, weights, down_exps_s, xq, out, in_dim, out_dim, bytes_per_expert, xq_tok_stride, xq_slot_stride, n_used, n_tok=1, stream=None",
             "moe_down followed by moe_combine in one launch"),
    REIN_DEF(swiglu_mul, "gate, up, out, n, stream=None", "swiglu_mul_f32 (kernels/swiglu.cpp:10-21)"),
    REIN_DEF(moe_combine, "experts, ids, weights, down_exps_s, out, n_tok, hidden, n_used, stream=None", "moe_combine_f32 (kernels/moe_combine.cpp:15-38)"),
    REIN_DEF(moe_ffn, "shape, x, logits, gate_exps, up_exps, down_exps, down_exps_s, workspace, out, stream=None",
             "routed-expert part of step_moe_ffn_batched (src/runtime/qwen35.rs:2788-2870)"),
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_native", "The launch calls of reinstinct_amd.runtime.", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void)
{
    PyObject *lib = PyImport_ImportModule("reinstinct_amd._lib"), *ctypes = PyImport_ImportModule("ctypes");
    if (!lib || !ctypes) return nullptr;
    const auto take = [](PyObject* m, const char* name, PyObject** to) { return (*to = PyObject_GetAttrString(m, name)) != nullptr; };
    const bool ok = take(lib, "check", &g_check) && take(lib, "MoeShape", &g_shape) && take(ctypes, "cast", &g_cast) &&
                    take(ctypes, "c_void_p", &g_void_p) && take(ctypes, "c_int", &g_int) && take(ctypes, "c_uint", &g_uint) &&
                    take(ctypes, "c_size_t", &g_size) && take(ctypes, "c_float", &g_float);
    Py_DECREF(lib);
    Py_DECREF(ctypes);
    if (!ok) return nullptr;
    g_as_parameter = PyUnicode_InternFromString("_as_parameter_");
    g_value = PyUnicode_InternFromString("value");
    g_raw = PyUnicode_InternFromString("raw");
    PyObject *one = PyLong_FromLong(1), *eps = PyFloat_FromDouble(1e-6);
    if (!g_as_parameter || !g_value || !g_raw || !one || !eps) return nullptr;
    g_none[0] = g_one_none[1] = g_one_eps_none[2] = g_eps_none[1] = Py_None;
    g_one_none[0] = g_one_eps_none[0] = one;
    g_one_eps_none[1] = g_eps_none[0] = eps;
    return PyModule_Create(&g_module);
}
