/*
 * fastcall.c — the per-call half of the Python binding, as a CPython extension.
 *
 * A step of a serving loop is a handful of calls per layer, and a small one
 * runs on the GPU in less time than the interpreter needs to read a dozen
 * tensors and fill ctypes structures (append + decode of 4 sequences: 15 us on
 * the host for 12 us of kernels).  Each function here reads its tensors'
 * attributes, fills the parameter structures of vllm_kv_amd.h and calls the
 * library through the addresses that bind() was given; the return value is the
 * library's status.  Argument rules are those of the ctypes structures in
 * vllm_kv_amd (append_params, decode_params, prefill_params).
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "vllm_kv_amd.h"

static PyObject *s_data_ptr, *s_shape, *s_stride, *s_dtype, *s_is_cuda, *s_numel, *s_element_size;
static PyObject *d_f32, *d_f16, *d_u8, *d_fp8;
static PyObject *c_device, *c_stream;  /* () -> current device, (device) -> its current raw stream */

static int (*f_append)(const vkv_append_params*, vkv_stream_t);
static int (*f_decode)(const vkv_decode_params*, vkv_stream_t);
static int (*f_decode_append)(const vkv_append_params*, const vkv_decode_params*, vkv_stream_t);
static int (*f_prefill)(const vkv_prefill_params*, vkv_stream_t);
static int (*f_rope)(const vkv_rope_append_params*, vkv_stream_t);

/* The device address of a tensor on the GPU (None: NULL); -1 with an exception set. */
static int gpu_ptr(PyObject* t, const void** out) {
    PyObject* r;
    int on;
    *out = NULL;
    if (t == Py_None) return 0;
    if (!(r = PyObject_GetAttr(t, s_is_cuda))) return -1;
    on = PyObject_IsTrue(r);
    Py_DECREF(r);
    if (on < 0) return -1;
    if (!on) {
        PyErr_SetString(PyExc_ValueError, "all tensors must be on the GPU");
        return -1;
    }
    if (!(r = PyObject_CallMethodNoArgs(t, s_data_ptr))) return -1;
    *out = PyLong_AsVoidPtr(r);
    Py_DECREF(r);
    return PyErr_Occurred() ? -1 : 0;
}

static int dtype_code(PyObject* t) {
    PyObject* d = PyObject_GetAttr(t, s_dtype);
    int code = -1;
    if (!d) return -1;
    if (d == d_f16) code = VKV_DTYPE_F16;
    else if (d == d_f32) code = VKV_DTYPE_F32;
    else if (d == d_u8 || d == d_fp8) code = VKV_DTYPE_FP8_E4M3;
    else PyErr_Format(PyExc_TypeError, "unsupported dtype %S", d);
    Py_DECREF(d);
    return code;
}

/* Up to n leading sizes of a tensor with exactly `rank` dimensions (0: any). */
static int sizes(PyObject* t, int rank, int n, int64_t* out) {
    PyObject* s = PyObject_GetAttr(t, s_shape);
    if (!s) return -1;
    if (!PyTuple_Check(s) || PyTuple_GET_SIZE(s) < n || (rank && PyTuple_GET_SIZE(s) != rank)) {
        PyErr_SetString(rank ? PyExc_ValueError : PyExc_IndexError, "a tensor has the wrong number of dimensions");
        Py_DECREF(s);
        return -1;
    }
    for (int i = 0; i < n; ++i) out[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(s, i));
    Py_DECREF(s);
    return PyErr_Occurred() ? -1 : 0;
}

static int stride0(PyObject* t, int64_t* out) {
    PyObject* s = PyObject_CallMethodNoArgs(t, s_stride);
    if (!s) return -1;
    if (!PyTuple_Check(s) || PyTuple_GET_SIZE(s) < 1) {
        PyErr_SetString(PyExc_IndexError, "a tensor has no dimensions");
        Py_DECREF(s);
        return -1;
    }
    *out = PyLong_AsLongLong(PyTuple_GET_ITEM(s, 0));
    Py_DECREF(s);
    return PyErr_Occurred() ? -1 : 0;
}

static int workspace(PyObject* t, void** p, size_t* bytes) {
    const void* q;
    PyObject *n, *e;
    *bytes = 0;
    if (gpu_ptr(t, &q)) return -1;
    *p = (void*)q;
    if (t == Py_None) return 0;
    n = PyObject_CallMethodNoArgs(t, s_numel);
    e = n ? PyObject_CallMethodNoArgs(t, s_element_size) : NULL;
    if (e) *bytes = (size_t)(PyLong_AsLongLong(n) * PyLong_AsLongLong(e));
    Py_XDECREF(n);
    Py_XDECREF(e);
    return PyErr_Occurred() ? -1 : 0;
}

/* A raw stream handle, or None: the current stream of the current device. */
static int stream_of(PyObject* o, vkv_stream_t* out) {
    PyObject *dev, *h;
    if (o != Py_None) {
        *out = (vkv_stream_t)PyLong_AsVoidPtr(o);
        return PyErr_Occurred() ? -1 : 0;
    }
    if (!(dev = PyObject_CallNoArgs(c_device))) return -1;
    h = PyObject_CallOneArg(c_stream, dev);
    Py_DECREF(dev);
    if (!h) return -1;
    *out = (vkv_stream_t)PyLong_AsVoidPtr(h);
    Py_DECREF(h);
    return PyErr_Occurred() ? -1 : 0;
}

/* int32 parameter from a Python int (its low 32 bits, as ctypes takes it) */
static int int32_of(PyObject* o, int32_t* out) {
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) return -1;
    *out = (int32_t)v;
    return 0;
}

static int fill_append(vkv_append_params* p, PyObject* key, PyObject* value, PyObject* kc, PyObject* vc, PyObject* slots,
                       PyObject* ks, PyObject* vs) {
    int64_t c[4], t[1];
    const void* q;
    int a, b;
    memset(p, 0, sizeof(*p));
    if (gpu_ptr(key, &p->key) || gpu_ptr(value, &p->value)) return -1;
    if (gpu_ptr(kc, &q)) return -1;
    p->key_cache = (void*)q;
    if (gpu_ptr(vc, &q)) return -1;
    p->value_cache = (void*)q;
    if (gpu_ptr(slots, &q)) return -1;
    p->slot_mapping = (const int32_t*)q;
    if (gpu_ptr(ks, &q)) return -1;
    p->key_scales = (float*)q;
    if (gpu_ptr(vs, &q)) return -1;
    p->value_scales = (float*)q;
    if (sizes(key, 0, 1, t) || sizes(kc, 4, 4, c) || stride0(key, &p->key_stride) || stride0(value, &p->value_stride)) return -1;
    if ((a = dtype_code(key)) < 0 || (b = dtype_code(kc)) < 0) return -1;
    p->num_tokens = (int32_t)t[0];
    p->num_blocks = (int32_t)c[0];
    p->block_size = (int32_t)c[1];
    p->num_kv_heads = (int32_t)c[2];
    p->head_dim = (int32_t)c[3];
    p->src_dtype = a;
    p->cache_dtype = b;
    return 0;
}

static int fill_decode(vkv_decode_params* p, PyObject* out, PyObject* query, PyObject* kc, PyObject* vc, PyObject* tables,
                       PyObject* lens, PyObject* scale, PyObject* ks, PyObject* vs, PyObject* max_ctx, PyObject* accumulate,
                       PyObject* partition, PyObject* ws) {
    int64_t c[4], o[3], m[2];
    const void* q;
    int a, b, acc;
    memset(p, 0, sizeof(*p));
    if (gpu_ptr(out, &q)) return -1;
    p->output = (void*)q;
    if (gpu_ptr(query, &p->query) || gpu_ptr(kc, &p->key_cache) || gpu_ptr(vc, &p->value_cache)) return -1;
    if (gpu_ptr(tables, &q)) return -1;
    p->block_tables = (const int32_t*)q;
    if (gpu_ptr(lens, &q)) return -1;
    p->context_lens = (const int32_t*)q;
    if (gpu_ptr(ks, &q)) return -1;
    p->key_scales = (const float*)q;
    if (gpu_ptr(vs, &q)) return -1;
    p->value_scales = (const float*)q;
    if (workspace(ws, &p->workspace, &p->workspace_bytes)) return -1;
    if (sizes(out, 3, 3, o) || sizes(kc, 4, 4, c) || sizes(tables, 0, 2, m) || stride0(query, &p->query_stride)) return -1;
    if ((a = dtype_code(out)) < 0 || (b = dtype_code(kc)) < 0 || (acc = PyObject_IsTrue(accumulate)) < 0) return -1;
    p->num_seqs = (int32_t)o[0];
    p->num_heads = (int32_t)o[1];
    p->head_dim = (int32_t)o[2];
    p->num_blocks = (int32_t)c[0];
    p->block_size = (int32_t)c[1];
    p->num_kv_heads = (int32_t)c[2];
    p->max_blocks_per_seq = (int32_t)m[1];
    p->max_context_len = (int32_t)(m[1] * c[1]);
    if (max_ctx != Py_None && int32_of(max_ctx, &p->max_context_len)) return -1;
    if (int32_of(partition, &p->partition_size)) return -1;
    p->scale = (float)PyFloat_AsDouble(scale);
    p->io_dtype = a;
    p->kv_dtype = b;
    p->accumulate = acc;
    return PyErr_Occurred() ? -1 : 0;
}

#define ARGS(n)                                                                  \
    if (nargs != (n)) {                                                          \
        PyErr_Format(PyExc_TypeError, "%d arguments wanted, got %zd", n, nargs); \
        return NULL;                                                             \
    }
#define CALL(expr)                          \
    do {                                    \
        int rc;                             \
        Py_BEGIN_ALLOW_THREADS rc = (expr); \
        Py_END_ALLOW_THREADS return PyLong_FromLong(rc); \
    } while (0)

/* append(key, value, key_cache, value_cache, slot_mapping, key_scales, value_scales, stream) */
static PyObject* py_append(PyObject* self, PyObject* const* a, Py_ssize_t nargs) {
    vkv_append_params p;
    vkv_stream_t st;
    ARGS(8)
    if (fill_append(&p, a[0], a[1], a[2], a[3], a[4], a[5], a[6]) || stream_of(a[7], &st)) return NULL;
    CALL(f_append(&p, st));
}

/* decode(out, query, key_cache, value_cache, block_tables, context_lens, scale, key_scales, value_scales,
 *        max_context_len, accumulate, partition_size, workspace, stream) */
static PyObject* py_decode(PyObject* self, PyObject* const* a, Py_ssize_t nargs) {
    vkv_decode_params p;
    vkv_stream_t st;
    ARGS(14)
    if (fill_decode(&p, a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9], a[10], a[11], a[12]) ||
        stream_of(a[13], &st))
        return NULL;
    CALL(f_decode(&p, st));
}

/* decode_append(<decode's arguments up to workspace>, key, value, slot_mapping, stream) */
static PyObject* py_decode_append(PyObject* self, PyObject* const* a, Py_ssize_t nargs) {
    vkv_decode_params p;
    vkv_append_params q;
    vkv_stream_t st;
    ARGS(17)
    if (fill_append(&q, a[13], a[14], a[2], a[3], a[15], a[7], a[8]) ||
        fill_decode(&p, a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9], a[10], a[11], a[12]) ||
        stream_of(a[16], &st))
        return NULL;
    CALL(f_decode_append(&q, &p, st));
}

/* prefill(out, query, key_cache, value_cache, block_tables, context_lens, query_start_loc, max_query_len, scale,
 *         key_scales, value_scales, max_context_len, workspace, multi_token_only, work_list, stream) */
static PyObject* py_prefill(PyObject* self, PyObject* const* a, Py_ssize_t nargs) {
    vkv_prefill_params p;
    vkv_stream_t st;
    int64_t c[4], o[3], m[2], s[1];
    const void* q;
    int x, y, multi;
    ARGS(16)
    memset(&p, 0, sizeof(p));
    if (gpu_ptr(a[0], &q)) return NULL;
    p.output = (void*)q;
    if (gpu_ptr(a[1], &p.query) || gpu_ptr(a[2], &p.key_cache) || gpu_ptr(a[3], &p.value_cache)) return NULL;
    if (gpu_ptr(a[4], &q)) return NULL;
    p.block_tables = (const int32_t*)q;
    if (gpu_ptr(a[5], &q)) return NULL;
    p.context_lens = (const int32_t*)q;
    if (gpu_ptr(a[6], &q)) return NULL;
    p.query_start_loc = (const int32_t*)q;
    if (gpu_ptr(a[9], &q)) return NULL;
    p.key_scales = (const float*)q;
    if (gpu_ptr(a[10], &q)) return NULL;
    p.value_scales = (const float*)q;
    if (workspace(a[12], &p.workspace, &p.workspace_bytes)) return NULL;
    if (gpu_ptr(a[14], &q)) return NULL;
    if (q) {
        PyObject* n = PyObject_CallMethodNoArgs(a[14], s_numel);
        if (!n) return NULL;
        p.work_list_words = (int32_t)PyLong_AsLong(n);
        Py_DECREF(n);
        p.work_list = p.work_list_words > 0 ? (const int32_t*)q : NULL;
    }
    if (sizes(a[0], 3, 3, o) || sizes(a[2], 4, 4, c) || sizes(a[4], 0, 2, m) || sizes(a[5], 0, 1, s) ||
        stride0(a[1], &p.query_stride))
        return NULL;
    if ((x = dtype_code(a[0])) < 0 || (y = dtype_code(a[2])) < 0 || (multi = PyObject_IsTrue(a[13])) < 0) return NULL;
    if (int32_of(a[7], &p.max_query_len) || int32_of(a[11], &p.max_context_len) || stream_of(a[15], &st)) return NULL;
    p.scale = (float)PyFloat_AsDouble(a[8]);
    if (PyErr_Occurred()) return NULL;
    p.num_seqs = (int32_t)s[0];
    p.num_query_tokens = (int32_t)o[0];
    p.num_heads = (int32_t)o[1];
    p.head_dim = (int32_t)o[2];
    p.num_blocks = (int32_t)c[0];
    p.block_size = (int32_t)c[1];
    p.num_kv_heads = (int32_t)c[2];
    p.max_blocks_per_seq = (int32_t)m[1];
    p.io_dtype = x;
    p.kv_dtype = y;
    p.multi_token_only = multi;
    CALL(f_prefill(&p, st));
}

/* rope(query, key, value, cos_sin, positions, start_pos, key_cache, value_cache, slot_mapping, key_scales,
 *      value_scales, stream) */
static PyObject* py_rope(PyObject* self, PyObject* const* a, Py_ssize_t nargs) {
    vkv_rope_append_params p;
    vkv_stream_t st;
    int64_t h[3], k[2], c[2] = {0, 0}, t[1];
    const void* q;
    int x, y = VKV_DTYPE_F16;
    ARGS(12)
    memset(&p, 0, sizeof(p));
    if (gpu_ptr(a[0], &q)) return NULL;
    p.query = (void*)q;
    if (gpu_ptr(a[1], &q)) return NULL;
    p.key = (void*)q;
    if (gpu_ptr(a[2], &p.value)) return NULL;
    if (gpu_ptr(a[3], &q)) return NULL;
    p.cos_sin = (const float*)q;
    if (gpu_ptr(a[4], &q)) return NULL;
    p.positions = (const int32_t*)q;
    if (gpu_ptr(a[6], &q)) return NULL;
    p.key_cache = (void*)q;
    if (gpu_ptr(a[7], &q)) return NULL;
    p.value_cache = (void*)q;
    if (gpu_ptr(a[8], &q)) return NULL;
    p.slot_mapping = (const int32_t*)q;
    if (gpu_ptr(a[9], &q)) return NULL;
    p.key_scales = (float*)q;
    if (gpu_ptr(a[10], &q)) return NULL;
    p.value_scales = (float*)q;
    if (sizes(a[0], 3, 3, h) || sizes(a[1], 0, 2, k) || sizes(a[3], 0, 1, t) || stride0(a[0], &p.query_stride) ||
        stride0(a[1], &p.key_stride) || (a[2] != Py_None && stride0(a[2], &p.value_stride)))
        return NULL;
    if (a[6] != Py_None && (sizes(a[6], 0, 2, c) || (y = dtype_code(a[6])) < 0)) return NULL;
    if ((x = dtype_code(a[0])) < 0 || int32_of(a[5], &p.start_pos) || stream_of(a[11], &st)) return NULL;
    p.max_position = (int32_t)t[0];
    p.num_tokens = (int32_t)h[0];
    p.num_heads = (int32_t)h[1];
    p.head_dim = (int32_t)h[2];
    p.num_kv_heads = (int32_t)k[1];
    p.num_blocks = (int32_t)c[0];
    p.block_size = (int32_t)c[1];
    p.src_dtype = x;
    p.cache_dtype = y;
    CALL(f_rope(&p, st));
}

/* bind((append, decode, decode_append, prefill, rope addresses), (float32, float16, uint8, float8_e4m3fn or None),
 *      (current device, current raw stream of a device)) */
static PyObject* py_bind(PyObject* self, PyObject* args) {
    unsigned long long f[5];
    PyObject* d[6];
    if (!PyArg_ParseTuple(args, "(KKKKK)(OOOO)(OO)", &f[0], &f[1], &f[2], &f[3], &f[4], &d[0], &d[1], &d[2], &d[3], &d[4],
                          &d[5]))
        return NULL;
    f_append = (int (*)(const vkv_append_params*, vkv_stream_t))(uintptr_t)f[0];
    f_decode = (int (*)(const vkv_decode_params*, vkv_stream_t))(uintptr_t)f[1];
    f_decode_append = (int (*)(const vkv_append_params*, const vkv_decode_params*, vkv_stream_t))(uintptr_t)f[2];
    f_prefill = (int (*)(const vkv_prefill_params*, vkv_stream_t))(uintptr_t)f[3];
    f_rope = (int (*)(const vkv_rope_append_params*, vkv_stream_t))(uintptr_t)f[4];
    for (int i = 0; i < 6; ++i) Py_INCREF(d[i]);
    d_f32 = d[0];
    d_f16 = d[1];
    d_u8 = d[2];
    d_fp8 = d[3];
    c_device = d[4];
    c_stream = d[5];
    Py_RETURN_NONE;
}

static PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, "library addresses and torch dtypes; once, before any call"},
    {"append", (PyCFunction)(void (*)(void))py_append, METH_FASTCALL, "vkv_reshape_and_cache"},
    {"decode", (PyCFunction)(void (*)(void))py_decode, METH_FASTCALL, "vkv_paged_decode"},
    {"decode_append", (PyCFunction)(void (*)(void))py_decode_append, METH_FASTCALL, "vkv_paged_decode_append"},
    {"prefill", (PyCFunction)(void (*)(void))py_prefill, METH_FASTCALL, "vkv_paged_prefill"},
    {"rope", (PyCFunction)(void (*)(void))py_rope, METH_FASTCALL, "vkv_rope_reshape_and_cache"},
    {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_vkv_fastcall", NULL, -1, methods};

PyMODINIT_FUNC PyInit__vkv_fastcall(void) {
    s_data_ptr = PyUnicode_InternFromString("data_ptr");
    s_shape = PyUnicode_InternFromString("shape");
    s_stride = PyUnicode_InternFromString("stride");
    s_dtype = PyUnicode_InternFromString("dtype");
    s_is_cuda = PyUnicode_InternFromString("is_cuda");
    s_numel = PyUnicode_InternFromString("numel");
    s_element_size = PyUnicode_InternFromString("element_size");
    return PyModule_Create(&module);
}
