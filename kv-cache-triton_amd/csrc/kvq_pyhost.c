/*
 * kvq_pyhost.c — the CPython side of the hot operators: calls into
 * libkvint4.so (include/kvint4.h) with arguments taken straight from tensors.
 *
 * A decode step is a 9 us launch whose C entry point takes 31 arguments (35
 * over a paged cache). Built up through ctypes (an array object per stride
 * list, a conversion per argument) an eager step of the cache class cost the
 * host 18.8 us; through this module it costs 9.6, and a prompt's append 21
 * instead of 34.
 *
 * Conventions of every function below: positional arguments; a tensor argument
 * is a torch tensor on the GPU (data_ptr() and stride() are called), a tuple
 * (pointer, strides) where the caller views it under other strides, or None
 * (a null pointer); plain pointers are integers or None; the result is the C
 * entry point's status (kvint4._native.check turns it into an exception, with
 * kvq_last_error() of the same thread). Checked here are the number of
 * arguments, their types and the tensors' device; the checks of values that a caller relies on are
 * the Python operator's and the C entry point's. The GIL is released around the
 * launch, as ctypes does.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <stdint.h>

#include "../../include/kvint4.h"

static PyObject *s_data_ptr, *s_stride, *s_is_cuda, *s_is_pinned;

typedef struct {
  void *p;
  int64_t st[4];
} tensor_arg;

/* Strides of `t` (at least n of them wanted) into out; -1 on error. */
static int read_strides(PyObject *t, int64_t *out, Py_ssize_t n) {
  if (!PyTuple_Check(t) || PyTuple_GET_SIZE(t) < n) {
    PyErr_Format(PyExc_ValueError, "expected at least %zd strides", n);
    return -1;
  }
  for (Py_ssize_t i = 0; i < n; ++i) {
    out[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(t, i));
    if (out[i] == -1 && PyErr_Occurred()) return -1;
  }
  return 0;
}

static int read_pointer(PyObject *o, void **p) {
  if (o == Py_None) {
    *p = NULL;
    return 0;
  }
  *p = PyLong_AsVoidPtr(o);
  return *p == NULL && PyErr_Occurred() ? -1 : 0;
}

static int read_tensor(PyObject *o, tensor_arg *a, Py_ssize_t n) {
  a->p = NULL;
  for (int i = 0; i < 4; ++i) a->st[i] = 0;
  if (o == Py_None) return 0;
  if (PyTuple_Check(o)) {
    if (PyTuple_GET_SIZE(o) != 2) {
      PyErr_SetString(PyExc_ValueError, "expected (pointer, strides)");
      return -1;
    }
    if (read_pointer(PyTuple_GET_ITEM(o, 0), &a->p) < 0) return -1;
    return read_strides(PyTuple_GET_ITEM(o, 1), a->st, n);
  }
  PyObject *p = PyObject_CallMethodNoArgs(o, s_data_ptr);
  if (p == NULL) return -1;
  const int rp = read_pointer(p, &a->p);
  Py_DECREF(p);
  if (rp < 0) return -1;
  /* a host pointer would fault the GPU at the kernel's first read (pinned memory, which it can read, does not) */
  PyObject *gpu = PyObject_GetAttr(o, s_is_cuda);
  if (gpu != NULL && gpu != Py_True) {
    Py_DECREF(gpu);
    gpu = PyObject_CallMethodNoArgs(o, s_is_pinned);
  }
  if (gpu == NULL) return -1;
  const int reachable = gpu == Py_True;
  Py_DECREF(gpu);
  if (!reachable) {
    PyErr_SetString(PyExc_ValueError, "expected GPU tensors (got one in host memory)");
    return -1;
  }
  PyObject *st = PyObject_CallMethodNoArgs(o, s_stride);
  if (st == NULL) return -1;
  const int rs = read_strides(st, a->st, n);
  Py_DECREF(st);
  return rs;
}

static int read_ints(PyObject *const *args, Py_ssize_t n, int64_t *out) {
  for (Py_ssize_t i = 0; i < n; ++i) {
    out[i] = PyLong_AsLongLong(args[i]);
    if (out[i] == -1 && PyErr_Occurred()) return -1;
  }
  return 0;
}

static int read_float(PyObject *o, float *f) {
  const double d = PyFloat_AsDouble(o);
  if (d == -1.0 && PyErr_Occurred()) return -1;
  *f = (float)d;
  return 0;
}

/* A block table's (pointer, row stride, columns, blocks, page size). */
typedef struct {
  void *bt;
  int64_t g[4];
} table_arg;

static int read_table(PyObject *o, table_arg *t) {
  if (!PyTuple_Check(o) || PyTuple_GET_SIZE(o) != 5) {
    PyErr_SetString(PyExc_ValueError, "expected a block table's five arguments");
    return -1;
  }
  if (read_pointer(PyTuple_GET_ITEM(o, 0), &t->bt) < 0) return -1;
  for (int i = 0; i < 4; ++i) {
    t->g[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(o, i + 1));
    if (t->g[i] == -1 && PyErr_Occurred()) return -1;
  }
  return 0;
}

#define WANT(n)                                                                                  \
  if (nargs != (n)) return PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", (n), nargs)
#define TENSOR(name, i, n) \
  tensor_arg name;         \
  if (read_tensor(args[i], &name, n) < 0) return NULL
#define POINTER(name, i) \
  void *name;            \
  if (read_pointer(args[i], &name) < 0) return NULL
#define INTS(name, i, n) \
  int64_t name[n];       \
  if (read_ints(args + (i), n, name) < 0) return NULL
#define FLOAT(name, i) \
  float name;          \
  if (read_float(args[i], &name) < 0) return NULL
#define TABLE(name, i) \
  table_arg name;      \
  if (read_table(args[i], &name) < 0) return NULL
#define CALL(expr)         \
  int rc;                  \
  Py_BEGIN_ALLOW_THREADS   \
  rc = (expr);             \
  Py_END_ALLOW_THREADS     \
  return PyLong_FromLong(rc)
#define FN(name) static PyObject *name(PyObject *self, PyObject *const *args, Py_ssize_t nargs)

/* (x, x_dtype, B, H, S, D, G, packed, scales, scale_dtype, write_pos, write_pos0, capacity, stream) */
FN(py_quantize) {
  WANT(14);
  TENSOR(x, 0, 4);
  INTS(s, 1, 6);
  TENSOR(p, 7, 3);
  TENSOR(c, 8, 3);
  INTS(sd, 9, 1);
  POINTER(wp, 10);
  INTS(w, 11, 2);
  POINTER(st, 13);
  CALL(kvq_quantize(x.p, (int)s[0], x.st, s[1], s[2], s[3], s[4], s[5], p.p, p.st, c.p, (int)sd[0], c.st,
                    (const int32_t *)wp, w[0], w[1], st));
}

/* (k, v, x_dtype, B, H, S, D, G, k_packed, k_scales, v_packed, v_scales, scale_dtype, write_pos, write_pos0,
   capacity, stream) */
FN(py_quantize_kv) {
  WANT(17);
  TENSOR(k, 0, 4);
  TENSOR(v, 1, 4);
  INTS(s, 2, 6);
  TENSOR(kp, 8, 3);
  TENSOR(ks, 9, 3);
  TENSOR(vp, 10, 3);
  TENSOR(vs, 11, 3);
  INTS(sd, 12, 1);
  POINTER(wp, 13);
  INTS(w, 14, 2);
  POINTER(st, 16);
  CALL(kvq_quantize_kv(k.p, k.st, v.p, v.st, (int)s[0], s[1], s[2], s[3], s[4], s[5], kp.p, kp.st, ks.p, ks.st, vp.p,
                       vp.st, vs.p, vs.st, (int)sd[0], (const int32_t *)wp, w[0], w[1], st));
}

/* (x, x_dtype, B, H, S, D, G, pool, scales, scale_dtype, table, write_pos, write_pos0, stream) */
FN(py_quantize_paged) {
  WANT(14);
  TENSOR(x, 0, 4);
  INTS(s, 1, 6);
  TENSOR(p, 7, 2);
  TENSOR(c, 8, 2);
  INTS(sd, 9, 1);
  TABLE(t, 10);
  POINTER(wp, 11);
  INTS(w, 12, 1);
  POINTER(st, 13);
  CALL(kvq_quantize_paged(x.p, (int)s[0], x.st, s[1], s[2], s[3], s[4], s[5], p.p, p.st, c.p, (int)sd[0], c.st,
                          (const int32_t *)t.bt, t.g[0], t.g[1], t.g[2], t.g[3], (const int32_t *)wp, w[0], st));
}

/* (k, v, x_dtype, B, H, S, D, G, k_pool, k_scales, v_pool, v_scales, scale_dtype, table, write_pos, write_pos0, stream) */
FN(py_quantize_kv_paged) {
  WANT(17);
  TENSOR(k, 0, 4);
  TENSOR(v, 1, 4);
  INTS(s, 2, 6);
  TENSOR(kp, 8, 2);
  TENSOR(ks, 9, 2);
  TENSOR(vp, 10, 2);
  TENSOR(vs, 11, 2);
  INTS(sd, 12, 1);
  TABLE(t, 13);
  POINTER(wp, 14);
  INTS(w, 15, 1);
  POINTER(st, 16);
  CALL(kvq_quantize_kv_paged(k.p, k.st, v.p, v.st, (int)s[0], s[1], s[2], s[3], s[4], s[5], kp.p, kp.st, ks.p, ks.st,
                             vp.p, vp.st, vs.p, vs.st, (int)sd[0], (const int32_t *)t.bt, t.g[0], t.g[1], t.g[2],
                             t.g[3], (const int32_t *)wp, w[0], st));
}

/* (packed, scales, scale_dtype, B, H, S, G, groups, out, out_dtype, d_out, stream) */
FN(py_dequantize) {
  WANT(12);
  TENSOR(p, 0, 3);
  TENSOR(c, 1, 3);
  INTS(s, 2, 6);
  TENSOR(o, 8, 4);
  INTS(d, 9, 2);
  POINTER(st, 11);
  CALL(kvq_dequantize(p.p, p.st, c.p, (int)s[0], c.st, s[1], s[2], s[3], s[4], s[5], o.p, (int)d[0], o.st, d[1], st));
}

/* (pool, scales, scale_dtype, table, B, H, S, G, groups, out, out_dtype, d_out, stream) */
FN(py_dequantize_paged) {
  WANT(13);
  TENSOR(p, 0, 2);
  TENSOR(c, 1, 2);
  INTS(sd, 2, 1);
  TABLE(t, 3);
  INTS(s, 4, 5);
  TENSOR(o, 9, 4);
  INTS(d, 10, 2);
  POINTER(st, 12);
  CALL(kvq_dequantize_paged(p.p, p.st, c.p, (int)sd[0], c.st, (const int32_t *)t.bt, t.g[0], t.g[1], t.g[2], t.g[3],
                            s[0], s[1], s[2], s[3], s[4], o.p, (int)d[0], o.st, d[1], st));
}

/* (B, Hq, Hkv, Sq, D, s_max, q_dtype, scale_dtype, num_cus, n_split or 0, whether the call has device lengths) ->
   (n_split, workspace bytes), either negative: a status of kvq_decode_attn_num_splits or
   kvq_decode_attn_workspace_bytes */
FN(py_plan) {
  WANT(11);
  INTS(s, 0, 11);
  int64_t n = s[9], w = 0;
  if (n < 1 && s[10]) {
    w = kvq_decode_attn_by_length_workspace_bytes(s[0], s[1], s[2], s[3], s[4], s[5], (int)s[6], (int)s[7]);
    if (w > 0) return Py_BuildValue("LL", (long long)KVQ_SPLIT_BY_LENGTH, (long long)w);
    w = 0;
  }
  if (n < 1) n = kvq_decode_attn_num_splits(s[0], s[1], s[2], s[3], s[4], s[5], (int)s[6], (int)s[7], s[8]);
  if (n > 0) w = kvq_decode_attn_workspace_bytes(s[0], s[1], s[2], s[3], s[4], (int)s[6], (int)s[7], n);
  return Py_BuildValue("LL", (long long)n, (long long)w);
}

/* (q, q_dtype, k_packed, k_scales, v_packed, v_scales, scale_dtype, out, B, Hq, Hkv, Sq, D, G, Sk, seq_lens, causal,
   sm_scale, n_split, workspace, workspace_bytes, stream) */
FN(py_decode_attn) {
  WANT(22);
  TENSOR(q, 0, 4);
  INTS(qd, 1, 1);
  TENSOR(kp, 2, 3);
  TENSOR(ks, 3, 3);
  TENSOR(vp, 4, 3);
  TENSOR(vs, 5, 3);
  INTS(sd, 6, 1);
  TENSOR(o, 7, 4);
  INTS(s, 8, 7);
  POINTER(sl, 15);
  INTS(c, 16, 1);
  FLOAT(f, 17);
  INTS(ns, 18, 1);
  POINTER(ws, 19);
  INTS(wb, 20, 1);
  POINTER(st, 21);
  CALL(kvq_decode_attn(q.p, (int)qd[0], q.st, kp.p, kp.st, ks.p, ks.st, vp.p, vp.st, vs.p, vs.st, (int)sd[0], o.p,
                       o.st, s[0], s[1], s[2], s[3], s[4], s[5], s[6], (const int32_t *)sl, (int)c[0], f, ns[0], ws,
                       wb[0], st));
}

/* (q, q_dtype, k_pool, k_scales, v_pool, v_scales, scale_dtype, table, out, B, Hq, Hkv, Sq, D, G, seq_lens, seq_len,
   causal, sm_scale, n_split, workspace, workspace_bytes, stream) */
FN(py_decode_attn_paged) {
  WANT(23);
  TENSOR(q, 0, 4);
  INTS(qd, 1, 1);
  TENSOR(kp, 2, 2);
  TENSOR(ks, 3, 2);
  TENSOR(vp, 4, 2);
  TENSOR(vs, 5, 2);
  INTS(sd, 6, 1);
  TABLE(t, 7);
  TENSOR(o, 8, 4);
  INTS(s, 9, 6);
  POINTER(sl, 15);
  INTS(c, 16, 2);
  FLOAT(f, 18);
  INTS(ns, 19, 1);
  POINTER(ws, 20);
  INTS(wb, 21, 1);
  POINTER(st, 22);
  CALL(kvq_decode_attn_paged(q.p, (int)qd[0], q.st, kp.p, kp.st, ks.p, ks.st, vp.p, vp.st, vs.p, vs.st, (int)sd[0],
                             (const int32_t *)t.bt, t.g[0], t.g[1], t.g[2], t.g[3], o.p, o.st, s[0], s[1], s[2], s[3],
                             s[4], s[5], (const int32_t *)sl, c[0], (int)c[1], f, ns[0], ws, wb[0], st));
}

/* (q, q_dtype, k_new, v_new, k_packed, k_scales, v_packed, v_scales, scale_dtype, out, B, Hq, Hkv, D, G, capacity,
   positions, pos0, sm_scale, n_split, workspace, workspace_bytes, stream) */
FN(py_decode_step) {
  WANT(23);
  TENSOR(q, 0, 4);
  INTS(qd, 1, 1);
  TENSOR(kn, 2, 4);
  TENSOR(vn, 3, 4);
  TENSOR(kp, 4, 3);
  TENSOR(ks, 5, 3);
  TENSOR(vp, 6, 3);
  TENSOR(vs, 7, 3);
  INTS(sd, 8, 1);
  TENSOR(o, 9, 4);
  INTS(s, 10, 6);
  POINTER(pp, 16);
  INTS(p0, 17, 1);
  FLOAT(f, 18);
  INTS(ns, 19, 1);
  POINTER(ws, 20);
  INTS(wb, 21, 1);
  POINTER(st, 22);
  CALL(kvq_decode_step(q.p, (int)qd[0], q.st, kn.p, kn.st, vn.p, vn.st, kp.p, kp.st, ks.p, ks.st, vp.p, vp.st, vs.p,
                       vs.st, (int)sd[0], o.p, o.st, s[0], s[1], s[2], s[3], s[4], s[5], (const int32_t *)pp, p0[0], f,
                       ns[0], ws, wb[0], st));
}

/* (q, q_dtype, k_new, v_new, k_pool, k_scales, v_pool, v_scales, scale_dtype, table, out, B, Hq, Hkv, D, G, positions,
   pos0, sm_scale, n_split, workspace, workspace_bytes, stream) */
FN(py_decode_step_paged) {
  WANT(23);
  TENSOR(q, 0, 4);
  INTS(qd, 1, 1);
  TENSOR(kn, 2, 4);
  TENSOR(vn, 3, 4);
  TENSOR(kp, 4, 2);
  TENSOR(ks, 5, 2);
  TENSOR(vp, 6, 2);
  TENSOR(vs, 7, 2);
  INTS(sd, 8, 1);
  TABLE(t, 9);
  TENSOR(o, 10, 4);
  INTS(s, 11, 5);
  POINTER(pp, 16);
  INTS(p0, 17, 1);
  FLOAT(f, 18);
  INTS(ns, 19, 1);
  POINTER(ws, 20);
  INTS(wb, 21, 1);
  POINTER(st, 22);
  CALL(kvq_decode_step_paged(q.p, (int)qd[0], q.st, kn.p, kn.st, vn.p, vn.st, kp.p, kp.st, ks.p, ks.st, vp.p, vp.st,
                             vs.p, vs.st, (int)sd[0], (const int32_t *)t.bt, t.g[0], t.g[1], t.g[2], t.g[3], o.p, o.st,
                             s[0], s[1], s[2], s[3], s[4], (const int32_t *)pp, p0[0], f, ns[0], ws, wb[0], st));
}

/* (q, q_dtype, k_packed, k_scales, v_packed, v_scales, scale_dtype, out, B, Hq, Hkv, Sq, D, G, Sk, causal, sm_scale,
   workspace, workspace_bytes, stream) */
FN(py_prefill_attn) {
  WANT(20);
  TENSOR(q, 0, 4);
  INTS(qd, 1, 1);
  TENSOR(kp, 2, 3);
  TENSOR(ks, 3, 3);
  TENSOR(vp, 4, 3);
  TENSOR(vs, 5, 3);
  INTS(sd, 6, 1);
  TENSOR(o, 7, 4);
  INTS(s, 8, 8);
  FLOAT(f, 16);
  POINTER(ws, 17);
  INTS(wb, 18, 1);
  POINTER(st, 19);
  CALL(kvq_prefill_attn(q.p, (int)qd[0], q.st, kp.p, kp.st, ks.p, ks.st, vp.p, vp.st, vs.p, vs.st, (int)sd[0], o.p,
                        o.st, s[0], s[1], s[2], s[3], s[4], s[5], s[6], (int)s[7], f, ws, wb[0], st));
}

/* (q, q_dtype, k_pool, k_scales, v_pool, v_scales, scale_dtype, table, out, B, Hq, Hkv, Sq, D, G, Sk, causal, sm_scale,
   workspace, workspace_bytes, stream) */
FN(py_prefill_attn_paged) {
  WANT(21);
  TENSOR(q, 0, 4);
  INTS(qd, 1, 1);
  TENSOR(kp, 2, 2);
  TENSOR(ks, 3, 2);
  TENSOR(vp, 4, 2);
  TENSOR(vs, 5, 2);
  INTS(sd, 6, 1);
  TABLE(t, 7);
  TENSOR(o, 8, 4);
  INTS(s, 9, 8);
  FLOAT(f, 17);
  POINTER(ws, 18);
  INTS(wb, 19, 1);
  POINTER(st, 20);
  CALL(kvq_prefill_attn_paged(q.p, (int)qd[0], q.st, kp.p, kp.st, ks.p, ks.st, vp.p, vp.st, vs.p, vs.st, (int)sd[0],
                              (const int32_t *)t.bt, t.g[0], t.g[1], t.g[2], t.g[3], o.p, o.st, s[0], s[1], s[2], s[3],
                              s[4], s[5], s[6], (int)s[7], f, ws, wb[0], st));
}

#define ENTRY(name) {#name, (PyCFunction)(void (*)(void))py_##name, METH_FASTCALL, NULL}
static PyMethodDef methods[] = {
    ENTRY(quantize),          ENTRY(quantize_kv),    ENTRY(quantize_paged),    ENTRY(quantize_kv_paged),
    ENTRY(dequantize),        ENTRY(dequantize_paged), ENTRY(plan),            ENTRY(decode_attn),
    ENTRY(decode_attn_paged), ENTRY(decode_step),    ENTRY(decode_step_paged), ENTRY(prefill_attn),
    ENTRY(prefill_attn_paged), {NULL, NULL, 0, NULL}};

static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_kvq_host", "libkvint4.so's entry points, taking tensors.",
                                    -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__kvq_host(void) {
  s_data_ptr = PyUnicode_InternFromString("data_ptr");
  s_stride = PyUnicode_InternFromString("stride");
  s_is_cuda = PyUnicode_InternFromString("is_cuda");
  s_is_pinned = PyUnicode_InternFromString("is_pinned");
  if (s_data_ptr == NULL || s_stride == NULL || s_is_cuda == NULL || s_is_pinned == NULL) return NULL;
  return PyModule_Create(&module);
}
