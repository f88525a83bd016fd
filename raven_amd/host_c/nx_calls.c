/* nx_calls.c — the per-primitive host path of raven_amd.nx_backend, in C.
 *
 * A primitive over small tensors is its host path: allocate the result, describe the operands,
 * call the library, give the storage of what has died back. In Python that was 2.1 us of an
 * elementwise call's 5.1 (the launch is 2.7), more for a scalar or a broadcast operand. Here the
 * handles are C objects, a descriptor is copied out of its view's image onto the stack, and the
 * allocation and the call run without the interpreter lock, as ctypes ran them.
 *
 * Types
 *   DeviceBuffer  one allocation of a context, given back when the last handle goes
 *   Tensor        buffer, view, dtype, context (nx_backend.ml:36-43)
 *   Calls         the base class of Backend: unary, binary, compare, where, cast, copy, assign, full,
 *                 reduce, matmul; and what the frontend makes of them over operands that broadcast:
 *                 broadcast_binary, broadcast_where, reduce_keep. A call whose arguments are out of the ordinary (axes that are no
 *                 plain integers, batches that broadcast, ...) goes to the Python method of the same
 *                 name with `_general` behind it.
 */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

#include <stdint.h>
#include <string.h>

#include "nxhip.h"

static struct {
  int (*alloc)(nxh_context *, size_t, void **);
  int (*free)(nxh_context *, void *);
  int (*fill)(nxh_context *, const nxh_tensor *, const void *);
  int (*unary)(nxh_context *, int, const nxh_tensor *, const nxh_tensor *);
  int (*binary)(nxh_context *, int, const nxh_tensor *, const nxh_tensor *, const nxh_tensor *);
  int (*compare)(nxh_context *, int, const nxh_tensor *, const nxh_tensor *, const nxh_tensor *);
  int (*where)(nxh_context *, const nxh_tensor *, const nxh_tensor *, const nxh_tensor *, const nxh_tensor *);
  int (*cast)(nxh_context *, const nxh_tensor *, const nxh_tensor *);
  int (*copy)(nxh_context *, const nxh_tensor *, const nxh_tensor *);
  int (*reduce)(nxh_context *, int, const nxh_tensor *, const nxh_tensor *, const int32_t *, int);
  int (*matmul)(nxh_context *, const nxh_tensor *, const nxh_tensor *, const nxh_tensor *);
} L;

/* what setup() hands over from Python */
static PyObject *contiguous_views, *view_create, *view_image, *stamp, *encode_scalar, *ndarray_type, *bool_dtype;
static PyObject *op_unary, *op_binary, *op_compare, *op_reduce;
static PyObject *s_image, *s_shape, *s_strides, *s_offset, *s_tag, *s_itemsize, *s_packed, *s_desc, *s_dtype, *s_name;

/* ── contexts ─────────────────────────────────────────────────────────────── */
typedef struct {
  PyObject_HEAD
  nxh_context *h; /* NULL: closed */
} Calls;
static PyTypeObject CallsType, BufferType, TensorType;

static PyObject *calls_get_h(Calls *self, void *u) {
  (void)u;
  if (!self->h) Py_RETURN_NONE;
  return PyLong_FromVoidPtr(self->h);
}
static int calls_set_h(Calls *self, PyObject *v, void *u) {
  (void)u;
  if (!v || v == Py_None) {
    self->h = NULL;
    return 0;
  }
  void *p = PyLong_AsVoidPtr(v);
  if (!p && PyErr_Occurred()) return -1;
  self->h = p;
  return 0;
}

/* ── storage ──────────────────────────────────────────────────────────────── */
typedef struct {
  PyObject_HEAD
  PyObject *ctx;
  void *ptr;
  Py_ssize_t nbytes;
  PyObject *weak;
} Buffer;

static PyObject *raise_status(PyObject *ctx, int rc) {
  PyObject *r = PyObject_CallMethod(ctx, "_check", "i", rc);
  if (r) { /* (a status that _check lets pass would be a result without a call) */
    Py_DECREF(r);
    PyErr_SetString(PyExc_RuntimeError, "call failed");
  }
  return NULL;
}

/* Handles are seen by the cycle collector: a tensor may be kept by its own context. They have nothing to clear; any
   such cycle runs through a dict or the like that has. */
static Buffer *buffer_wrap(PyObject *ctx, void *ptr, Py_ssize_t nbytes) {
  Buffer *b = PyObject_GC_New(Buffer, &BufferType);
  if (!b) {
    nxh_context *h = ((Calls *)ctx)->h;
    if (h) L.free(h, ptr);
    return NULL;
  }
  Py_INCREF(ctx);
  b->ctx = ctx;
  b->ptr = ptr;
  b->nbytes = nbytes;
  b->weak = NULL;
  PyObject_GC_Track(b);
  return b;
}
static PyObject *buffer_new(PyTypeObject *type, PyObject *args, PyObject *kw) {
  (void)type;
  static char *names[] = {"ctx", "nbytes", NULL};
  PyObject *ctx;
  Py_ssize_t nbytes;
  if (!PyArg_ParseTupleAndKeywords(args, kw, "O!n", names, &CallsType, &ctx, &nbytes)) return NULL;
  void *p = NULL;
  nxh_context *h = ((Calls *)ctx)->h;
  int rc;
  Py_BEGIN_ALLOW_THREADS rc = L.alloc(h, (size_t)nbytes, &p);
  Py_END_ALLOW_THREADS
  if (rc) return raise_status(ctx, rc);
  return (PyObject *)buffer_wrap(ctx, p, nbytes);
}
static int buffer_traverse(Buffer *b, visitproc visit, void *arg) {
  Py_VISIT(b->ctx);
  return 0;
}
static void buffer_dealloc(Buffer *b) {
  PyObject_GC_UnTrack(b);
  if (b->weak) PyObject_ClearWeakRefs((PyObject *)b);
  nxh_context *h = b->ctx ? ((Calls *)b->ctx)->h : NULL;
  if (h && b->ptr) {
    /* another thread may be waiting for the device inside the library */
    PyThreadState *t = _Py_IsFinalizing() ? NULL : PyEval_SaveThread();
    L.free(h, b->ptr);
    if (t) PyEval_RestoreThread(t);
  }
  Py_XDECREF(b->ctx);
  PyObject_GC_Del(b);
}
static PyObject *buffer_ptr(Buffer *b, void *u) {
  (void)u;
  if (!b->ptr) Py_RETURN_NONE; /* as a ctypes pointer's value */
  return PyLong_FromVoidPtr(b->ptr);
}
static PyMemberDef buffer_members[] = {{"ctx", T_OBJECT_EX, offsetof(Buffer, ctx), READONLY, NULL},
                                       {"nbytes", T_PYSSIZET, offsetof(Buffer, nbytes), READONLY, NULL},
                                       {NULL, 0, 0, 0, NULL}};
static PyGetSetDef buffer_getset[] = {{"ptr", (getter)buffer_ptr, NULL, NULL, NULL}, {NULL, NULL, NULL, NULL, NULL}};
static PyTypeObject BufferType = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "raven_amd._nxcalls.DeviceBuffer",
    .tp_basicsize = sizeof(Buffer),
    .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC,
    .tp_traverse = (traverseproc)buffer_traverse,
    .tp_doc = "One device allocation, shared by every view of a tensor. Returned to the context's caching\n"
              "allocator when the last handle goes away (the OCaml binding does the same from a\n"
              "custom-block finaliser).",
    .tp_new = buffer_new,
    .tp_dealloc = (destructor)buffer_dealloc,
    .tp_weaklistoffset = offsetof(Buffer, weak),
    .tp_members = buffer_members,
    .tp_getset = buffer_getset,
};

/* ── tensors ──────────────────────────────────────────────────────────────── */
typedef struct {
  PyObject_HEAD
  PyObject *buffer, *view, *shape, *dtype, *context, *d;
} Tensor;

static PyObject *tensor_make(PyObject *buffer, PyObject *view, PyObject *shape, PyObject *dtype, PyObject *context) {
  Tensor *t = PyObject_GC_New(Tensor, &TensorType);
  if (!t) return NULL;
  Py_INCREF(buffer), Py_INCREF(view), Py_INCREF(shape), Py_INCREF(dtype), Py_INCREF(context);
  t->buffer = buffer;
  t->view = view;
  t->shape = shape;
  t->dtype = dtype;
  t->context = context;
  t->d = NULL;
  PyObject_GC_Track(t);
  return (PyObject *)t;
}
static PyObject *tensor_new(PyTypeObject *type, PyObject *args, PyObject *kw) {
  (void)type;
  static char *names[] = {"buffer", "view", "dtype", "context", NULL};
  PyObject *buffer, *view, *dtype, *context;
  if (!PyArg_ParseTupleAndKeywords(args, kw, "OOOO", names, &buffer, &view, &dtype, &context)) return NULL;
  PyObject *shape = PyObject_GetAttr(view, s_shape);
  if (!shape) return NULL;
  PyObject *t = tensor_make(buffer, view, shape, dtype, context);
  Py_DECREF(shape);
  return t;
}
static int tensor_traverse(Tensor *t, visitproc visit, void *arg) {
  Py_VISIT(t->buffer);
  Py_VISIT(t->view);
  Py_VISIT(t->shape);
  Py_VISIT(t->dtype);
  Py_VISIT(t->context);
  Py_VISIT(t->d);
  return 0;
}
static void tensor_dealloc(Tensor *t) {
  PyObject_GC_UnTrack(t);
  Py_XDECREF(t->buffer);
  Py_XDECREF(t->view);
  Py_XDECREF(t->shape);
  Py_XDECREF(t->dtype);
  Py_XDECREF(t->context);
  Py_XDECREF(t->d);
  PyObject_GC_Del(t);
}

/* The bytes of a view's descriptor (storage pointer and dtype tag zero), made once per view. */
static PyObject *image_of(PyObject *view) {
  PyObject *image = PyObject_GetAttr(view, s_image);
  if (!image || image != Py_None) return image;
  Py_DECREF(image);
  PyObject *shape = PyObject_GetAttr(view, s_shape), *strides = PyObject_GetAttr(view, s_strides), *offset = PyObject_GetAttr(view, s_offset);
  image = shape && strides && offset ? PyObject_CallFunctionObjArgs(view_image, shape, strides, offset, NULL) : NULL;
  Py_XDECREF(shape);
  Py_XDECREF(strides);
  Py_XDECREF(offset);
  if (!image) return NULL;
  if (!PyBytes_Check(image) || PyBytes_GET_SIZE(image) != (Py_ssize_t)sizeof(nxh_tensor)) {
    Py_DECREF(image);
    PyErr_SetString(PyExc_RuntimeError, "a view's image has the size of a descriptor");
    return NULL;
  }
  if (PyObject_SetAttr(view, s_image, image)) {
    Py_DECREF(image);
    return NULL;
  }
  return image;
}
/* Copies the part of an image that its rank uses. */
static int describe_view(nxh_tensor *d, PyObject *view) {
  PyObject *image = image_of(view);
  if (!image) return -1;
  const nxh_tensor *m = (const nxh_tensor *)PyBytes_AS_STRING(image);
  d->ndim = m->ndim;
  d->offset = m->offset;
  memcpy(d->shape, m->shape, sizeof(int64_t) * (size_t)m->ndim);
  memcpy(d->strides, m->strides, sizeof(int64_t) * (size_t)m->ndim);
  Py_DECREF(image);
  return 0;
}

/* What the calls need of a dtype; the table's dtypes are few and live for good. */
typedef struct {
  PyObject *dtype;
  int tag, packed;
  int64_t itemsize;
} DInfo;
static DInfo dinfo[64];
static int dinfo_n;
static const DInfo *dtype_info(PyObject *dtype) {
  for (int i = 0; i < dinfo_n; i++)
    if (dinfo[i].dtype == dtype) return &dinfo[i];
  PyObject *tag = PyObject_GetAttr(dtype, s_tag), *size = PyObject_GetAttr(dtype, s_itemsize), *packed = PyObject_GetAttr(dtype, s_packed);
  static DInfo once;
  DInfo d = {dtype, 0, 0, 0};
  if (tag && size && packed) {
    d.tag = (int)PyLong_AsLong(tag);
    d.itemsize = PyLong_AsLongLong(size);
    d.packed = PyObject_IsTrue(packed);
  }
  Py_XDECREF(tag);
  Py_XDECREF(size);
  Py_XDECREF(packed);
  if (PyErr_Occurred()) return NULL;
  if (dinfo_n == (int)(sizeof dinfo / sizeof *dinfo)) { /* (read before the lock is let go) */
    once = d;
    return &once;
  }
  Py_INCREF(dtype);
  dinfo[dinfo_n] = d;
  return &dinfo[dinfo_n++];
}

static PyObject *tensor_desc(Tensor *t, PyObject *unused) {
  (void)unused;
  if (!t->d) {
    const DInfo *di = dtype_info(t->dtype);
    PyObject *image = di ? image_of(t->view) : NULL, *ptr = image ? PyObject_GetAttrString(t->buffer, "ptr") : NULL;
    if (ptr) t->d = PyObject_CallFunction(stamp, "OiO", ptr, di->tag, image);
    Py_XDECREF(ptr);
    Py_XDECREF(image);
    if (!t->d) return NULL;
  }
  Py_INCREF(t->d);
  return t->d;
}
static PyObject *tensor_copy(Tensor *t, PyObject *unused) {
  (void)unused;
  return tensor_make(t->buffer, t->view, t->shape, t->dtype, t->context);
}
static PyObject *tensor_strides(Tensor *t, void *u) {
  (void)u;
  return PyObject_GetAttr(t->view, s_strides);
}
static PyObject *tensor_offset(Tensor *t, void *u) {
  (void)u;
  return PyObject_GetAttr(t->view, s_offset);
}
static PyObject *tensor_repr(Tensor *t) {
  PyObject *name = PyObject_GetAttr(t->dtype, s_name), *strides = tensor_strides(t, NULL), *offset = tensor_offset(t, NULL), *r = NULL;
  if (name && strides && offset) r = PyUnicode_FromFormat("Tensor(%S, shape=%S, strides=%S, offset=%S)", name, t->shape, strides, offset);
  Py_XDECREF(name);
  Py_XDECREF(strides);
  Py_XDECREF(offset);
  return r;
}
static PyMemberDef tensor_members[] = {{"buffer", T_OBJECT_EX, offsetof(Tensor, buffer), READONLY, NULL},
                                       {"view", T_OBJECT_EX, offsetof(Tensor, view), READONLY, NULL},
                                       {"shape", T_OBJECT_EX, offsetof(Tensor, shape), READONLY, NULL},
                                       {"dtype", T_OBJECT_EX, offsetof(Tensor, dtype), READONLY, NULL},
                                       {"context", T_OBJECT_EX, offsetof(Tensor, context), READONLY, NULL},
                                       {NULL, 0, 0, 0, NULL}};
static PyGetSetDef tensor_getset[] = {{"strides", (getter)tensor_strides, NULL, NULL, NULL},
                                      {"offset", (getter)tensor_offset, NULL, NULL, NULL},
                                      {NULL, NULL, NULL, NULL, NULL}};
static PyMethodDef tensor_methods[] = {
    {"_desc", (PyCFunction)tensor_desc, METH_NOARGS,
     "The C descriptor, made once: handle, view and storage do not change. The library reads it during a call\n"
     "and keeps no pointer to it."},
    {"__copy__", (PyCFunction)tensor_copy, METH_NOARGS, "Another handle of the same storage (copy.copy)."},
    {NULL, NULL, 0, NULL}};
static PyTypeObject TensorType = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "raven_amd._nxcalls.Tensor",
    .tp_basicsize = sizeof(Tensor),
    .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC,
    .tp_traverse = (traverseproc)tensor_traverse,
    .tp_doc = "The backend's tensor handle (nx_backend.ml:36-43).",
    .tp_new = tensor_new,
    .tp_dealloc = (destructor)tensor_dealloc,
    .tp_repr = (reprfunc)tensor_repr,
    .tp_members = tensor_members,
    .tp_getset = tensor_getset,
    .tp_methods = tensor_methods,
};

/* ── operands and results ─────────────────────────────────────────────────── */
/* The descriptor of an operand: a Tensor's, or what anything with a `_desc` says it is. */
static int describe(nxh_tensor *d, PyObject *o) {
  if (Py_TYPE(o) == &TensorType) {
    const Tensor *t = (const Tensor *)o;
    const DInfo *di = dtype_info(t->dtype);
    if (!di || describe_view(d, t->view)) return -1;
    d->dtype = di->tag;
    if (Py_TYPE(t->buffer) == &BufferType) {
      d->data = ((const Buffer *)t->buffer)->ptr;
      return 0;
    }
    PyObject *p = PyObject_GetAttrString(t->buffer, "ptr");
    if (!p) return -1;
    d->data = p == Py_None ? NULL : PyLong_AsVoidPtr(p);
    Py_DECREF(p);
    return PyErr_Occurred() ? -1 : 0;
  }
  PyObject *c = PyObject_CallMethodNoArgs(o, s_desc);
  if (!c) return -1;
  Py_buffer b;
  int bad = PyObject_GetBuffer(c, &b, PyBUF_SIMPLE);
  if (!bad) {
    if (b.len == (Py_ssize_t)sizeof(nxh_tensor)) memcpy(d, b.buf, sizeof(nxh_tensor));
    else bad = -1, PyErr_SetString(PyExc_TypeError, "not a tensor descriptor");
    PyBuffer_Release(&b);
  }
  Py_DECREF(c);
  return bad;
}
static PyObject *shape_of(PyObject *o) {
  if (Py_TYPE(o) == &TensorType) {
    Py_INCREF(((Tensor *)o)->shape);
    return ((Tensor *)o)->shape;
  }
  return PyObject_GetAttr(o, s_shape);
}
static PyObject *dtype_of(PyObject *o) {
  if (Py_TYPE(o) == &TensorType) {
    Py_INCREF(((Tensor *)o)->dtype);
    return ((Tensor *)o)->dtype;
  }
  return PyObject_GetAttr(o, s_dtype);
}

/* A result that is being made: its view and size, then its storage. */
typedef struct {
  PyObject *view, *shape, *dtype;
  Py_ssize_t nbytes;
  nxh_tensor d;
} Result;
static int result_plan(Result *r, PyObject *shape, PyObject *dtype) {
  r->view = PyTuple_CheckExact(shape) ? PyDict_GetItemWithError(contiguous_views, shape) : NULL;
  if (r->view) Py_INCREF(r->view);
  else if (PyErr_Occurred() || !(r->view = PyObject_CallOneArg(view_create, shape))) return -1;
  r->shape = NULL;
  const DInfo *di = dtype_info(dtype);
  if (!di || describe_view(&r->d, r->view) || !(r->shape = PyObject_GetAttr(r->view, s_shape))) {
    Py_DECREF(r->view);
    return -1;
  }
  int64_t n = 1;
  for (int i = 0; i < r->d.ndim; i++)
    if (__builtin_mul_overflow(n, r->d.shape[i], &n)) n = INT64_MAX / 32;
  r->nbytes = (Py_ssize_t)(di->packed ? (n + 1) / 2 : n * di->itemsize);
  r->d.dtype = di->tag;
  r->dtype = dtype;
  Py_INCREF(dtype);
  return 0;
}
static void result_drop(Result *r) {
  Py_DECREF(r->dtype);
  Py_DECREF(r->view);
  Py_DECREF(r->shape);
}
/* The tensor, or the error of `rc` with the storage given back. */
static PyObject *result_finish(Result *r, PyObject *ctx, int alloc_rc, int rc) {
  PyObject *t = NULL;
  if (alloc_rc) raise_status(ctx, alloc_rc);
  else {
    Buffer *b = buffer_wrap(ctx, r->d.data, r->nbytes);
    if (b && rc) raise_status(ctx, rc);
    else if (b) t = tensor_make((PyObject *)b, r->view, r->shape, r->dtype, ctx);
    Py_XDECREF(b);
  }
  result_drop(r);
  return t;
}
/* Allocates the result and runs `call`, without the interpreter lock. */
#define RUN(r, self, call)                                                      \
  int arc__, rc__ = 0;                                                          \
  nxh_context *h = (self)->h;                                                   \
  Py_BEGIN_ALLOW_THREADS                                                        \
  (r).d.data = NULL;                                                            \
  arc__ = L.alloc(h, (size_t)(r).nbytes, &(r).d.data);                          \
  if (!arc__) rc__ = (call);                                                    \
  Py_END_ALLOW_THREADS                                                          \
  return result_finish(&(r), (PyObject *)(self), arc__, rc__)

/* Arguments by position or by name. */
static int take(const char *fn, const char *const *names, Py_ssize_t n, PyObject *const *args, Py_ssize_t nargs, PyObject *kwnames,
                PyObject **out) {
  Py_ssize_t nk = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
  if (nargs + nk != n) {
    PyErr_Format(PyExc_TypeError, "%s() takes %zd arguments (%zd given)", fn, n, nargs + nk);
    return -1;
  }
  for (Py_ssize_t i = 0; i < n; i++) out[i] = i < nargs ? args[i] : NULL;
  for (Py_ssize_t k = 0; k < nk; k++) {
    PyObject *name = PyTuple_GET_ITEM(kwnames, k);
    Py_ssize_t i = 0;
    while (i < n && PyUnicode_CompareWithASCIIString(name, names[i])) i++;
    if (i == n || out[i]) {
      PyErr_Format(PyExc_TypeError, i == n ? "%s() got an unexpected keyword argument '%U'" : "%s() got multiple values for argument '%U'", fn, name);
      return -1;
    }
    out[i] = args[nargs + k];
  }
  return 0;
}
static int op_number(PyObject *table, PyObject *name) {
  PyObject *i = PyDict_GetItemWithError(table, name);
  if (i) return (int)PyLong_AsLong(i);
  if (!PyErr_Occurred()) PyErr_Format(PyExc_ValueError, "%R is not in list", name);
  return -1;
}
/* A result with the shape of `like` and the given dtype (or, when null, that of `like`). */
static int plan_like(Result *r, PyObject *like, PyObject *dtype) {
  PyObject *shape = shape_of(like), *own = !dtype && shape ? dtype_of(like) : NULL;
  int bad = !shape || (!dtype && !own) || result_plan(r, shape, dtype ? dtype : own);
  Py_XDECREF(shape);
  Py_XDECREF(own);
  return bad ? -1 : 0;
}

typedef PyObject *const *Args;
static PyObject *calls_unary(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  static const char *const names[] = {"op", "x"};
  PyObject *a[2];
  if (take("unary", names, 2, args, n, kw, a)) return NULL;
  int op = op_number(op_unary, a[0]);
  Result r;
  nxh_tensor x;
  if (op < 0 || describe(&x, a[1]) || plan_like(&r, a[1], NULL)) return NULL;
  RUN(r, self, L.unary(h, op, &r.d, &x));
}
static PyObject *two_operands(Calls *self, const char *fn, PyObject *table, int (*call)(nxh_context *, int, const nxh_tensor *, const nxh_tensor *, const nxh_tensor *),
                              PyObject *dtype, Args args, Py_ssize_t n, PyObject *kw) {
  static const char *const names[] = {"op", "x", "y"};
  PyObject *a[3];
  if (take(fn, names, 3, args, n, kw, a)) return NULL;
  int op = op_number(table, a[0]);
  Result r;
  nxh_tensor x, y;
  if (op < 0 || describe(&x, a[1]) || describe(&y, a[2]) || plan_like(&r, a[1], dtype)) return NULL;
  RUN(r, self, call(h, op, &r.d, &x, &y));
}
static PyObject *calls_binary(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  return two_operands(self, "binary", op_binary, L.binary, NULL, args, n, kw);
}
static PyObject *calls_compare(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  return two_operands(self, "compare", op_compare, L.compare, bool_dtype, args, n, kw);
}
static PyObject *calls_where(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  static const char *const names[] = {"cond", "if_true", "if_false"};
  PyObject *a[3];
  Result r;
  nxh_tensor c, x, y;
  if (take("where", names, 3, args, n, kw, a) || describe(&c, a[0]) || describe(&x, a[1]) || describe(&y, a[2]) || plan_like(&r, a[1], NULL)) return NULL;
  RUN(r, self, L.where(h, &r.d, &c, &x, &y));
}
static PyObject *calls_cast(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  static const char *const names[] = {"x", "dtype"};
  PyObject *a[2];
  Result r;
  nxh_tensor x;
  if (take("cast", names, 2, args, n, kw, a) || describe(&x, a[0]) || plan_like(&r, a[0], a[1])) return NULL;
  RUN(r, self, L.cast(h, &r.d, &x));
}
static PyObject *calls_copy(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  static const char *const names[] = {"x"};
  PyObject *a[1];
  Result r;
  nxh_tensor x;
  if (take("copy", names, 1, args, n, kw, a) || describe(&x, a[0]) || plan_like(&r, a[0], NULL)) return NULL;
  RUN(r, self, L.copy(h, &r.d, &x));
}
static PyObject *calls_assign(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  static const char *const names[] = {"dst", "src"};
  PyObject *a[2];
  nxh_tensor d, s;
  if (take("assign", names, 2, args, n, kw, a) || describe(&d, a[0]) || describe(&s, a[1])) return NULL;
  int rc;
  nxh_context *h = self->h;
  Py_BEGIN_ALLOW_THREADS rc = L.copy(h, &d, &s);
  Py_END_ALLOW_THREADS
  if (rc) return raise_status((PyObject *)self, rc);
  Py_RETURN_NONE;
}
static PyObject *calls_full(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  static const char *const names[] = {"dtype", "shape", "value"};
  PyObject *a[3];
  if (take("full", names, 3, args, n, kw, a)) return NULL;
  int array = PyObject_IsInstance(a[2], ndarray_type);
  if (array < 0) return NULL;
  PyObject *enc = array ? (Py_INCREF(a[2]), a[2]) : PyObject_CallFunctionObjArgs(encode_scalar, a[0], a[2], NULL);
  if (!enc) return NULL;
  Py_buffer b;
  if (PyObject_GetBuffer(enc, &b, PyBUF_STRIDED_RO)) {
    Py_DECREF(enc);
    return NULL;
  }
  unsigned char value[64] = {0};
  const int one = b.len == b.itemsize && b.len <= (Py_ssize_t)sizeof value;
  if (one) memcpy(value, b.buf, (size_t)b.len);
  PyBuffer_Release(&b);
  Py_DECREF(enc);
  if (!one) {
    PyErr_SetString(PyExc_ValueError, "full: the value is one element");
    return NULL;
  }
  Result r;
  if (result_plan(&r, a[1], a[0])) return NULL;
  RUN(r, self, L.fill(h, &r.d, value));
}
/* ── operands that broadcast ───────────────────────────────────────────────── */
/* The frontend's rule (frontend.ml:293-296, view.ml expand) applied to descriptors: no reshaped and expanded
 * handles are made of the operands (a forward of GPT-2, 48 tokens, issued call by call: 429 such steps, 74 reductions
 * that keep their axes, 73 products whose batches broadcast: 2119 us -> 1512). What is out of the ordinary (no plain
 * Tensor, extents that do not fit, empty results) answers NotImplemented, and the frontend goes the long way. */
static int broadcast_extents(int64_t *shape, int *ndim, const nxh_tensor *t) {
  const int n = *ndim > t->ndim ? *ndim : t->ndim;
  for (int i = 0; i < n; i++) { /* from the last dim on */
    const int64_t a = i < *ndim ? shape[NXH_MAX_NDIM - 1 - i] : 1, b = i < t->ndim ? t->shape[t->ndim - 1 - i] : 1;
    if (a != b && a != 1 && b != 1) return 0;
    shape[NXH_MAX_NDIM - 1 - i] = a == 1 ? b : a;
    if (a == 0 || b == 0) return 0;
  }
  *ndim = n;
  return 1;
}
/* `t` seen with `ndim` extents: a dim that is not there, or is 1 where the other is not, is read in place. */
static void broadcast_view(nxh_tensor *t, const int64_t *shape, int ndim) {
  const int pad = ndim - t->ndim;
  for (int i = ndim - 1; i >= 0; i--) {
    t->strides[i] = i >= pad && t->shape[i - pad] == shape[i] ? t->strides[i - pad] : 0;
    t->shape[i] = shape[i];
  }
  t->ndim = ndim;
}
static int same_extents(const nxh_tensor *t, const int64_t *shape, int ndim) {
  return t->ndim == ndim && !memcmp(t->shape, shape, sizeof(int64_t) * (size_t)ndim);
}
/* Describes n operands, broadcast together, and plans a result of their extents. 0: go the long way; -1: an error. */
static int broadcast_plan(Result *r, nxh_tensor *t, PyObject *const *a, int n, PyObject *dtype) {
  int64_t extents[NXH_MAX_NDIM];
  int ndim = 0;
  for (int i = 0; i < n; i++)
    if (Py_TYPE(a[i]) != &TensorType) return 0;
  for (int i = 0; i < n; i++) {
    if (describe(&t[i], a[i])) return -1;
    if (!broadcast_extents(extents, &ndim, &t[i])) return 0;
  }
  const int64_t *shape = extents + NXH_MAX_NDIM - ndim;
  PyObject *like = NULL; /* the extents as a tuple: an operand's where one has them */
  for (int i = 0; i < n; i++) {
    if (!same_extents(&t[i], shape, ndim)) broadcast_view(&t[i], shape, ndim);
    else if (!like) like = ((Tensor *)a[i])->shape;
  }
  if (like) return result_plan(r, like, dtype) ? -1 : 1;
  if (!(like = PyTuple_New(ndim))) return -1;
  for (int i = 0; i < ndim; i++) {
    PyObject *e = PyLong_FromLongLong(shape[i]);
    if (!e) {
      Py_DECREF(like);
      return -1;
    }
    PyTuple_SET_ITEM(like, i, e);
  }
  const int bad = result_plan(r, like, dtype);
  Py_DECREF(like);
  return bad ? -1 : 1;
}
static PyObject *calls_broadcast_binary(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  static const char *const names[] = {"op", "x", "y"};
  PyObject *a[3];
  if (take("broadcast_binary", names, 3, args, n, kw, a)) return NULL;
  int op = op_number(op_binary, a[0]);
  if (op < 0) return NULL;
  Result r;
  nxh_tensor t[2];
  const int planned = Py_TYPE(a[1]) == &TensorType ? broadcast_plan(&r, t, a + 1, 2, ((Tensor *)a[1])->dtype) : 0;
  if (planned < 0) return NULL;
  if (!planned) Py_RETURN_NOTIMPLEMENTED;
  RUN(r, self, L.binary(h, op, &r.d, &t[0], &t[1]));
}
static PyObject *calls_broadcast_where(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  static const char *const names[] = {"cond", "if_true", "if_false"};
  PyObject *a[3];
  if (take("broadcast_where", names, 3, args, n, kw, a)) return NULL;
  Result r;
  nxh_tensor t[3];
  const int planned = Py_TYPE(a[1]) == &TensorType ? broadcast_plan(&r, t, a, 3, ((Tensor *)a[1])->dtype) : 0;
  if (planned < 0) return NULL;
  if (!planned) Py_RETURN_NOTIMPLEMENTED;
  RUN(r, self, L.where(h, &r.d, &t[0], &t[1], &t[2]));
}

static PyObject *general(Calls *self, const char *name, PyObject **a, Py_ssize_t n) {
  PyObject *m = PyObject_GetAttrString((PyObject *)self, name);
  if (!m) return NULL;
  PyObject *r = PyObject_Vectorcall(m, a, (size_t)n, NULL);
  Py_DECREF(m);
  return r;
}
/* The view of a result whose reduced axes stay as dims of extent 1 (a fresh result is contiguous either way). */
static int keep_axes(Result *r, PyObject *shape, const int32_t *axes, Py_ssize_t na) {
  const Py_ssize_t nd = PyTuple_GET_SIZE(shape);
  PyObject *kept = PyTuple_New(nd);
  if (!kept) return -1;
  for (Py_ssize_t i = 0, k = 0; i < nd; i++) {
    PyObject *e = k < na && axes[k] == i ? PyLong_FromLong(1) : PyTuple_GET_ITEM(shape, i);
    if (k < na && axes[k] == i) k++;
    else Py_INCREF(e);
    PyTuple_SET_ITEM(kept, i, e);
  }
  PyObject *view = PyDict_GetItemWithError(contiguous_views, kept);
  if (view) Py_INCREF(view);
  else if (!PyErr_Occurred()) view = PyObject_CallOneArg(view_create, kept);
  Py_DECREF(kept);
  PyObject *own = view ? PyObject_GetAttr(view, s_shape) : NULL;
  if (!own) {
    Py_XDECREF(view);
    return -1;
  }
  Py_SETREF(r->view, view);
  Py_SETREF(r->shape, own);
  return 0;
}
static PyObject *reduce_over(Calls *self, PyObject **a, int keep) {
  int op = op_number(op_reduce, a[0]);
  if (op < 0) return NULL;
  if (Py_TYPE(a[2]) == &TensorType && (PyList_CheckExact(a[1]) || PyTuple_CheckExact(a[1]))) {
    PyObject *shape = ((Tensor *)a[2])->shape;
    const Py_ssize_t nd = PyTuple_GET_SIZE(shape), na = PySequence_Fast_GET_SIZE(a[1]);
    int32_t axes[NXH_MAX_NDIM];
    int fine = nd <= NXH_MAX_NDIM && na <= nd;
    for (Py_ssize_t i = 0; i < na && fine; i++) { /* ascending, in range, each once */
      PyObject *v = PySequence_Fast_GET_ITEM(a[1], i);
      long x = PyLong_CheckExact(v) ? PyLong_AsLong(v) : -1;
      fine = x >= 0 && x < nd && (i == 0 || x > axes[i - 1]);
      if (fine) axes[i] = (int32_t)x;
    }
    if (PyErr_Occurred()) PyErr_Clear();
    nxh_tensor x;
    if (fine) {
      if (describe(&x, a[2])) return NULL;
      for (Py_ssize_t i = 0; i < na; i++) fine = fine && x.shape[axes[i]] != 0;
    }
    if (fine) {
      PyObject *kept = PyTuple_New(nd - na);
      if (!kept) return NULL;
      for (Py_ssize_t i = 0, j = 0, k = 0; i < nd; i++) {
        if (k < na && axes[k] == i) {
          k++;
          continue;
        }
        PyObject *e = PyTuple_GET_ITEM(shape, i);
        Py_INCREF(e);
        PyTuple_SET_ITEM(kept, j++, e);
      }
      Result r;
      int bad = result_plan(&r, kept, ((Tensor *)a[2])->dtype);
      Py_DECREF(kept);
      if (bad) return NULL;
      if (keep && keep_axes(&r, shape, axes, na)) {
        result_drop(&r);
        return NULL;
      }
      RUN(r, self, L.reduce(h, op, &r.d, &x, axes, (int)na));
    }
  }
  if (keep) Py_RETURN_NOTIMPLEMENTED;
  return general(self, "_reduce_general", a, 3);
}
static PyObject *calls_reduce(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  static const char *const names[] = {"op", "axes", "x"};
  PyObject *a[3];
  return take("reduce", names, 3, args, n, kw, a) ? NULL : reduce_over(self, a, 0);
}
static PyObject *calls_reduce_keep(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  static const char *const names[] = {"op", "axes", "x"};
  PyObject *a[3];
  return take("reduce_keep", names, 3, args, n, kw, a) ? NULL : reduce_over(self, a, 1);
}
static PyObject *calls_matmul(Calls *self, Args args, Py_ssize_t n, PyObject *kw) {
  static const char *const names[] = {"x", "y"};
  PyObject *a[2];
  if (take("matmul", names, 2, args, n, kw, a)) return NULL;
  if (Py_TYPE(a[0]) == &TensorType && Py_TYPE(a[1]) == &TensorType) {
    nxh_tensor x, y;
    if (describe(&x, a[0]) || describe(&y, a[1])) return NULL;
    /* rows that take no padded pitch; a batch extent is the larger one, as the library checks it */
    if (x.ndim >= 2 && y.ndim >= 2 && y.shape[y.ndim - 1] < 4096) {
      PyObject *sx = ((Tensor *)a[0])->shape, *sy = ((Tensor *)a[1])->shape;
      const int nd = x.ndim > y.ndim ? x.ndim : y.ndim;
      PyObject *shape = PyTuple_New(nd);
      if (!shape) return NULL;
      for (int i = 0; i < nd; i++) {
        const int ix = i - (nd - x.ndim), iy = i - (nd - y.ndim);
        PyObject *e = i == nd - 2   ? PyTuple_GET_ITEM(sx, ix)
                      : i == nd - 1 ? PyTuple_GET_ITEM(sy, iy)
                      : ix < 0      ? PyTuple_GET_ITEM(sy, iy)
                      : iy < 0 || x.shape[ix] >= y.shape[iy] ? PyTuple_GET_ITEM(sx, ix) : PyTuple_GET_ITEM(sy, iy);
        Py_INCREF(e);
        PyTuple_SET_ITEM(shape, i, e);
      }
      Result r;
      int bad = result_plan(&r, shape, ((Tensor *)a[0])->dtype);
      Py_DECREF(shape);
      if (bad) return NULL;
      RUN(r, self, L.matmul(h, &r.d, &x, &y));
    }
  }
  return general(self, "_matmul_general", a, 2);
}

#define FAST METH_FASTCALL | METH_KEYWORDS
static PyMethodDef calls_methods[] = {
    {"unary", (PyCFunction)(void (*)(void))calls_unary, FAST, "unary($self, op, x)\n--\n\n"},
    {"binary", (PyCFunction)(void (*)(void))calls_binary, FAST, "binary($self, op, x, y)\n--\n\n"},
    {"compare", (PyCFunction)(void (*)(void))calls_compare, FAST, "compare($self, op, x, y)\n--\n\n"},
    {"where", (PyCFunction)(void (*)(void))calls_where, FAST, "where($self, cond, if_true, if_false)\n--\n\n"},
    {"cast", (PyCFunction)(void (*)(void))calls_cast, FAST, "cast($self, x, dtype)\n--\n\n"},
    {"copy", (PyCFunction)(void (*)(void))calls_copy, FAST, "copy($self, x)\n--\n\n"},
    {"assign", (PyCFunction)(void (*)(void))calls_assign, FAST,
     "assign($self, dst, src)\n--\n\nWrites ``src`` through ``dst``'s strides (visible through every view sharing dst's buffer)."},
    {"full", (PyCFunction)(void (*)(void))calls_full, FAST,
     "full($self, dtype, shape, value)\n--\n\nEvery element is ``value`` (a Python number, or one already-encoded storage element as a numpy array)."},
    {"reduce", (PyCFunction)(void (*)(void))calls_reduce, FAST, "reduce($self, op, axes, x)\n--\n\n"},
    {"matmul", (PyCFunction)(void (*)(void))calls_matmul, FAST, "matmul($self, x, y)\n--\n\n"},
    {"broadcast_binary", (PyCFunction)(void (*)(void))calls_broadcast_binary, FAST,
     "broadcast_binary($self, op, x, y)\n--\n\nbinary of operands broadcast together; NotImplemented where that is out of the ordinary."},
    {"broadcast_where", (PyCFunction)(void (*)(void))calls_broadcast_where, FAST,
     "broadcast_where($self, cond, if_true, if_false)\n--\n\nwhere, likewise."},
    {"reduce_keep", (PyCFunction)(void (*)(void))calls_reduce_keep, FAST,
     "reduce_keep($self, op, axes, x)\n--\n\nreduce whose reduced axes (ascending) stay as dims of extent 1; NotImplemented likewise."},
    {NULL, NULL, 0, NULL}};
static PyGetSetDef calls_getset[] = {{"_h", (getter)calls_get_h, (setter)calls_set_h, NULL, NULL}, {NULL, NULL, NULL, NULL, NULL}};
static PyTypeObject CallsType = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "raven_amd._nxcalls.Calls",
    .tp_basicsize = sizeof(Calls),
    .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE,
    .tp_new = PyType_GenericNew,
    .tp_methods = calls_methods,
    .tp_getset = calls_getset,
};

/* ── module ───────────────────────────────────────────────────────────────── */
/* bind(addresses): the library's entry points, by name. */
static PyObject *bind(PyObject *m, PyObject *d) {
  (void)m;
  struct {
    const char *name;
    void **to;
  } e[] = {{"nxh_alloc", (void **)&L.alloc},     {"nxh_free", (void **)&L.free},       {"nxh_fill", (void **)&L.fill},
           {"nxh_unary", (void **)&L.unary},     {"nxh_binary", (void **)&L.binary},   {"nxh_compare", (void **)&L.compare},
           {"nxh_where", (void **)&L.where},     {"nxh_cast", (void **)&L.cast},       {"nxh_copy", (void **)&L.copy},
           {"nxh_reduce", (void **)&L.reduce},   {"nxh_matmul", (void **)&L.matmul}};
  for (size_t i = 0; i < sizeof e / sizeof *e; i++) {
    PyObject *v = PyMapping_GetItemString(d, e[i].name);
    if (!v) return NULL;
    *e[i].to = PyLong_AsVoidPtr(v);
    Py_DECREF(v);
    if (PyErr_Occurred()) return NULL;
  }
  Py_RETURN_NONE;
}
static PyObject *setup(PyObject *m, PyObject *args) {
  (void)m;
  PyObject **to[] = {&contiguous_views, &view_create, &view_image, &stamp, &encode_scalar, &ndarray_type, &bool_dtype,
                     &op_unary, &op_binary, &op_compare, &op_reduce};
  const Py_ssize_t n = sizeof to / sizeof *to;
  if (PyTuple_GET_SIZE(args) != n) {
    PyErr_SetString(PyExc_TypeError, "setup() takes the objects listed in nx_calls.c");
    return NULL;
  }
  for (Py_ssize_t i = 0; i < n; i++) {
    PyObject *v = PyTuple_GET_ITEM(args, i), *old = *to[i];
    Py_INCREF(v);
    *to[i] = v;
    Py_XDECREF(old);
  }
  Py_RETURN_NONE;
}
static PyMethodDef module_methods[] = {{"bind", bind, METH_O, "The library's entry points: a dict of addresses by name."},
                                       {"setup", setup, METH_VARARGS, "What the calls use of the Python side."},
                                       {NULL, NULL, 0, NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_nxcalls", "The per-primitive host path, in C.", -1, module_methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__nxcalls(void) {
  struct {
    PyObject **to;
    const char *s;
  } names[] = {{&s_image, "image"}, {&s_shape, "shape"}, {&s_strides, "strides"}, {&s_offset, "offset"}, {&s_tag, "tag"}, {&s_itemsize, "itemsize"},
               {&s_packed, "packed"}, {&s_desc, "_desc"}, {&s_dtype, "dtype"}, {&s_name, "name"}};
  for (size_t i = 0; i < sizeof names / sizeof *names; i++)
    if (!(*names[i].to = PyUnicode_InternFromString(names[i].s))) return NULL;
  if (PyType_Ready(&CallsType) || PyType_Ready(&BufferType) || PyType_Ready(&TensorType)) return NULL;
  PyObject *m = PyModule_Create(&module);
  if (!m) return NULL;
  if (PyModule_AddObjectRef(m, "Calls", (PyObject *)&CallsType) || PyModule_AddObjectRef(m, "DeviceBuffer", (PyObject *)&BufferType) ||
      PyModule_AddObjectRef(m, "Tensor", (PyObject *)&TensorType)) {
    Py_DECREF(m);
    return NULL;
  }
  return m;
}
