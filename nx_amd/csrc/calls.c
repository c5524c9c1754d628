/* The host side of a callback without its Python: buffer handles, calls whose arguments are known per signature, and whole
 * traced functions as a list of such calls.
 *
 * A callback through ctypes cost 3-5 us of Python beside the 4.2 us of the library (2.7 of them the launch): the argument
 * conversions of the call, of the allocation in front of it and of the release behind its operands.  A traced function
 * paid 5-7 us more per node to its evaluator.  Here a callback's arguments are laid out once per signature (Call), a traced
 * function's calls are recorded once and issued again from C (Replay); the library is called through the same entry points
 * with the same arguments.  add, multiply, exp, sum of 1024 x 1024, one callback at a time: 30.6 -> 18.6 us a pass; a number as
 * an operand, whose constant was looked up on every call, is laid out with the call (multiply by 0.5 5.6 -> 3.9 us), and a traced function's
 * arguments are looked at here (layer normalisation 64 x 512 5.5 -> 4.2 us).
 *
 * Every entry point of include/hipnx.h takes integers and pointers only, at most MAX_ARGS of them: they are called through
 * one function type of 64-bit arguments (an int argument is the low half of its register or stack slot). */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>
#include <stdint.h>
#include "../../include/hipnx.h"

#define MAX_ARGS 20
typedef int (*entry_t)(int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t,
                       int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t);

static int enter(int64_t fn, const int64_t *a) {
  return ((entry_t)(intptr_t)fn)(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9], a[10], a[11], a[12], a[13], a[14], a[15],
                                a[16], a[17], a[18], a[19]);
}

static int (*buf_alloc)(void *, size_t, void **);
static int (*buf_destroy)(void *);
static PyTypeObject *tensor_type, *backend_type;
static PyObject *raise_status;        /* raises what the library reports with a status */
static PyObject *s_data, *s_type, *s_shape, *s_names, *s_ref, *s_device, *s_released;
static PyObject *freed_log;           /* the list that takes the handles `freed_thread` releases, while a function is recorded */
static unsigned long freed_thread;

/* While a thread's evaluation is recorded its calls go through the library's stand-in, which writes them down. */
static int is_recording(void) { return freed_log && freed_thread == PyThread_get_thread_ident(); }

/* Whether a status is an error of the call to raise at once.  The others (an operand gone, no memory, nothing that the kernels
 * take) are found again by the general path, which reports them; these may not be: what an earlier kernel recorded is
 * reported once, to the call that waits, and so is an error of the device. */
static int is_raised(int status) { return status == HIPNX_EHIP || status == HIPNX_EINDEX || status == HIPNX_ERAISED; }
static PyObject *raised(int status) {
  PyObject *r = PyObject_CallFunction(raise_status, "i", status);
  Py_XDECREF(r);
  if (r) PyErr_Format(PyExc_RuntimeError, "status %d", status);
  return NULL;
}

/* ---- Ref: owns one buffer handle ------------------------------------------------------------- */
typedef struct {
  PyObject_HEAD
  PyObject *ctx, *keep;
  void *handle;
  Py_ssize_t nbytes, sharers;
} Ref;

static void ref_dealloc(Ref *self) {
  PyObject_GC_UnTrack(self);
  if (self->handle && buf_destroy) {
    if (is_recording()) {
      PyObject *h = PyLong_FromVoidPtr(self->handle);
      if (!h || PyList_Append(freed_log, h) < 0) PyErr_Clear();
      Py_XDECREF(h);
    }
    void *h = self->handle;
    self->handle = NULL;
    Py_BEGIN_ALLOW_THREADS
    buf_destroy(h);
    Py_END_ALLOW_THREADS
  }
  Py_XDECREF(self->ctx);
  Py_XDECREF(self->keep);
  Py_TYPE(self)->tp_free((PyObject *)self);
}

static int ref_init(Ref *self, PyObject *args, PyObject *kw) {
  static char *names[] = {"ctx", "handle", "nbytes", "keep", NULL};
  PyObject *ctx, *keep = Py_None;
  unsigned long long handle;
  Py_ssize_t nbytes;
  if (!PyArg_ParseTupleAndKeywords(args, kw, "OKn|O", names, &ctx, &handle, &nbytes, &keep)) return -1;
  if (self->handle) {
    PyErr_SetString(PyExc_RuntimeError, "a buffer reference is made once");
    return -1;
  }
  Py_INCREF(ctx);
  Py_XSETREF(self->ctx, ctx);
  Py_INCREF(keep);
  Py_XSETREF(self->keep, keep);
  self->handle = (void *)(uintptr_t)handle;
  self->nbytes = nbytes;
  self->sharers = 1;
  return 0;
}

/* The owner of borrowed memory may lead back here (an object that holds the tensor it lends its memory to). */
static int ref_traverse(Ref *self, visitproc visit, void *arg) {
  Py_VISIT(self->ctx);
  Py_VISIT(self->keep);
  return 0;
}
static int ref_clear(Ref *self) {
  PyObject *keep = self->keep;
  Py_INCREF(Py_None);
  self->keep = Py_None;
  Py_XDECREF(keep);
  return 0;
}

static PyObject *ref_get_handle(Ref *self, void *unused) { return PyLong_FromVoidPtr(self->handle); }
static PyMemberDef ref_members[] = {{"ctx", T_OBJECT, offsetof(Ref, ctx), READONLY, NULL},
                                    {"keep", T_OBJECT, offsetof(Ref, keep), READONLY, NULL},
                                    {"nbytes", T_PYSSIZET, offsetof(Ref, nbytes), READONLY, NULL},
                                    {"sharers", T_PYSSIZET, offsetof(Ref, sharers), 0, NULL},
                                    {NULL}};
static PyGetSetDef ref_getset[] = {{"handle", (getter)ref_get_handle, NULL, "the hipnx_buf pointer", NULL}, {NULL}};
static PyTypeObject RefType = {PyVarObject_HEAD_INIT(NULL, 0).tp_name = "hipnx_calls.Ref", .tp_basicsize = sizeof(Ref),
                               .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_GC, .tp_new = PyType_GenericNew, .tp_init = (initproc)ref_init,
                               .tp_traverse = (traverseproc)ref_traverse, .tp_clear = (inquiry)ref_clear, .tp_dealloc = (destructor)ref_dealloc, .tp_members = ref_members, .tp_getset = ref_getset,
                               .tp_doc = "Owns one device buffer; shared by metadata-only callbacks."};

static Ref *new_ref(PyObject *ctx, void *handle, Py_ssize_t nbytes) {
  Ref *r = (Ref *)RefType.tp_alloc(&RefType, 0);
  if (!r) return NULL;
  PyObject_GC_UnTrack(r); /* it owns its memory: nothing for the collector to follow */
  Py_INCREF(ctx);
  r->ctx = ctx;
  Py_INCREF(Py_None);
  r->keep = Py_None;
  r->handle = handle;
  r->nbytes = nbytes;
  r->sharers = 1;
  return r;
}

/* a tensor of the backend over `ref` (whose reference is taken) */
static PyObject *new_tensor(Ref *ref, PyObject *device, PyObject *type, PyObject *shape, PyObject *names) {
  PyObject *data = backend_type->tp_alloc(backend_type, 0), *t = data ? tensor_type->tp_alloc(tensor_type, 0) : NULL;
  if (!t || PyObject_GenericSetAttr(data, s_ref, (PyObject *)ref) < 0 || PyObject_GenericSetAttr(data, s_device, device) < 0 ||
      PyObject_GenericSetAttr(data, s_released, Py_False) < 0 || PyObject_GenericSetAttr(t, s_data, data) < 0 ||
      PyObject_GenericSetAttr(t, s_type, type) < 0 || PyObject_GenericSetAttr(t, s_shape, shape) < 0 ||
      PyObject_GenericSetAttr(t, s_names, names) < 0)
    Py_CLEAR(t);
  Py_XDECREF(data);
  Py_DECREF(ref);
  return t;
}

/* the live buffer of a tensor on `device`, as a new reference, or NULL (without an error) */
static Ref *live_ref(PyObject *tensor, PyObject *device) {
  if (Py_TYPE(tensor) != tensor_type) return NULL;
  Ref *found = NULL;
  PyObject *data = PyObject_GenericGetAttr(tensor, s_data);
  if (data && Py_TYPE(data) == backend_type) {
    PyObject *ref = PyObject_GenericGetAttr(data, s_ref), *released = PyObject_GenericGetAttr(data, s_released),
             *on = PyObject_GenericGetAttr(data, s_device);
    if (ref && released == Py_False && on && Py_TYPE(ref) == &RefType && ((Ref *)ref)->handle &&
        (on == device || PyObject_RichCompareBool(on, device, Py_EQ) == 1)) {
      found = (Ref *)ref;
      Py_INCREF(found);
    }
    Py_XDECREF(ref);
    Py_XDECREF(released);
    Py_XDECREF(on);
  }
  Py_XDECREF(data);
  PyErr_Clear();
  return found;
}

/* ---- Call: one entry point with everything but its buffers laid out ------------------------------ */
typedef struct {
  PyObject_HEAD
  PyObject *ctx, *device, *type, *shape, *names, *keep;
  int64_t fn, args[MAX_ARGS], ctx_value;
  Py_ssize_t nbytes;
  int n_in, out_at, in_at[4];
} Call;

static void call_dealloc(Call *self) {
  Py_XDECREF(self->ctx);
  Py_XDECREF(self->device);
  Py_XDECREF(self->type);
  Py_XDECREF(self->shape);
  Py_XDECREF(self->names);
  Py_XDECREF(self->keep);
  Py_TYPE(self)->tp_free((PyObject *)self);
}

static PyObject *call_call(Call *self, PyObject *args, PyObject *kw);
static PyObject *call_bind(Call *from, PyObject *args);
static PyMethodDef call_methods[] = {{"bind", (PyCFunction)call_bind, METH_VARARGS, NULL}, {NULL}};
static PyTypeObject CallType = {PyVarObject_HEAD_INIT(NULL, 0).tp_name = "hipnx_calls.Call", .tp_basicsize = sizeof(Call),
                                .tp_flags = Py_TPFLAGS_DEFAULT, .tp_dealloc = (destructor)call_dealloc,
                                .tp_call = (ternaryfunc)call_call, .tp_methods = call_methods,
                                .tp_doc = "call(*tensors) -> the result, or None where the tensors are not what it was made for, or the "
                                          "library refused (the general path then reports it); raises what the call itself reports"};

/* prepare(fn, args, in_at, out_at, nbytes, ctx, ctx_value, device, type, shape, names, keep) */
static PyObject *prepare(PyObject *mod, PyObject *a) {
  long long fn, ctx_value;
  PyObject *list, *in_at, *ctx, *device, *type, *shape, *names, *keep;
  int out_at;
  Py_ssize_t nbytes;
  if (!PyArg_ParseTuple(a, "LO!O!inOLOOOOO", &fn, &PyList_Type, &list, &PyList_Type, &in_at, &out_at, &nbytes, &ctx, &ctx_value, &device, &type,
                        &shape, &names, &keep))
    return NULL;
  const Py_ssize_t n = PyList_GET_SIZE(list), n_in = PyList_GET_SIZE(in_at);
  if (n > MAX_ARGS || n_in < 1 || n_in > 4 || out_at < 0 || out_at >= n) return PyErr_Format(PyExc_ValueError, "prepare: too many arguments");
  Call *c = (Call *)CallType.tp_alloc(&CallType, 0);
  if (!c) return NULL;
  c->fn = fn, c->ctx_value = ctx_value, c->nbytes = nbytes, c->out_at = out_at, c->n_in = (int)n_in;
#define KEEP(x) (Py_INCREF(x), c->x = x)
  KEEP(ctx), KEEP(device), KEEP(type), KEEP(shape), KEEP(names), KEEP(keep);
#undef KEEP
  for (Py_ssize_t i = 0; i < n; i++) c->args[i] = PyLong_AsLongLong(PyList_GET_ITEM(list, i));
  for (Py_ssize_t i = 0; i < n_in; i++) {
    c->in_at[i] = (int)PyLong_AsLong(PyList_GET_ITEM(in_at, i));
    if (!PyErr_Occurred() && (c->in_at[i] < 0 || c->in_at[i] >= n)) PyErr_SetString(PyExc_ValueError, "prepare: an operand that is no argument");
  }
  if (PyErr_Occurred()) Py_CLEAR(c);
  return (PyObject *)c;
}

static PyObject *call_call(Call *self, PyObject *args, PyObject *kw) {
  Ref *in[4] = {NULL, NULL, NULL, NULL};
  int64_t a[MAX_ARGS];
  void *out = NULL;
  int ok = PyTuple_GET_SIZE(args) == self->n_in && !is_recording(), status = HIPNX_EINVAL;
  memcpy(a, self->args, sizeof(a));
  for (int i = 0; ok && i < self->n_in; i++) {
    in[i] = live_ref(PyTuple_GET_ITEM(args, i), self->device);
    if (!in[i]) ok = 0;
    else a[self->in_at[i]] = (int64_t)(intptr_t)in[i]->handle;
  }
  if (ok) {
    Py_BEGIN_ALLOW_THREADS
    status = buf_alloc((void *)(intptr_t)self->ctx_value, (size_t)self->nbytes, &out);
    if (!status) {
      a[self->out_at] = (int64_t)(intptr_t)out;
      status = enter(self->fn, a);
      if (status) buf_destroy(out);
    }
    Py_END_ALLOW_THREADS
  }
  for (int i = 0; i < self->n_in; i++) Py_XDECREF(in[i]);
  if (is_raised(status)) return raised(status);
  if (status) Py_RETURN_NONE;
  Ref *ref = new_ref(self->ctx, out, self->nbytes);
  if (!ref) {
    buf_destroy(out);
    return NULL;
  }
  return new_tensor(ref, self->device, self->type, self->shape, self->names);
}

/* call.bind(position, tensor) -> the same call with that operand laid out too, or None (a tensor that is not on its device) */
static PyObject *call_bind(Call *from, PyObject *a) {
  int at;
  PyObject *tensor;
  if (!PyArg_ParseTuple(a, "iO", &at, &tensor)) return NULL;
  Ref *ref = at >= 0 && at < from->n_in && from->n_in > 1 ? live_ref(tensor, from->device) : NULL;
  if (!ref) Py_RETURN_NONE;
  Call *c = (Call *)CallType.tp_alloc(&CallType, 0);
  PyObject *keep = c ? PyTuple_Pack(2, from->keep, (PyObject *)ref) : NULL;
  if (keep) {
#define KEEP(x) (Py_INCREF(from->x), c->x = from->x)
    KEEP(ctx), KEEP(device), KEEP(type), KEEP(shape), KEEP(names);
#undef KEEP
    c->keep = keep;
    c->fn = from->fn, c->ctx_value = from->ctx_value, c->nbytes = from->nbytes, c->out_at = from->out_at, c->n_in = from->n_in - 1;
    memcpy(c->args, from->args, sizeof(c->args));
    c->args[from->in_at[at]] = (int64_t)(intptr_t)ref->handle;
    for (int i = 0, j = 0; i < from->n_in; i++)
      if (i != at) c->in_at[j++] = from->in_at[i];
  } else Py_CLEAR(c);
  Py_DECREF(ref);
  return (PyObject *)c;
}

/* ---- Replay: the calls of a traced function ------------------------------------------------------- */
enum { OP_ALLOC, OP_FREE, OP_CALL };
typedef struct {
  int kind, slot, first_patch, n_patches, first_list, n_lists;
  int64_t value;  /* bytes of an allocation, the entry point of a call */
  int64_t args[MAX_ARGS];
} Op;
typedef struct { int at, slot; } Patch;            /* argument `at` is the handle in `slot` */
typedef struct { int at, first, count; } HandleList; /* argument `at` is an array of the handles in these slots */
typedef struct {
  PyObject_HEAD
  PyObject *ctx, *device, *keep, *shapes;  /* shapes: (type, shape) of each argument that a caller has not checked */
  int64_t ctx_value;
  int n_params, n_slots, n_ops, n_outs;
  Op *ops;
  Patch *patches;
  HandleList *lists;
  int *list_slots, *outs;
  Py_ssize_t *out_bytes;
  PyObject **out_type, **out_shape, **out_names;
} Replay;

static void replay_dealloc(Replay *self) {
  for (int i = 0; i < self->n_outs; i++) {
    Py_XDECREF(self->out_type[i]);
    Py_XDECREF(self->out_shape[i]);
    Py_XDECREF(self->out_names[i]);
  }
  PyMem_Free(self->ops), PyMem_Free(self->patches), PyMem_Free(self->lists), PyMem_Free(self->list_slots), PyMem_Free(self->outs);
  PyMem_Free(self->out_bytes), PyMem_Free(self->out_type), PyMem_Free(self->out_shape), PyMem_Free(self->out_names);
  Py_XDECREF(self->ctx);
  Py_XDECREF(self->device);
  Py_XDECREF(self->keep);
  Py_XDECREF(self->shapes);
  Py_TYPE(self)->tp_free((PyObject *)self);
}

static PyObject *replay_call(Replay *self, PyObject *args, PyObject *kw);
static PyTypeObject ReplayType = {PyVarObject_HEAD_INIT(NULL, 0).tp_name = "hipnx_calls.Replay", .tp_basicsize = sizeof(Replay),
                                  .tp_flags = Py_TPFLAGS_DEFAULT, .tp_dealloc = (destructor)replay_dealloc,
                                  .tp_call = (ternaryfunc)replay_call,
                                  .tp_doc = "replay(*tensors) -> [results], or None where the tensors are not what it was recorded for, or a "
                                            "call was refused (nothing is kept then: the function is evaluated the general way); raises what a call "
                                            "itself reports"};

/* record(ops, n_params, n_slots, outs, ctx, ctx_value, device, keep, shapes)
 * shapes: a tuple of (type, shape), of the first arguments: what a call is refused for otherwise
 * ops: ("alloc", slot, nbytes) | ("free", slot) | ("call", fn, [argument | ("slot", s) | ("list", [s, ...])])
 * outs: [(slot, nbytes, type, shape, names)] */
static PyObject *record(PyObject *mod, PyObject *a) {
  PyObject *ops, *outs, *ctx, *device, *keep, *shapes;
  int n_params, n_slots;
  long long ctx_value;
  if (!PyArg_ParseTuple(a, "O!iiO!OLOOO!", &PyList_Type, &ops, &n_params, &n_slots, &PyList_Type, &outs, &ctx, &ctx_value, &device, &keep, &PyTuple_Type, &shapes)) return NULL;
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(shapes); i++)
    if (i >= n_params || !PyTuple_Check(PyTuple_GET_ITEM(shapes, i)) || PyTuple_GET_SIZE(PyTuple_GET_ITEM(shapes, i)) != 2)
      return PyErr_Format(PyExc_ValueError, "record: (type, shape) of the arguments");
  int n_patches = 0, n_lists = 0, n_list_slots = 0;
  const int n_ops = (int)PyList_GET_SIZE(ops), n_outs = (int)PyList_GET_SIZE(outs);
  for (int i = 0; i < n_ops; i++) {
    PyObject *op = PyList_GET_ITEM(ops, i);
    if (PyTuple_GET_SIZE(op) != 3 || !PyList_Check(PyTuple_GET_ITEM(op, 2))) continue;
    PyObject *list = PyTuple_GET_ITEM(op, 2);
    for (Py_ssize_t j = 0; j < PyList_GET_SIZE(list); j++) {
      PyObject *v = PyList_GET_ITEM(list, j);
      if (!PyTuple_Check(v)) continue;
      if (PyList_Check(PyTuple_GET_ITEM(v, 1))) n_lists++, n_list_slots += (int)PyList_GET_SIZE(PyTuple_GET_ITEM(v, 1));
      else n_patches++;
    }
  }
  Replay *r = (Replay *)ReplayType.tp_alloc(&ReplayType, 0);
  if (!r) return NULL;
  Py_INCREF(ctx), Py_INCREF(device), Py_INCREF(keep), Py_INCREF(shapes);
  r->ctx = ctx, r->device = device, r->keep = keep, r->shapes = shapes, r->ctx_value = ctx_value;
  r->n_params = n_params, r->n_slots = n_slots, r->n_ops = n_ops;
  r->ops = PyMem_Calloc(n_ops + 1, sizeof(Op));
  r->patches = PyMem_Calloc(n_patches + 1, sizeof(Patch));
  r->lists = PyMem_Calloc(n_lists + 1, sizeof(HandleList));
  r->list_slots = PyMem_Calloc(n_list_slots + 1, sizeof(int));
  r->outs = PyMem_Calloc(n_outs + 1, sizeof(int));
  r->out_bytes = PyMem_Calloc(n_outs + 1, sizeof(Py_ssize_t));
  r->out_type = PyMem_Calloc(n_outs + 1, sizeof(PyObject *));
  r->out_shape = PyMem_Calloc(n_outs + 1, sizeof(PyObject *));
  r->out_names = PyMem_Calloc(n_outs + 1, sizeof(PyObject *));
  if (!r->ops || !r->patches || !r->lists || !r->list_slots || !r->outs || !r->out_bytes || !r->out_type || !r->out_shape || !r->out_names) {
    PyErr_NoMemory();
    goto fail;
  }
  int patch = 0, list_no = 0, list_slot = 0;
#define SLOT(o, s)                                                              \
  do {                                                                          \
    s = (int)PyLong_AsLong(o);                                                  \
    if (!PyErr_Occurred() && (s < 0 || s >= n_slots)) PyErr_SetString(PyExc_ValueError, "record: a slot that is not there"); \
    if (PyErr_Occurred()) goto fail;                                            \
  } while (0)
  for (int i = 0; i < n_ops; i++) {
    PyObject *op = PyList_GET_ITEM(ops, i);
    const char *kind = PyUnicode_AsUTF8(PyTuple_GET_ITEM(op, 0));
    Op *o = &r->ops[i];
    if (!kind) goto fail;
    if (kind[0] == 'a') {
      o->kind = OP_ALLOC;
      SLOT(PyTuple_GET_ITEM(op, 1), o->slot);
      o->value = PyLong_AsLongLong(PyTuple_GET_ITEM(op, 2));
    } else if (kind[0] == 'f') {
      o->kind = OP_FREE;
      SLOT(PyTuple_GET_ITEM(op, 1), o->slot);
    } else {
      o->kind = OP_CALL;
      o->value = PyLong_AsLongLong(PyTuple_GET_ITEM(op, 1));
      PyObject *list = PyTuple_GET_ITEM(op, 2);
      const Py_ssize_t n = PyList_GET_SIZE(list);
      if (n > MAX_ARGS) {
        PyErr_SetString(PyExc_ValueError, "record: too many arguments");
        goto fail;
      }
      o->first_patch = patch, o->first_list = list_no;
      for (Py_ssize_t j = 0; j < n; j++) {
        PyObject *v = PyList_GET_ITEM(list, j);
        if (!PyTuple_Check(v)) o->args[j] = PyLong_AsLongLong(v);
        else if (PyList_Check(PyTuple_GET_ITEM(v, 1))) {
          PyObject *slots = PyTuple_GET_ITEM(v, 1);
          HandleList *h = &r->lists[list_no++];
          h->at = (int)j, h->first = list_slot, h->count = (int)PyList_GET_SIZE(slots);
          for (int q = 0; q < h->count; q++, list_slot++) SLOT(PyList_GET_ITEM(slots, q), r->list_slots[list_slot]);
        } else {
          Patch *p = &r->patches[patch++];
          p->at = (int)j;
          SLOT(PyTuple_GET_ITEM(v, 1), p->slot);
        }
        if (PyErr_Occurred()) goto fail;
      }
      o->n_patches = patch - o->first_patch, o->n_lists = list_no - o->first_list;
    }
    if (PyErr_Occurred()) goto fail;
  }
  for (int i = 0; i < n_outs; i++) {
    PyObject *type, *shape, *names;
    int slot;
    if (!PyArg_ParseTuple(PyList_GET_ITEM(outs, i), "inOOO", &slot, &r->out_bytes[i], &type, &shape, &names)) goto fail;
    if (slot < n_params || slot >= n_slots) {
      PyErr_SetString(PyExc_ValueError, "record: a result that was not made here");
      goto fail;
    }
    Py_INCREF(type), Py_INCREF(shape), Py_INCREF(names);
    r->out_type[i] = type, r->out_shape[i] = shape, r->out_names[i] = names;
    r->outs[i] = slot;
    r->n_outs = i + 1;
  }
#undef SLOT
  return (PyObject *)r;
fail:
  Py_DECREF(r);
  return NULL;
}

/* whether a tensor has this (type, shape) */
static int is_shaped(PyObject *tensor, PyObject *want) {
  if (Py_TYPE(tensor) != tensor_type) return 0;
  int same = 1;
  for (int i = 0; same && i < 2; i++) {
    PyObject *have = PyObject_GenericGetAttr(tensor, i ? s_shape : s_type), *w = PyTuple_GET_ITEM(want, i);
    same = have && (have == w || PyObject_RichCompareBool(have, w, Py_EQ) == 1);
    Py_XDECREF(have);
  }
  PyErr_Clear();
  return same;
}

static PyObject *replay_call(Replay *self, PyObject *args, PyObject *kw) {
  enum { ON_STACK = 64 };
  void *stack_slots[ON_STACK], *handles[MAX_ARGS * 2], **slot = stack_slots;
  Ref *stack_refs[ON_STACK], **in = stack_refs;
  PyObject *result = NULL;
  if (PyTuple_GET_SIZE(args) != self->n_params || is_recording()) Py_RETURN_NONE;
  if (self->n_slots > ON_STACK) {
    slot = PyMem_Calloc(self->n_slots, sizeof(void *));
    in = PyMem_Calloc(self->n_slots, sizeof(Ref *));
    if (!slot || !in) {
      PyMem_Free(slot);
      PyMem_Free(in);
      return PyErr_NoMemory();
    }
  }
  memset(slot, 0, self->n_slots * sizeof(void *));
  int n_in = 0, status = 0;
  for (; n_in < self->n_params; n_in++) {
    if (n_in < PyTuple_GET_SIZE(self->shapes) && !is_shaped(PyTuple_GET_ITEM(args, n_in), PyTuple_GET_ITEM(self->shapes, n_in))) break;
    in[n_in] = live_ref(PyTuple_GET_ITEM(args, n_in), self->device);
    if (!in[n_in]) break;
    slot[n_in] = in[n_in]->handle;
  }
  if (n_in < self->n_params) goto refused;
  Py_BEGIN_ALLOW_THREADS
  for (int i = 0; i < self->n_ops && !status; i++) {
    const Op *o = &self->ops[i];
    if (o->kind == OP_ALLOC) status = buf_alloc((void *)(intptr_t)self->ctx_value, (size_t)o->value, &slot[o->slot]);
    else if (o->kind == OP_FREE) {
      buf_destroy(slot[o->slot]);
      slot[o->slot] = NULL;
    } else {
      int64_t a[MAX_ARGS];
      int used = 0;
      memcpy(a, o->args, sizeof(a));
      for (int p = 0; p < o->n_patches; p++) {
        const Patch *q = &self->patches[o->first_patch + p];
        a[q->at] = (int64_t)(intptr_t)slot[q->slot];
      }
      for (int l = 0; l < o->n_lists; l++) {
        const HandleList *h = &self->lists[o->first_list + l];
        if (used + h->count > MAX_ARGS * 2) {
          status = HIPNX_EINVAL;
          break;
        }
        a[h->at] = (int64_t)(intptr_t)&handles[used];
        for (int q = 0; q < h->count; q++) handles[used++] = slot[self->list_slots[h->first + q]];
      }
      if (!status) status = enter(o->value, a);
    }
  }
  if (status)
    for (int s = self->n_params; s < self->n_slots; s++)
      if (slot[s]) buf_destroy(slot[s]);
  Py_END_ALLOW_THREADS
  if (is_raised(status)) {
    raised(status);
    goto done;
  }
  if (status) goto refused;
  result = PyList_New(self->n_outs);
  for (int i = 0; result && i < self->n_outs; i++) {
    Ref *ref = new_ref(self->ctx, slot[self->outs[i]], self->out_bytes[i]);
    if (ref) slot[self->outs[i]] = NULL;
    PyObject *t = ref ? new_tensor(ref, self->device, self->out_type[i], self->out_shape[i], self->out_names[i]) : NULL;
    if (!t) Py_CLEAR(result);
    else PyList_SET_ITEM(result, i, t);
  }
  for (int s = self->n_params; s < self->n_slots; s++)  /* (what was not released on the way) */
    if (slot[s]) buf_destroy(slot[s]);
  goto done;
refused:
  result = Py_None;
  Py_INCREF(result);
done:
  for (int i = 0; i < n_in; i++) Py_DECREF(in[i]);
  if (slot != stack_slots) {
    PyMem_Free(slot);
    PyMem_Free(in);
  }
  return result;
}

/* ---- module ------------------------------------------------------------------------------------- */
static PyObject *setup(PyObject *mod, PyObject *a) {
  unsigned long long alloc, destroy;
  PyTypeObject *tensor, *backend;
  PyObject *check;
  if (!PyArg_ParseTuple(a, "KKO!O!O", &alloc, &destroy, &PyType_Type, &tensor, &PyType_Type, &backend, &check)) return NULL;
  buf_alloc = (int (*)(void *, size_t, void **))(uintptr_t)alloc;
  buf_destroy = (int (*)(void *))(uintptr_t)destroy;
  Py_INCREF(tensor);
  Py_INCREF(backend);
  Py_INCREF(check);
  raise_status = check;
  tensor_type = tensor, backend_type = backend;
  Py_RETURN_NONE;
}

/* fresh(ctx, ctx_value, nbytes) -> a Ref of the pool, or the library's status */
static PyObject *fresh(PyObject *mod, PyObject *const *a, Py_ssize_t n) {
  if (n != 3) return PyErr_Format(PyExc_TypeError, "fresh: three arguments");
  void *ctx = PyLong_AsVoidPtr(a[1]), *out = NULL;
  const Py_ssize_t nbytes = PyLong_AsSsize_t(a[2]);
  if (PyErr_Occurred()) return NULL;
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = buf_alloc(ctx, (size_t)nbytes, &out);
  Py_END_ALLOW_THREADS
  if (status) return PyLong_FromLong(status);
  Ref *r = new_ref(a[0], out, nbytes);
  if (!r) buf_destroy(out);
  return (PyObject *)r;
}

/* log_freed(list | None): the handles this thread releases go to the list from now on */
static PyObject *log_freed(PyObject *mod, PyObject *list) {
  freed_thread = PyThread_get_thread_ident();
  if (list != Py_None) Py_INCREF(list);
  PyObject *old = freed_log;
  freed_log = list == Py_None ? NULL : list;
  Py_XDECREF(old);
  Py_RETURN_NONE;
}

static PyMethodDef methods[] = {{"setup", setup, METH_VARARGS, NULL}, {"prepare", prepare, METH_VARARGS, NULL}, {"record", record, METH_VARARGS, NULL},
                                {"fresh", (PyCFunction)(void (*)(void))fresh, METH_FASTCALL, NULL}, {"log_freed", log_freed, METH_O, NULL}, {NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "hipnx_calls", "Callbacks and traced functions issued without Python in between.", -1, methods};

PyMODINIT_FUNC PyInit_hipnx_calls(void) {
  if (PyType_Ready(&RefType) < 0 || PyType_Ready(&CallType) < 0 || PyType_Ready(&ReplayType) < 0) return NULL;
  s_data = PyUnicode_InternFromString("data"), s_type = PyUnicode_InternFromString("type"), s_shape = PyUnicode_InternFromString("shape");
  s_names = PyUnicode_InternFromString("names"), s_ref = PyUnicode_InternFromString("ref"), s_device = PyUnicode_InternFromString("device");
  s_released = PyUnicode_InternFromString("released");
  PyObject *m = PyModule_Create(&module);
  if (m) {
    Py_INCREF(&RefType);
    PyModule_AddObject(m, "Ref", (PyObject *)&RefType);
  }
  return m;
}
