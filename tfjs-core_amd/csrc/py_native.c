/* The part of the Python host that runs once or more per operation, as a CPython extension: the
 * tensor record, the engine's reference counts and scopes (tfjs-core/src/engine.ts:365-411,
 * 435-498, 502-572), the backend's table of buffers, and the entry points of the C ABI that
 * programs call most, without ctypes in between.  An eager program is a chain of short kernels
 * (2.4 us of host time each to launch), so what the host does around a launch decides its speed.
 * In interpreted code around ctypes tf.add took 8.8 us and tf.matmul 13.5 on the host.
 *
 * Everything here keeps the interfaces of the Python classes derived from it: engine.Tensor, engine.Engine
 * and backend_hip.MathBackendHIP.  Backends written in Python take part through their methods.
 * The interpreter lock is released around every call into the library, as ctypes does. */
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <dlfcn.h>
#include <structmember.h>

#include "tfjs_hip.h"

/* ---- the library ------------------------------------------------------------------------- */
#define API_LIST(X)                                                                              \
  X(tfhip_last_error) X(tfhip_register) X(tfhip_dispose) X(tfhip_write) X(tfhip_binary) X(tfhip_unary) \
  X(tfhip_matmul) X(tfhip_reduce) X(tfhip_reduce_axis) X(tfhip_softmax_rows) X(tfhip_conv2d)     \
  X(tfhip_separable_conv2d) X(tfhip_depthwise_conv2d) X(tfhip_pool2d)
#define MEMBER(name) __typeof__(&name) name;
static struct { API_LIST(MEMBER) } api;

static PyObject* native_load(PyObject* self, PyObject* arg) {
  (void)self;
  const char* path = PyUnicode_AsUTF8(arg);
  if (!path) return NULL;
  void* lib = dlopen(path, RTLD_NOW);
  if (!lib) return PyErr_Format(PyExc_RuntimeError, "%s", dlerror());
  __typeof__(api) found;
#define RESOLVE(name)                               \
  if (!(*(void**)&found.name = dlsym(lib, #name))) \
    return PyErr_Format(PyExc_RuntimeError, "%s has no %s", path, #name);
  API_LIST(RESOLVE)
  api = found;
  Py_RETURN_NONE;
}

/* ---- interned names and the classes derived in Python --------------------------------------- */
static PyObject *s_float32, *s_int32, *s_bool, *s_uint8q, *s_register, *s_dispose_data, *s_write, *s_dispose,
    *s_backend, *s_move_here, *s_data_id, *s_is_disposed;
static PyTypeObject *tensor_class, *backend_class;  /* engine.Tensor, MathBackendHIP */
static PyObject* flatten_tensors;                   /* engine._flatten_tensors */

static int same_text(PyObject* a, PyObject* interned, const char* text) {
  return a == interned || (PyUnicode_Check(a) && PyUnicode_CompareWithASCIIString(a, text) == 0);
}

/* ---- DataId: the opaque key of one backend buffer (tensor.ts:416) ---------------------------- */
typedef struct {
  PyObject_HEAD
  PyObject* weakrefs;
} DataIdObject;
static void DataId_dealloc(DataIdObject* self) {
  if (self->weakrefs) PyObject_ClearWeakRefs((PyObject*)self);
  Py_TYPE(self)->tp_free((PyObject*)self);
}
static PyTypeObject DataId_Type = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "tfhip._native.DataId",
    .tp_doc = "Opaque key of one backend buffer (tensor.ts:416).",
    .tp_basicsize = sizeof(DataIdObject),
    .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE,
    .tp_new = PyType_GenericNew,
    .tp_dealloc = (destructor)DataId_dealloc,
    .tp_weaklistoffset = offsetof(DataIdObject, weakrefs),
};

/* ---- types ------------------------------------------------------------------------------------ */
typedef struct {
  PyObject_HEAD
  PyObject *shape, *dtype, *size, *rank, *data_id, *quant, *is_disposed, *id;
} TensorObject;
typedef struct {
  PyObject_HEAD
  PyObject *ref;      /* data id -> [reference count, backend, bytes] */
  PyObject* scopes;   /* lists of tensors, the innermost last */
  PyObject* backend;  /* the active one, or None */
  long long num_tensors, num_bytes, num_data_buffers;
} EngineObject;
typedef struct {
  PyObject_HEAD
  PyObject* data;  /* data id -> (handle, code of the stored type, elements) */
  tfhip_ctx* ctx;
  long long next;
} BackendObject;
static PyTypeObject Tensor_Type, Engine_Type, Backend_Type;
static EngineObject* engine;
static long long next_tensor_id;

/* A field that was never set (a record made by __new__ alone) or was deleted: what Python says then. */
static int there(PyObject* field, const char* name) {
  if (!field) PyErr_Format(PyExc_AttributeError, "'%s' is not set", name);
  return field != NULL;
}

/* The arguments of a call by position or by name (METH_FASTCALL | METH_KEYWORDS) -> out, of which the first
 * `needed` have to be there; the others stay NULL.  At most 4. */
static int named(const char* call, PyObject* const* args, Py_ssize_t n, PyObject* keywords, const char* const* names,
                 int count, int needed, PyObject** out) {
  if (n > count) {
    PyErr_Format(PyExc_TypeError, "%s takes %d arguments, got %zd", call, count, n);
    return -1;
  }
  for (int i = 0; i < count; i++) out[i] = i < n ? args[i] : NULL;
  for (Py_ssize_t k = 0; keywords && k < PyTuple_GET_SIZE(keywords); k++) {
    PyObject* name = PyTuple_GET_ITEM(keywords, k);
    int i = 0;
    while (i < count && PyUnicode_CompareWithASCIIString(name, names[i])) i++;
    if (i == count || out[i]) {
      PyErr_Format(PyExc_TypeError, "%s: %s argument '%U'", call, i == count ? "no" : "a second", name);
      return -1;
    }
    out[i] = args[n + k];
  }
  for (int i = 0; i < needed; i++)
    if (!out[i]) {
      PyErr_Format(PyExc_TypeError, "%s needs the argument '%s'", call, names[i]);
      return -1;
    }
  return 0;
}
#define ARGUMENTS(call, count, needed, ...)                                      \
  PyObject* a[count];                                                            \
  static const char* const arg_names[] = {__VA_ARGS__};                          \
  if (named(call, args, n, keywords, arg_names, count, needed, a)) return NULL

/* ---- shapes ------------------------------------------------------------------------------------ */
static PyObject* as_shape(PyObject* shape) {  /* a tuple of ints; new reference */
  if (!there(shape, "shape")) return NULL;
  if (PyTuple_CheckExact(shape)) {
    Py_ssize_t i, n = PyTuple_GET_SIZE(shape);
    for (i = 0; i < n && PyLong_CheckExact(PyTuple_GET_ITEM(shape, i)); i++) {}
    if (i == n) {
      Py_INCREF(shape);
      return shape;
    }
  }
  PyObject* items = PySequence_List(shape);
  if (!items) return NULL;
  PyObject* out = PyTuple_New(PyList_GET_SIZE(items));
  for (Py_ssize_t i = 0; out && i < PyList_GET_SIZE(items); i++) {
    PyObject* d = PyNumber_Long(PyList_GET_ITEM(items, i));
    if (d) PyTuple_SET_ITEM(out, i, d);
    else Py_CLEAR(out);
  }
  Py_DECREF(items);
  return out;
}

/* The product of a shape as a Python int (any size). */
static PyObject* product(PyObject* shape) {
  long long n = 1;
  Py_ssize_t i, rank = PyTuple_GET_SIZE(shape);
  for (i = 0; i < rank; i++) {
    const long long d = PyLong_AsLongLong(PyTuple_GET_ITEM(shape, i));
    if (d == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      break;
    }
    if (__builtin_mul_overflow(n, d, &n)) break;
  }
  if (i == rank) return PyLong_FromLongLong(n);
  PyObject* p = PyLong_FromLong(1);
  for (i = 0; p && i < rank; i++) {
    PyObject* q = PyNumber_Multiply(p, PyTuple_GET_ITEM(shape, i));
    Py_DECREF(p);
    p = q;
  }
  return p;
}

#define MAX_DIMS 64
/* Dimensions as the library takes them (it checks the rank itself: 8 at most). */
static int dims_of(PyObject* shape, int32_t* dims) {
  if (!there(shape, "shape")) return -1;
  if (!PyTuple_Check(shape)) {
    PyErr_SetString(PyExc_TypeError, "a tensor's shape is a tuple");
    return -1;
  }
  const Py_ssize_t n = PyTuple_GET_SIZE(shape);
  for (Py_ssize_t i = 0; i < n && i < MAX_DIMS; i++)
    dims[i] = (int32_t)PyLong_AsUnsignedLongLongMask(PyTuple_GET_ITEM(shape, i));
  return PyErr_Occurred() ? -1 : (int)n;
}

/* ---- the backend's buffers ------------------------------------------------------------------ */
static int check(BackendObject* be, int rc) {
  if (rc == 0) return 0;
  PyErr_SetString(PyExc_RuntimeError, api.tfhip_last_error(be->ctx));
  return -1;
}

static int backend_register(BackendObject* be, PyObject* data_id, PyObject* shape, PyObject* dtype) {
  const int known = PyDict_Contains(be->data, data_id);
  if (known < 0) return -1;
  if (known) {
    PyErr_SetString(PyExc_RuntimeError, "Data buffer is already registered");
    return -1;
  }
  int code;
  if (same_text(dtype, s_float32, "float32")) code = TFHIP_FLOAT32;
  else if (same_text(dtype, s_int32, "int32")) code = TFHIP_INT32;
  else if (same_text(dtype, s_bool, "bool")) code = TFHIP_BOOL;
  else if (same_text(dtype, s_uint8q, "uint8q")) code = TFHIP_UINT8Q;
  else {
    PyErr_SetObject(PyExc_KeyError, dtype);
    return -1;
  }
  int32_t dims[MAX_DIMS];
  const int rank = dims_of(shape, dims);
  if (rank < 0) return -1;
  const long long handle = be->next++;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.tfhip_register(be->ctx, handle, dims, rank, code);
  Py_END_ALLOW_THREADS
  if (check(be, rc)) return -1;
  PyObject* n = product(shape);
  PyObject* rec = n ? Py_BuildValue("(LiN)", handle, code, n) : NULL;
  if (!rec) return -1;
  const int set = PyDict_SetItem(be->data, data_id, rec);
  Py_DECREF(rec);
  return set;
}

static int backend_dispose_data(BackendObject* be, PyObject* data_id) {
  PyObject* rec = PyDict_GetItemWithError(be->data, data_id);
  if (!rec) return PyErr_Occurred() ? -1 : 0;
  const long long handle = PyLong_AsLongLong(PyTuple_GET_ITEM(rec, 0));
  if (PyDict_DelItem(be->data, data_id)) return -1;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.tfhip_dispose(be->ctx, handle);
  Py_END_ALLOW_THREADS
  return check(be, rc);
}

/* The library's handle of a tensor's buffer; one that lives on another backend is moved here first. */
static int handle_of(BackendObject* be, PyObject* t, int64_t* handle) {
  PyObject* id;
  if (PyObject_TypeCheck(t, &Tensor_Type) && ((TensorObject*)t)->data_id) {
    id = ((TensorObject*)t)->data_id;
    Py_INCREF(id);
  } else if (!(id = PyObject_GetAttr(t, s_data_id))) {
    return -1;
  }
  PyObject* rec = PyDict_GetItemWithError(be->data, id);
  Py_DECREF(id);
  if (rec) {
    *handle = PyLong_AsLongLong(PyTuple_GET_ITEM(rec, 0));
    return 0;
  }
  if (PyErr_Occurred()) return -1;
  PyObject* moved = PyObject_CallMethodObjArgs((PyObject*)be, s_move_here, t, NULL);
  if (!moved) return -1;
  *handle = PyLong_AsLongLong(moved);
  Py_DECREF(moved);
  return *handle == -1 && PyErr_Occurred() ? -1 : 0;
}

/* Contiguous values of the stored type straight to the library; 0: not such values (the Python
 * method converts them, or refuses), 1: written, -1: failed. */
static int backend_write_plain(BackendObject* be, PyObject* data_id, PyObject* values) {
  static const char formats[] = {'f', 'i', 'B', 'B'};
  PyObject* rec = PyDict_GetItemWithError(be->data, data_id);
  if (!rec) return PyErr_Occurred() ? -1 : 0;
  const long long handle = PyLong_AsLongLong(PyTuple_GET_ITEM(rec, 0));
  const long code = PyLong_AsLong(PyTuple_GET_ITEM(rec, 1));
  const long long count = PyLong_AsLongLong(PyTuple_GET_ITEM(rec, 2));
  if (PyErr_Occurred()) return -1;
  Py_buffer view;
  if (!PyObject_CheckBuffer(values)) return 0;
  if (PyObject_GetBuffer(values, &view, PyBUF_C_CONTIGUOUS | PyBUF_FORMAT)) {
    PyErr_Clear();
    return 0;
  }
  int rc = 0;
  const int fits = code >= 0 && code < 4 && view.format && view.format[0] == formats[code] && !view.format[1] &&
                   view.itemsize == (code == TFHIP_FLOAT32 || code == TFHIP_INT32 ? 4 : 1) &&
                   view.len == count * view.itemsize;
  if (fits) {
    Py_BEGIN_ALLOW_THREADS
    rc = api.tfhip_write(be->ctx, handle, view.buf, (size_t)view.len);
    Py_END_ALLOW_THREADS
  }
  PyBuffer_Release(&view);
  if (!fits) return 0;
  return check(be, rc) ? -1 : 1;
}

/* ---- engine -------------------------------------------------------------------------------- */
static int engine_register(EngineObject* e, TensorObject* t, PyObject* backend, PyObject* storage) {
  PyObject* be = backend && backend != Py_None ? backend : e->backend;
  if (be && be != Py_None) Py_INCREF(be);
  else if (!(be = PyObject_GetAttr((PyObject*)e, s_backend))) return -1;
  int rc = -1;
  PyObject* rec = PyDict_GetItemWithError(e->ref, t->data_id);
  if (!rec) {
    if (PyErr_Occurred()) goto out;
    const int narrow = same_text(storage, s_bool, "bool") || same_text(storage, s_uint8q, "uint8q");
    long long bytes = PyLong_AsLongLong(t->size);
    if (bytes == -1 && PyErr_Occurred()) goto out;
    bytes *= narrow ? 1 : 4;
    if (!(rec = Py_BuildValue("[iOL]", 0, be, bytes))) goto out;
    const int set = PyDict_SetItem(e->ref, t->data_id, rec);
    Py_DECREF(rec);  /* (the dict holds it) */
    if (set) goto out;
    e->num_data_buffers++;
    e->num_bytes += bytes;
    if (Py_TYPE(be) == backend_class) {
      if (backend_register((BackendObject*)be, t->data_id, t->shape, storage)) goto out;
    } else {
      PyObject* r = PyObject_CallMethodObjArgs(be, s_register, t->data_id, t->shape, storage, NULL);
      if (!r) goto out;
      Py_DECREF(r);
    }
    if (!(rec = PyDict_GetItemWithError(e->ref, t->data_id))) {
      if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, t->data_id);
      goto out;
    }
  }
  PyObject* count = PyLong_FromLongLong(PyLong_AsLongLong(PyList_GET_ITEM(rec, 0)) + 1);
  if (!count || PyList_SetItem(rec, 0, count)) goto out;
  e->num_tensors++;
  const Py_ssize_t depth = PyList_GET_SIZE(e->scopes);
  if (depth && PyList_Append(PyList_GET_ITEM(e->scopes, depth - 1), (PyObject*)t)) goto out;
  rc = 0;
out:
  Py_DECREF(be);
  return rc;
}

static int engine_dispose(EngineObject* e, TensorObject* t) {
  if (!there(t->data_id, "data_id")) return -1;
  PyObject* rec = PyDict_GetItemWithError(e->ref, t->data_id);
  if (!rec) return PyErr_Occurred() ? -1 : 0;
  e->num_tensors--;
  const long long count = PyLong_AsLongLong(PyList_GET_ITEM(rec, 0));
  if (count > 1) {
    PyObject* less = PyLong_FromLongLong(count - 1);
    return less ? PyList_SetItem(rec, 0, less) : -1;
  }
  PyObject *be = PyList_GET_ITEM(rec, 1), *id = t->data_id;
  const long long bytes = PyLong_AsLongLong(PyList_GET_ITEM(rec, 2));
  Py_INCREF(be);
  Py_INCREF(id);
  int rc;
  if (Py_TYPE(be) == backend_class) {
    rc = backend_dispose_data((BackendObject*)be, id);
  } else {
    PyObject* r = PyObject_CallMethodObjArgs(be, s_dispose_data, id, NULL);
    rc = r ? 0 : -1;
    Py_XDECREF(r);
  }
  if (!rc) {
    e->num_data_buffers--;
    e->num_bytes -= bytes;
    rc = PyDict_DelItem(e->ref, id);
  }
  Py_DECREF(be);
  Py_DECREF(id);
  return rc;
}

static int tensor_dispose(TensorObject* t) {
  if (!there(t->is_disposed, "is_disposed") || !there((PyObject*)engine, "engine")) return -1;
  const int gone = PyObject_IsTrue(t->is_disposed);
  if (gone) return gone < 0 ? -1 : 0;
  if (engine_dispose(engine, t)) return -1;
  Py_INCREF(Py_True);
  Py_SETREF(t->is_disposed, Py_True);
  return 0;
}

/* The innermost scope ends: what `result` holds moves to the scope around it, the rest is disposed. */
static int engine_end_scope(EngineObject* e, PyObject* result) {
  const Py_ssize_t depth = PyList_GET_SIZE(e->scopes);
  if (!depth) {
    PyErr_SetString(PyExc_IndexError, "pop from empty list");
    return -1;
  }
  PyObject* scope = PyList_GET_ITEM(e->scopes, depth - 1);
  Py_INCREF(scope);
  if (PyList_SetSlice(e->scopes, depth - 1, depth, NULL)) {
    Py_DECREF(scope);
    return -1;
  }
  PyObject *outer = NULL, *held = NULL;
  PyObject *keep = NULL, *ids = NULL;  /* a list of tensors; their addresses, where it is long */
  int rc = -1;
  if (PyList_GET_SIZE(scope) == 0) {
    rc = 0;
    goto out;
  }
  if (result != Py_None && !PyObject_TypeCheck(result, &Tensor_Type)) {
    if (!(keep = PyObject_CallFunctionObjArgs(flatten_tensors, result, NULL))) goto out;
    if (PyList_GET_SIZE(keep) > 16) {
      if (!(ids = PySet_New(NULL))) goto out;
      for (Py_ssize_t i = 0; i < PyList_GET_SIZE(keep); i++) {
        PyObject* a = PyLong_FromVoidPtr(PyList_GET_ITEM(keep, i));
        if (!a || PySet_Add(ids, a)) {
          Py_XDECREF(a);
          goto out;
        }
        Py_DECREF(a);
      }
    }
  }
  /* (a backend written in Python may do anything while a tensor goes: hold what is looked at) */
  if (depth > 1) {
    outer = PyList_GET_ITEM(e->scopes, depth - 2);
    Py_INCREF(outer);
  }
  for (Py_ssize_t i = 0; i < PyList_GET_SIZE(scope); i++) {
    PyObject* t = PyList_GET_ITEM(scope, i);
    Py_INCREF(t);
    Py_XSETREF(held, t);
    int kept = t == result;
    if (ids) {
      PyObject* a = PyLong_FromVoidPtr(t);
      kept = a ? PySet_Contains(ids, a) : -1;
      Py_XDECREF(a);
      if (kept < 0) goto out;
    } else if (keep) {
      for (Py_ssize_t j = 0; j < PyList_GET_SIZE(keep) && !kept; j++) kept = PyList_GET_ITEM(keep, j) == t;
    }
    if (kept) {
      if (outer && PyList_Append(outer, t)) goto out;
    } else if (Py_TYPE(t) == tensor_class) {
      if (tensor_dispose((TensorObject*)t)) goto out;
    } else {
      PyObject* gone = PyObject_GetAttr(t, s_is_disposed);
      const int is = gone ? PyObject_IsTrue(gone) : -1;
      Py_XDECREF(gone);
      if (is < 0) goto out;
      if (!is) {
        PyObject* r = PyObject_CallMethodObjArgs(t, s_dispose, NULL);
        if (!r) goto out;
        Py_DECREF(r);
      }
    }
  }
  rc = 0;
out:
  Py_XDECREF(held);
  Py_XDECREF(outer);
  Py_XDECREF(ids);
  Py_XDECREF(keep);
  Py_DECREF(scope);
  return rc;
}

static int engine_start_scope(EngineObject* e) {
  PyObject* scope = PyList_New(0);
  if (!scope) return -1;
  const int rc = PyList_Append(e->scopes, scope);
  Py_DECREF(scope);
  return rc;
}

/* fn(arg) (or fn()) inside a scope of its own. */
static PyObject* engine_scoped(EngineObject* e, PyObject* fn, PyObject* arg) {
  if (engine_start_scope(e)) return NULL;
  PyObject* result = arg ? PyObject_CallOneArg(fn, arg) : PyObject_CallNoArgs(fn);
  if (!result) {
    PyObject *type, *value, *trace;
    PyErr_Fetch(&type, &value, &trace);
    if (engine_end_scope(e, Py_None)) PyErr_Clear();
    PyErr_Restore(type, value, trace);
    return NULL;
  }
  if (engine_end_scope(e, result)) Py_CLEAR(result);
  return result;
}

static int Engine_traverse(EngineObject* e, visitproc visit, void* arg) {
  Py_VISIT(e->ref);
  Py_VISIT(e->scopes);
  Py_VISIT(e->backend);
  return 0;
}
static int Engine_clear(EngineObject* e) {
  Py_CLEAR(e->ref);
  Py_CLEAR(e->scopes);
  Py_CLEAR(e->backend);
  return 0;
}
static void Engine_dealloc(EngineObject* e) {
  PyObject_GC_UnTrack(e);
  Engine_clear(e);
  Py_TYPE(e)->tp_free((PyObject*)e);
}
static PyObject* Engine_new(PyTypeObject* type, PyObject* args, PyObject* kwds) {
  (void)args, (void)kwds;
  EngineObject* e = (EngineObject*)type->tp_alloc(type, 0);
  if (!e) return NULL;
  e->ref = PyDict_New();
  e->scopes = PyList_New(0);
  Py_INCREF(Py_None);
  e->backend = Py_None;
  if (!e->ref || !e->scopes) Py_CLEAR(e);
  return (PyObject*)e;
}
static PyObject* Engine_register_tensor(EngineObject* e, PyObject* const* args, Py_ssize_t n, PyObject* keywords) {
  ARGUMENTS("register_tensor", 3, 3, "t", "backend", "storage_dtype");
  if (!PyObject_TypeCheck(a[0], &Tensor_Type)) return PyErr_Format(PyExc_TypeError, "register_tensor: not a tensor");
  TensorObject* t = (TensorObject*)a[0];
  if (!there(t->data_id, "data_id") || !there(t->shape, "shape") || !there(t->size, "size")) return NULL;
  const int given = PyObject_IsTrue(a[1]);
  if (given < 0 || engine_register(e, t, given ? a[1] : Py_None, a[2])) return NULL;
  Py_RETURN_NONE;
}
static PyObject* Engine_dispose_tensor(EngineObject* e, PyObject* const* args, Py_ssize_t n, PyObject* keywords) {
  ARGUMENTS("dispose_tensor", 1, 1, "t");
  if (!PyObject_TypeCheck(a[0], &Tensor_Type)) return PyErr_Format(PyExc_TypeError, "dispose_tensor: not a tensor");
  if (engine_dispose(e, (TensorObject*)a[0])) return NULL;
  Py_RETURN_NONE;
}
static PyObject* Engine_start(EngineObject* e, PyObject* unused) {
  (void)unused;
  if (engine_start_scope(e)) return NULL;
  Py_RETURN_NONE;
}
static PyObject* Engine_end(EngineObject* e, PyObject* const* args, Py_ssize_t n, PyObject* keywords) {
  ARGUMENTS("end_scope", 1, 0, "result");
  if (engine_end_scope(e, a[0] ? a[0] : Py_None)) return NULL;
  Py_RETURN_NONE;
}
static PyObject* Engine_scoped(EngineObject* e, PyObject* fn) { return engine_scoped(e, fn, NULL); }
static PyObject* Engine_run_kernel(EngineObject* e, PyObject* const* args, Py_ssize_t n, PyObject* keywords) {
  ARGUMENTS("run_kernel", 1, 1, "forward");
  PyObject* be = e->backend;
  if (!there(be, "_backend")) return NULL;
  if (be != Py_None) Py_INCREF(be);
  else if (!(be = PyObject_GetAttr((PyObject*)e, s_backend))) return NULL;
  PyObject* r = engine_scoped(e, a[0], be);
  Py_DECREF(be);
  return r;
}
static PyMemberDef Engine_members[] = {
    {"ref", T_OBJECT_EX, offsetof(EngineObject, ref), READONLY, "data id -> [reference count, backend, bytes]"},
    {"scopes", T_OBJECT_EX, offsetof(EngineObject, scopes), READONLY, "open scopes, the innermost last"},
    {"_backend", T_OBJECT_EX, offsetof(EngineObject, backend), 0, "the active backend, or None"},
    {"num_tensors", T_LONGLONG, offsetof(EngineObject, num_tensors), 0, NULL},
    {"num_bytes", T_LONGLONG, offsetof(EngineObject, num_bytes), 0, NULL},
    {"num_data_buffers", T_LONGLONG, offsetof(EngineObject, num_data_buffers), 0, NULL},
    {NULL}};
#define NAMED(name, fn, doc) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL | METH_KEYWORDS, doc}
static PyMethodDef Engine_methods[] = {
    NAMED("register_tensor", Engine_register_tensor, "register_tensor(t, backend, storage_dtype): engine.ts:502-530"),
    NAMED("dispose_tensor", Engine_dispose_tensor, "dispose_tensor(t): engine.ts:540-572"),
    {"start_scope", (PyCFunction)Engine_start, METH_NOARGS, "engine.ts:675-690"},
    NAMED("end_scope", Engine_end, "end_scope(result=None): engine.ts:691-718"),
    {"scoped", (PyCFunction)Engine_scoped, METH_O, "fn() inside a scope of its own; what it returns is kept."},
    NAMED("run_kernel", Engine_run_kernel,
          "run_kernel(forward): ENGINE.runKernel without a tape (engine.ts:435-498): the forward function gets the "
          "active backend; intermediates made inside are released when it returns."),
    {NULL}};
static PyTypeObject Engine_Type = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "tfhip._native.EngineCore",
    .tp_doc = "Reference counts of data ids and tidy scopes.",
    .tp_basicsize = sizeof(EngineObject),
    .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC,
    .tp_new = Engine_new,
    .tp_traverse = (traverseproc)Engine_traverse,
    .tp_clear = (inquiry)Engine_clear,
    .tp_dealloc = (destructor)Engine_dealloc,
    .tp_members = Engine_members,
    .tp_methods = Engine_methods,
};

/* ---- tensor -------------------------------------------------------------------------------- */
/* Fills a fresh record and registers it; `shape` is a tuple of ints. */
static int tensor_fill(TensorObject* t, PyObject* shape, PyObject* dtype, PyObject* data_id, PyObject* backend,
                       PyObject* quant, PyObject* storage) {
  Py_INCREF(shape);
  Py_XSETREF(t->shape, shape);
  Py_INCREF(dtype);
  Py_XSETREF(t->dtype, dtype);
  Py_XSETREF(t->size, product(shape));
  Py_XSETREF(t->rank, PyLong_FromSsize_t(PyTuple_GET_SIZE(shape)));
  if (data_id && data_id != Py_None) Py_INCREF(data_id);
  else data_id = DataId_Type.tp_alloc(&DataId_Type, 0);
  Py_XSETREF(t->data_id, data_id);
  Py_INCREF(quant);
  Py_XSETREF(t->quant, quant);
  Py_INCREF(Py_False);
  Py_XSETREF(t->is_disposed, Py_False);
  Py_XSETREF(t->id, PyLong_FromLongLong(next_tensor_id++));
  if (!t->size || !t->rank || !t->data_id || !t->id) return -1;
  return engine_register(engine, t, backend, storage);
}

/* A tensor of the class derived in Python. */
static PyObject* make_tensor(PyObject* shape, PyObject* dtype, PyObject* data_id, PyObject* backend, PyObject* quant,
                             PyObject* storage) {
  PyObject* dims = as_shape(shape);
  if (!dims) return NULL;
  TensorObject* t = (TensorObject*)tensor_class->tp_alloc(tensor_class, 0);
  if (t && tensor_fill(t, dims, dtype, data_id, backend, quant, storage)) Py_CLEAR(t);
  Py_DECREF(dims);
  return (PyObject*)t;
}

static int Tensor_init(TensorObject* t, PyObject* args, PyObject* kwds) {
  static char* names[] = {"shape", "dtype", "data_id", "values", "backend", "quant", "storage_dtype", NULL};
  PyObject *shape, *dtype, *data_id = Py_None, *values = Py_None, *backend = Py_None, *quant = Py_None,
                           *storage = Py_None;
  if (!PyArg_ParseTupleAndKeywords(args, kwds, "OO|OOOOO", names, &shape, &dtype, &data_id, &values, &backend, &quant,
                                   &storage))
    return -1;
  if (!engine) {
    PyErr_SetString(PyExc_RuntimeError, "tfhip._native: no engine");
    return -1;
  }
  const int typed = PyObject_IsTrue(dtype), quantised = PyObject_IsTrue(quant), stored = PyObject_IsTrue(storage);
  if (typed < 0 || quantised < 0 || stored < 0) return -1;
  if (!typed) dtype = s_float32;
  if (!stored) storage = quantised ? s_uint8q : dtype;
  PyObject* dims = as_shape(shape);
  if (!dims) return -1;
  int rc = tensor_fill(t, dims, dtype, data_id, backend, quant, storage);
  Py_DECREF(dims);
  if (!rc && values != Py_None) {
    PyObject* to = backend != Py_None ? backend : engine->backend;
    if (to && Py_TYPE(to) == backend_class) {
      const int written = backend_write_plain((BackendObject*)to, t->data_id, values);
      if (written) return written > 0 ? 0 : -1;
    }
    PyObject* r = PyObject_CallMethodObjArgs((PyObject*)engine, s_write, backend, t->data_id, values, NULL);
    rc = r ? 0 : -1;
    Py_XDECREF(r);
  }
  return rc;
}
static int Tensor_traverse(TensorObject* t, visitproc visit, void* arg) {
  Py_VISIT(t->shape);
  Py_VISIT(t->dtype);
  Py_VISIT(t->data_id);
  Py_VISIT(t->quant);
  return 0;
}
static int Tensor_clear(TensorObject* t) {
  Py_CLEAR(t->shape);
  Py_CLEAR(t->dtype);
  Py_CLEAR(t->size);
  Py_CLEAR(t->rank);
  Py_CLEAR(t->data_id);
  Py_CLEAR(t->quant);
  Py_CLEAR(t->is_disposed);
  Py_CLEAR(t->id);
  return 0;
}
static void Tensor_dealloc(TensorObject* t) {
  PyObject_GC_UnTrack(t);
  Tensor_clear(t);
  Py_TYPE(t)->tp_free((PyObject*)t);
}
static PyObject* Tensor_dispose(TensorObject* t, PyObject* unused) {
  (void)unused;
  if (tensor_dispose(t)) return NULL;
  Py_RETURN_NONE;
}
static PyMemberDef Tensor_members[] = {
    {"shape", T_OBJECT_EX, offsetof(TensorObject, shape), 0, NULL},
    {"dtype", T_OBJECT_EX, offsetof(TensorObject, dtype), 0, NULL},
    {"size", T_OBJECT_EX, offsetof(TensorObject, size), 0, NULL},
    {"rank", T_OBJECT_EX, offsetof(TensorObject, rank), 0, NULL},
    {"data_id", T_OBJECT_EX, offsetof(TensorObject, data_id), 0, NULL},
    {"quant", T_OBJECT_EX, offsetof(TensorObject, quant), 0,
     "(scale, min) when the buffer holds uint8 affine-quantised weights"},
    {"is_disposed", T_OBJECT_EX, offsetof(TensorObject, is_disposed), 0, NULL},
    {"id", T_OBJECT_EX, offsetof(TensorObject, id), 0, NULL},
    {NULL}};
static PyMethodDef Tensor_methods[] = {{"dispose", (PyCFunction)Tensor_dispose, METH_NOARGS, "engine.ts:540-572"},
                                       {NULL}};
static PyTypeObject Tensor_Type = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "tfhip._native.TensorBase",
    .tp_doc = "Tensor(shape, dtype, data_id=None, values=None, backend=None, quant=None, storage_dtype=None)",
    .tp_basicsize = sizeof(TensorObject),
    .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC,
    .tp_new = PyType_GenericNew,
    .tp_init = (initproc)Tensor_init,
    .tp_traverse = (traverseproc)Tensor_traverse,
    .tp_clear = (inquiry)Tensor_clear,
    .tp_dealloc = (destructor)Tensor_dealloc,
    .tp_members = Tensor_members,
    .tp_methods = Tensor_methods,
};

/* ---- backend: buffers and the operations programs call most ------------------------------------ */
static int Backend_traverse(BackendObject* be, visitproc visit, void* arg) {
  Py_VISIT(be->data);
  return 0;
}
static int Backend_clear(BackendObject* be) {
  Py_CLEAR(be->data);
  return 0;
}
static void Backend_dealloc(BackendObject* be) {
  PyObject_GC_UnTrack(be);
  Backend_clear(be);
  Py_TYPE(be)->tp_free((PyObject*)be);
}
static PyObject* Backend_new(PyTypeObject* type, PyObject* args, PyObject* kwds) {
  (void)args, (void)kwds;
  if (!api.tfhip_last_error || !engine)
    return PyErr_Format(PyExc_RuntimeError, "tfhip._native: load the library and make the engine first");
  BackendObject* be = (BackendObject*)type->tp_alloc(type, 0);
  if (!be) return NULL;
  be->next = 1;
  if (!(be->data = PyDict_New())) Py_CLEAR(be);
  return (PyObject*)be;
}

static int arguments(const char* name, Py_ssize_t n, Py_ssize_t want) {
  if (n == want) return 0;
  PyErr_Format(PyExc_TypeError, "%s takes %zd arguments, got %zd", name, want, n);
  return -1;
}
/* Integer arguments: args[from .. from + count) -> out. */
static int integers(PyObject* const* args, int from, int count, long long* out) {
  for (int i = 0; i < count; i++)
    if ((out[i] = PyLong_AsLongLong(args[from + i])) == -1 && PyErr_Occurred()) return -1;
  return 0;
}
/* An operand that a call may go without: None, or a layout of 0, is -1. */
static int optional_handle(BackendObject* be, PyObject* t, long long kind, int64_t* handle) {
  *handle = -1;
  return t == Py_None || !kind ? 0 : handle_of(be, t, handle);
}
/* (scale, min) of quantised weights, in any sequence; None, or anything empty, for others. */
static int quant_of(PyObject* t, tfhip_qparams* q, const tfhip_qparams** out) {
  *out = NULL;
  if (!PyObject_TypeCheck(t, &Tensor_Type)) return 0;
  PyObject* v = ((TensorObject*)t)->quant;
  if (!there(v, "quant")) return -1;
  const int given = PyObject_IsTrue(v);
  if (given <= 0) return given;
  double* const values[] = {&q->scale, &q->min};
  for (int i = 0; i < 2; i++) {
    PyObject* item = PySequence_GetItem(v, i);
    if (!item) return -1;
    *values[i] = PyFloat_AsDouble(item);
    Py_DECREF(item);
    if (*values[i] == -1.0 && PyErr_Occurred()) return -1;
  }
  *out = q;
  return 0;
}
/* The geometry of a convolution or a pool, packed by the caller. */
static int geometry(PyObject* packed, tfhip_conv2d_info* info) {
  if (!PyBytes_Check(packed) || PyBytes_GET_SIZE(packed) != (Py_ssize_t)sizeof *info) {
    PyErr_SetString(PyExc_TypeError, "a packed tfhip_conv2d_info is needed");
    return -1;
  }
  memcpy(info, PyBytes_AS_STRING(packed), sizeof *info);
  return 0;
}
static PyObject* output(BackendObject* be, PyObject* shape, PyObject* dtype, int64_t* handle) {
  PyObject* t = make_tensor(shape, dtype, NULL, (PyObject*)be, Py_None, dtype);
  if (t && handle_of(be, t, handle)) Py_CLEAR(t);
  return t;
}
/* The call's result: the output, or what the library says went wrong. */
static PyObject* finish(BackendObject* be, int rc, PyObject* out) {
  if (check(be, rc)) Py_CLEAR(out);
  return out;
}
#define RUN(call)          \
  int rc;                  \
  Py_BEGIN_ALLOW_THREADS   \
  rc = (call);             \
  Py_END_ALLOW_THREADS     \
  return finish(be, rc, out)
#define NEED(name, want) \
  if (arguments(name, n, want)) return NULL
#define OR_DROP(test)  \
  if (test) {          \
    Py_DECREF(out);    \
    return NULL;       \
  }

static PyObject* Backend_bind(BackendObject* be, PyObject* address) {
  void* p = PyLong_AsVoidPtr(address);
  if (PyErr_Occurred()) return NULL;
  be->ctx = (tfhip_ctx*)p;
  Py_RETURN_NONE;
}
static PyObject* Backend_register(BackendObject* be, PyObject* const* args, Py_ssize_t n, PyObject* keywords) {
  ARGUMENTS("register", 3, 3, "data_id", "shape", "dtype");
  PyObject* dims = as_shape(a[1]);
  if (!dims) return NULL;
  const int rc = backend_register(be, a[0], dims, a[2]);
  Py_DECREF(dims);
  if (rc) return NULL;
  Py_RETURN_NONE;
}
static PyObject* Backend_dispose_data(BackendObject* be, PyObject* const* args, Py_ssize_t n, PyObject* keywords) {
  ARGUMENTS("dispose_data", 1, 1, "data_id");
  if (backend_dispose_data(be, a[0])) return NULL;
  Py_RETURN_NONE;
}
/* _write(data_id, contiguous array): the caller has checked its type and length. */
static PyObject* Backend_write(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  NEED("_write", 2);
  PyObject* rec = PyDict_GetItemWithError(be->data, args[0]);
  if (!rec) {
    if (!PyErr_Occurred()) PyErr_SetObject(PyExc_KeyError, args[0]);
    return NULL;
  }
  const long long handle = PyLong_AsLongLong(PyTuple_GET_ITEM(rec, 0));
  Py_buffer view;
  if (PyObject_GetBuffer(args[1], &view, PyBUF_SIMPLE)) return NULL;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.tfhip_write(be->ctx, handle, view.buf, (size_t)view.len);
  Py_END_ALLOW_THREADS
  PyBuffer_Release(&view);
  if (check(be, rc)) return NULL;
  Py_RETURN_NONE;
}
static PyObject* Backend_h(BackendObject* be, PyObject* t) {
  int64_t h;
  if (handle_of(be, t, &h)) return NULL;
  return PyLong_FromLongLong(h);
}
/* _out(shape, dtype="float32") */
static PyObject* Backend_out(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  if (n < 1 || n > 2) return PyErr_Format(PyExc_TypeError, "_out takes a shape and a dtype");
  PyObject* dtype = n == 2 ? args[1] : s_float32;
  return make_tensor(args[0], dtype, NULL, (PyObject*)be, Py_None, dtype);
}
/* _alias(x, shape): another tensor over x's data. */
static PyObject* Backend_alias(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  NEED("_alias", 2);
  if (!PyObject_TypeCheck(args[0], &Tensor_Type)) return PyErr_Format(PyExc_TypeError, "_alias: not a tensor");
  TensorObject* x = (TensorObject*)args[0];
  if (!there(x->data_id, "data_id") || !there(x->dtype, "dtype") || !there(x->quant, "quant")) return NULL;
  return make_tensor(args[1], x->dtype, x->data_id, (PyObject*)be, x->quant, x->dtype);
}
/* _binary_out(op, a, b, dtype): None when the shapes do not broadcast. */
static PyObject* Backend_binary(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  NEED("_binary_out", 4);
  const int op = (int)PyLong_AsLong(args[0]);
  if (op == -1 && PyErr_Occurred()) return NULL;
  if (!PyObject_TypeCheck(args[1], &Tensor_Type) || !PyObject_TypeCheck(args[2], &Tensor_Type))
    return PyErr_Format(PyExc_TypeError, "_binary_out: not a tensor");
  TensorObject *a = (TensorObject*)args[1], *b = (TensorObject*)args[2];
  int32_t da[MAX_DIMS], db[MAX_DIMS];
  const int ra = dims_of(a->shape, da), rb = dims_of(b->shape, db);
  if (ra < 0 || rb < 0) return NULL;
  if (ra > MAX_DIMS || rb > MAX_DIMS) Py_RETURN_NONE;
  PyObject* shape;
  if (ra == rb && memcmp(da, db, sizeof(int32_t) * (size_t)ra) == 0) {
    shape = a->shape;
    Py_INCREF(shape);
  } else {
    const int r = ra > rb ? ra : rb;
    if (!(shape = PyTuple_New(r))) return NULL;
    for (int i = 0; i < r; i++) {
      const int ia = i - (r - ra), ib = i - (r - rb);
      PyObject* pick;
      if (ia < 0 || (ib >= 0 && da[ia] == 1)) pick = PyTuple_GET_ITEM(b->shape, ib);
      else if (ib < 0 || db[ib] == 1 || da[ia] == db[ib]) pick = PyTuple_GET_ITEM(a->shape, ia);
      else {
        Py_DECREF(shape);
        Py_RETURN_NONE;
      }
      Py_INCREF(pick);
      PyTuple_SET_ITEM(shape, i, pick);
    }
  }
  int64_t ha, hb, ho;
  PyObject* out = output(be, shape, args[3], &ho);
  Py_DECREF(shape);
  if (!out) return NULL;
  OR_DROP(handle_of(be, args[1], &ha) || handle_of(be, args[2], &hb));
  RUN(api.tfhip_binary(be->ctx, op, ha, da, ra, hb, db, rb, ho));
}
/* _unary_out(op, x, dtype, p0, p1) */
static PyObject* Backend_unary(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  NEED("_unary_out", 5);
  const int op = (int)PyLong_AsLong(args[0]);
  const double p0 = PyFloat_AsDouble(args[3]), p1 = PyFloat_AsDouble(args[4]);
  if (PyErr_Occurred()) return NULL;
  if (!PyObject_TypeCheck(args[1], &Tensor_Type)) return PyErr_Format(PyExc_TypeError, "_unary_out: not a tensor");
  int64_t hx, ho;
  PyObject* out = output(be, ((TensorObject*)args[1])->shape, args[2], &ho);
  if (!out) return NULL;
  OR_DROP(handle_of(be, args[1], &hx));
  RUN(api.tfhip_unary(be->ctx, op, hx, ho, (float)p0, (float)p1));
}
/* _matmul_out(a, b, out_shape, batch, m, n, k, ta, tb, bias, bias_kind, act, prelu, prelu_kind) */
static PyObject* Backend_matmul(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  NEED("_matmul_out", 14);
  long long v[6], bk, act, pk;
  if (integers(args, 3, 6, v) || integers(args, 10, 1, &bk) || integers(args, 11, 1, &act) || integers(args, 13, 1, &pk))
    return NULL;
  int64_t ha, hb, ho, hbias, hprelu;
  tfhip_qparams qs;
  const tfhip_qparams* q;
  if (quant_of(args[1], &qs, &q)) return NULL;
  PyObject* out = output(be, args[2], s_float32, &ho);
  if (!out) return NULL;
  OR_DROP(handle_of(be, args[0], &ha) || handle_of(be, args[1], &hb) || optional_handle(be, args[9], bk, &hbias) ||
          optional_handle(be, args[12], pk, &hprelu));
  RUN(api.tfhip_matmul(be->ctx, ha, hb, ho, (int)v[0], (int)v[1], (int)v[2], (int)v[3], (int)v[4], (int)v[5], hbias,
                       (int)bk, (int)act, hprelu, (int)pk, q));
}
/* _reduce_axis_out(op, x, out_shape, dtype, outer, red, inner, divisor) */
static PyObject* Backend_reduce_axis(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  NEED("_reduce_axis_out", 8);
  long long op, v[3];
  if (integers(args, 0, 1, &op) || integers(args, 4, 3, v)) return NULL;
  const double divisor = PyFloat_AsDouble(args[7]);
  if (PyErr_Occurred()) return NULL;
  int64_t hx, ho;
  PyObject* out = output(be, args[2], args[3], &ho);
  if (!out) return NULL;
  OR_DROP(handle_of(be, args[1], &hx));
  RUN(api.tfhip_reduce_axis(be->ctx, (int)op, hx, ho, v[0], v[1], v[2], divisor));
}
/* _reduce_out(op, x, out_shape, dtype, outer, inner) */
static PyObject* Backend_reduce(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  NEED("_reduce_out", 6);
  long long op, v[2];
  if (integers(args, 0, 1, &op) || integers(args, 4, 2, v)) return NULL;
  int64_t hx, ho;
  PyObject* out = output(be, args[2], args[3], &ho);
  if (!out) return NULL;
  OR_DROP(handle_of(be, args[1], &hx));
  RUN(api.tfhip_reduce(be->ctx, (int)op, hx, ho, v[0], v[1]));
}
/* _softmax_out(x, rows, cols) */
static PyObject* Backend_softmax(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  NEED("_softmax_out", 3);
  long long v[2];
  if (integers(args, 1, 2, v)) return NULL;
  if (!PyObject_TypeCheck(args[0], &Tensor_Type)) return PyErr_Format(PyExc_TypeError, "_softmax_out: not a tensor");
  int64_t hx, ho;
  PyObject* out = output(be, ((TensorObject*)args[0])->shape, s_float32, &ho);
  if (!out) return NULL;
  OR_DROP(handle_of(be, args[0], &hx));
  RUN(api.tfhip_softmax_rows(be->ctx, hx, ho, v[0], v[1]));
}
/* _conv2d_out(x, filter, out_shape, info, bias, bias_kind, act, prelu, prelu_kind) */
static PyObject* Backend_conv2d(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  NEED("_conv2d_out", 9);
  long long v[2], pk;
  tfhip_conv2d_info info;
  tfhip_qparams qs;
  const tfhip_qparams* q;
  if (integers(args, 5, 2, v) || integers(args, 8, 1, &pk) || geometry(args[3], &info) || quant_of(args[1], &qs, &q))
    return NULL;
  int64_t hx, hw, ho, hb, hp;
  PyObject* out = output(be, args[2], s_float32, &ho);
  if (!out) return NULL;
  OR_DROP(handle_of(be, args[0], &hx) || handle_of(be, args[1], &hw) || optional_handle(be, args[4], v[0], &hb) ||
          optional_handle(be, args[7], pk, &hp));
  RUN(api.tfhip_conv2d(be->ctx, hx, hw, ho, &info, hb, (int)v[0], (int)v[1], hp, (int)pk, q));
}
/* _depthwise_out(x, filter, out_shape, info, bias, bias_kind, act) */
static PyObject* Backend_depthwise(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  NEED("_depthwise_out", 7);
  long long v[2];
  tfhip_conv2d_info info;
  tfhip_qparams qs;
  const tfhip_qparams* q;
  if (integers(args, 5, 2, v) || geometry(args[3], &info) || quant_of(args[1], &qs, &q)) return NULL;
  int64_t hx, hw, ho, hb;
  PyObject* out = output(be, args[2], s_float32, &ho);
  if (!out) return NULL;
  OR_DROP(handle_of(be, args[0], &hx) || handle_of(be, args[1], &hw) || optional_handle(be, args[4], v[0], &hb));
  RUN(api.tfhip_depthwise_conv2d(be->ctx, hx, hw, ho, &info, hb, (int)v[0], (int)v[1], q));
}
/* _separable_out(x, depthwise, pointwise, out_shape, info, dw_bias, dw_kind, dw_act, bias, kind, act) */
static PyObject* Backend_separable(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  NEED("_separable_out", 11);
  long long d[2], p[2];
  tfhip_conv2d_info info;
  tfhip_qparams dqs, pqs;
  const tfhip_qparams *dq, *pq;
  if (integers(args, 6, 2, d) || integers(args, 9, 2, p) || geometry(args[4], &info) || quant_of(args[1], &dqs, &dq) ||
      quant_of(args[2], &pqs, &pq))
    return NULL;
  int64_t hx, hd, hp, ho, hdb, hpb;
  PyObject* out = output(be, args[3], s_float32, &ho);
  if (!out) return NULL;
  OR_DROP(handle_of(be, args[0], &hx) || handle_of(be, args[1], &hd) || handle_of(be, args[2], &hp) ||
          optional_handle(be, args[5], d[0], &hdb) || optional_handle(be, args[8], p[0], &hpb));
  RUN(api.tfhip_separable_conv2d(be->ctx, hx, hd, hp, ho, &info, hdb, (int)d[0], (int)d[1], hpb, (int)p[0], (int)p[1],
                                 dq, pq));
}
/* _pool_out(x, out_shape, info, kind) */
static PyObject* Backend_pool(BackendObject* be, PyObject* const* args, Py_ssize_t n) {
  NEED("_pool_out", 4);
  long long kind;
  tfhip_conv2d_info info;
  if (integers(args, 3, 1, &kind) || geometry(args[2], &info)) return NULL;
  int64_t hx, ho;
  PyObject* out = output(be, args[1], s_float32, &ho);
  if (!out) return NULL;
  OR_DROP(handle_of(be, args[0], &hx));
  RUN(api.tfhip_pool2d(be->ctx, hx, ho, &info, (int)kind));
}
#define FAST(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, NULL}
static PyMemberDef Backend_members[] = {
    {"data", T_OBJECT_EX, offsetof(BackendObject, data), READONLY, "data id -> (handle, storage dtype code, numel)"},
    {NULL}};
static PyMethodDef Backend_methods[] = {
    {"_bind", (PyCFunction)Backend_bind, METH_O, "the address of the library's context, 0 for none"},
    NAMED("register", Backend_register, "register(data_id, shape, dtype)"),
    NAMED("dispose_data", Backend_dispose_data, "dispose_data(data_id)"),
    FAST("_write", Backend_write),
    {"_h", (PyCFunction)Backend_h, METH_O, "the library's handle of a tensor's buffer"},
    FAST("_out", Backend_out),
    FAST("_alias", Backend_alias),
    FAST("_binary_out", Backend_binary),
    FAST("_unary_out", Backend_unary),
    FAST("_matmul_out", Backend_matmul),
    FAST("_reduce_axis_out", Backend_reduce_axis),
    FAST("_reduce_out", Backend_reduce),
    FAST("_softmax_out", Backend_softmax),
    FAST("_conv2d_out", Backend_conv2d),
    FAST("_depthwise_out", Backend_depthwise),
    FAST("_separable_out", Backend_separable),
    FAST("_pool_out", Backend_pool),
    {NULL}};
static PyTypeObject Backend_Type = {
    PyVarObject_HEAD_INIT(NULL, 0).tp_name = "tfhip._native.BackendCore",
    .tp_doc = "Buffers of a context of libtfjs_hip.so and its most frequent entry points.",
    .tp_basicsize = sizeof(BackendObject),
    .tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_BASETYPE | Py_TPFLAGS_HAVE_GC,
    .tp_new = Backend_new,
    .tp_traverse = (traverseproc)Backend_traverse,
    .tp_clear = (inquiry)Backend_clear,
    .tp_dealloc = (destructor)Backend_dealloc,
    .tp_members = Backend_members,
    .tp_methods = Backend_methods,
};

/* ---- module ----------------------------------------------------------------------------------- */
static PyObject* native_set_engine(PyObject* self, PyObject* args) {
  (void)self;
  PyObject *e, *cls, *flatten;
  if (!PyArg_ParseTuple(args, "O!O!O", &Engine_Type, &e, &PyType_Type, &cls, &flatten)) return NULL;
  if (!PyType_IsSubtype((PyTypeObject*)cls, &Tensor_Type)) return PyErr_Format(PyExc_TypeError, "not a Tensor class");
  Py_INCREF(e);
  Py_XSETREF(engine, (EngineObject*)e);
  Py_INCREF(cls);
  Py_XSETREF(tensor_class, (PyTypeObject*)cls);
  Py_INCREF(flatten);
  Py_XSETREF(flatten_tensors, flatten);
  Py_RETURN_NONE;
}
static PyObject* native_set_backend_class(PyObject* self, PyObject* cls) {
  (void)self;
  if (!PyType_Check(cls) || !PyType_IsSubtype((PyTypeObject*)cls, &Backend_Type))
    return PyErr_Format(PyExc_TypeError, "not a class derived from BackendCore");
  Py_INCREF(cls);
  Py_XSETREF(backend_class, (PyTypeObject*)cls);
  Py_RETURN_NONE;
}
static PyMethodDef module_methods[] = {
    {"load", native_load, METH_O, "load(path): resolve the entry points of libtfjs_hip.so."},
    {"set_engine", native_set_engine, METH_VARARGS, "set_engine(engine, Tensor, flatten)"},
    {"set_backend_class", native_set_backend_class, METH_O, NULL},
    {NULL}};
static struct PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", NULL, -1, module_methods};

PyMODINIT_FUNC PyInit__native(void) {
  struct { PyObject** at; const char* text; } names[] = {
      {&s_float32, "float32"}, {&s_int32, "int32"}, {&s_bool, "bool"}, {&s_uint8q, "uint8q"},
      {&s_register, "register"}, {&s_dispose_data, "dispose_data"}, {&s_write, "write"}, {&s_dispose, "dispose"},
      {&s_backend, "backend"}, {&s_move_here, "_move_here"}, {&s_data_id, "data_id"},
      {&s_is_disposed, "is_disposed"}};
  for (size_t i = 0; i < sizeof names / sizeof *names; i++)
    if (!(*names[i].at = PyUnicode_InternFromString(names[i].text))) return NULL;
  PyObject* m = PyModule_Create(&module);
  if (!m || PyModule_AddType(m, &DataId_Type) || PyModule_AddType(m, &Tensor_Type) ||
      PyModule_AddType(m, &Engine_Type) || PyModule_AddType(m, &Backend_Type)) {
    Py_XDECREF(m);
    return NULL;
  }
  return m;
}
