// The Python entry points of capi.py without ctypes' per-call work: a callable holds a C function, the names,
// defaults and kinds of its Python parameters and the order in which the C function takes them.
//
// What bounds the smallest calls is the host: through ctypes a call of 1 x 64 x 256 took 3.98 us in a loop, a C loop over the
// same function 2.55; through these callables 2.66 (1 x 4096 x 4096 back to back 3.95 -> 3.45, a batched paged
// attention call's host side 4.5 -> 2.9, a cache quantizer's 3.9 -> 2.6).
//
// Arguments of the usual types are converted here: a view of exactly the expected type, an int, and None for an
// address.  Anything else (another type, None for a number, a missing or unknown argument) goes to the ctypes function that
// stands behind the callable.
// Errors are raised as check() in capi.py raises them.  The interpreter lock is given up around the C function,
// as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>
#include <stddef.h>
#include <stdint.h>

namespace {

constexpr int MAX_ARGS = 16;
typedef int (*c_function)(long, long, long, long, long, long, long, long, long, long, long, long, long, long, long, long);

struct Call {
  PyObject_HEAD
  vectorcallfunc call;
  c_function fn;
  const char* (*last_error)(void);
  PyObject* slow;             // the same function through ctypes
  PyObject* names[MAX_ARGS];  // interned
  PyObject* views[MAX_ARGS];  // the type of a view argument, or null: an integer or an address
  bool addresses[MAX_ARGS];   // whether it is an address
  long defaults[MAX_ARGS];
  int slots[MAX_ARGS];        // place of the parameter among the C function's
  int count, required;
};

PyObject* call_vector(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  Call* const c = (Call*)self;
  const Py_ssize_t given = PyVectorcall_NARGS(nargsf), named = kwnames ? PyTuple_GET_SIZE(kwnames) : 0;
  PyObject* value[MAX_ARGS] = {};
  long a[MAX_ARGS] = {};
  Py_buffer held[4];
  int nheld = 0;
  bool usual = given <= c->count;
  if (usual) {
    for (Py_ssize_t i = 0; i < given; ++i) value[i] = args[i];
    for (Py_ssize_t k = 0; k < named && usual; ++k) {
      PyObject* const name = PyTuple_GET_ITEM(kwnames, k);
      int i = 0;
      while (i < c->count && c->names[i] != name) ++i;
      usual = i < c->count && !value[i];
      if (usual) value[i] = args[given + k];
    }
  }
  for (int i = 0; i < c->count && usual; ++i) {
    PyObject* const v = value[i];
    long out = c->defaults[i];
    if (!v) {
      usual = i >= c->required;
    } else if (c->views[i]) {
      usual = (PyObject*)Py_TYPE(v) == c->views[i] && nheld < 4 && PyObject_GetBuffer(v, &held[nheld], PyBUF_SIMPLE) == 0;
      if (usual) out = (long)(intptr_t)held[nheld++].buf;
    } else if (PyLong_Check(v)) {
      out = (long)PyLong_AsUnsignedLongLongMask(v);
      usual = !(out == -1 && PyErr_Occurred());
    } else {
      usual = v == Py_None && c->addresses[i];
      out = 0;
    }
    a[c->slots[i]] = out;
  }
  int rc = 0;
  if (usual) {
    Py_BEGIN_ALLOW_THREADS
    rc = c->fn(a[0], a[1], a[2], a[3], a[4], a[5], a[6], a[7], a[8], a[9], a[10], a[11], a[12], a[13], a[14], a[15]);
    Py_END_ALLOW_THREADS
  }
  while (nheld) PyBuffer_Release(&held[--nheld]);
  if (!usual) {
    PyErr_Clear();
    return PyObject_Vectorcall(c->slow, args, nargsf, kwnames);
  }
  if (rc == 0) Py_RETURN_NONE;
  PyErr_SetString(rc == 1 ? PyExc_ValueError : PyExc_RuntimeError, c->last_error());  // (1: W4_EINVAL)
  return nullptr;
}

void call_dealloc(PyObject* self) {
  Call* const c = (Call*)self;
  Py_XDECREF(c->slow);
  for (int i = 0; i < MAX_ARGS; ++i) {
    Py_XDECREF(c->names[i]);
    Py_XDECREF(c->views[i]);
  }
  PyTypeObject* const t = Py_TYPE(self);
  t->tp_free(self);
  Py_DECREF(t);
}

// What a function says of itself, from the one behind; pickled, as functions are, by its name in its module.
PyObject* call_attribute(PyObject* self, void* name) { return PyObject_GetAttrString(((Call*)self)->slow, (const char*)name); }
PyObject* call_reduce(PyObject* self, PyObject*) { return PyObject_GetAttrString(((Call*)self)->slow, "__qualname__"); }
PyObject* call_slow(PyObject* self, void*) {
  PyObject* const s = ((Call*)self)->slow;
  Py_INCREF(s);
  return s;
}
PyGetSetDef call_getset[] = {{"__doc__", call_attribute, nullptr, nullptr, (void*)"__doc__"},
                             {"__name__", call_attribute, nullptr, nullptr, (void*)"__name__"},
                             {"__qualname__", call_attribute, nullptr, nullptr, (void*)"__qualname__"},
                             {"__module__", call_attribute, nullptr, nullptr, (void*)"__module__"},
                             {"__wrapped__", call_slow, nullptr, nullptr, nullptr},
                             {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyMemberDef call_members[] = {{"__vectorcalloffset__", T_PYSSIZET, offsetof(Call, call), 1, nullptr},
                              {nullptr, 0, 0, 0, nullptr}};
PyMethodDef call_methods[] = {{"__reduce__", call_reduce, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};

PyType_Slot call_slots[] = {{Py_tp_dealloc, (void*)call_dealloc},
                            {Py_tp_call, (void*)PyVectorcall_Call},
                            {Py_tp_getset, (void*)call_getset},
                            {Py_tp_members, (void*)call_members},
                            {Py_tp_methods, (void*)call_methods},
                            {0, nullptr}};
PyType_Spec call_spec = {"w4calls.Call", sizeof(Call), 0, Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL, call_slots};
PyTypeObject* call_type = nullptr;

// make(function, last_error, slow, names, views, addresses, defaults, slots, required): addresses, the ctypes function,
// and a tuple for each property of the parameters
PyObject* make(PyObject*, PyObject* args) {
  unsigned long long fn, last_error;
  PyObject *slow, *names, *views, *addresses, *defaults, *slots;
  int required;
  if (!PyArg_ParseTuple(args, "KKOO!O!O!O!O!i", &fn, &last_error, &slow, &PyTuple_Type, &names, &PyTuple_Type, &views,
                        &PyTuple_Type, &addresses, &PyTuple_Type, &defaults, &PyTuple_Type, &slots, &required))
    return nullptr;
  const Py_ssize_t n = PyTuple_GET_SIZE(names);
  if (n > MAX_ARGS || PyTuple_GET_SIZE(views) != n || PyTuple_GET_SIZE(addresses) != n || PyTuple_GET_SIZE(defaults) != n ||
      PyTuple_GET_SIZE(slots) != n) {
    PyErr_SetString(PyExc_ValueError, "w4calls: the parameters' properties do not match");
    return nullptr;
  }
  Call* const c = (Call*)PyType_GenericAlloc(call_type, 0);
  if (!c) return nullptr;
  c->call = call_vector;
  c->fn = (c_function)(uintptr_t)fn;
  c->last_error = (const char* (*)(void))(uintptr_t)last_error;
  Py_INCREF(slow);
  c->slow = slow;
  c->count = (int)n;
  c->required = required;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* name = PyTuple_GET_ITEM(names, i);
    Py_INCREF(name);
    PyUnicode_InternInPlace(&name);
    c->names[i] = name;
    PyObject* const view = PyTuple_GET_ITEM(views, i);
    if (view != Py_None) {
      Py_INCREF(view);
      c->views[i] = view;
    }
    c->addresses[i] = PyTuple_GET_ITEM(addresses, i) == Py_True;
    c->defaults[i] = PyLong_AsLong(PyTuple_GET_ITEM(defaults, i));
    c->slots[i] = (int)PyLong_AsLong(PyTuple_GET_ITEM(slots, i));
    if (!PyErr_Occurred() && (c->slots[i] < 0 || c->slots[i] >= MAX_ARGS)) PyErr_SetString(PyExc_ValueError, "w4calls: bad slot");
    if (PyErr_Occurred()) {
      Py_DECREF(c);
      return nullptr;
    }
  }
  return (PyObject*)c;
}

PyMethodDef methods[] = {{"make", make, METH_VARARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "w4calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_w4calls(void) {
  if (!call_type) call_type = (PyTypeObject*)PyType_FromSpec(&call_spec);
  return call_type ? PyModule_Create(&module) : nullptr;
}
