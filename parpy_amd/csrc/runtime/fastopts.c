// Options of a call, built without the interpreter: `threads(n)` and `par({...})`.
//
// Programs write `opts=parpy.par({'i': parpy.threads(n), ...})` where the call stands, so two or three small objects are
// made per call.  The Python statements of it take 0.52 us of the 4.06 us that a call on 10 x 1000 floats takes, 2.6 of which are
// the launch; these take 0.23 (the call 3.74 us: medians of 25 times 4000 calls of each kind in turn, half of them within 0.02).  What is not plainly an int, or a dict of strings and LoopPar, goes to the Python
// functions, which decide and report everything.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>

typedef struct {
  PyTypeObject* par_type;       // LoopPar, and where it keeps nthreads, reduction and _tpb
  Py_ssize_t fields[3];
  PyObject* tpb;                // its default
  PyObject* options_type;
  PyObject *threads, *par;      // the Python functions
  PyObject* parallelize;        // the name
} State;

static State st;

static PyObject* plain_threads(PyObject* n) {
  PyObject* o = st.par_type->tp_alloc(st.par_type, 0);
  if (!o) return NULL;
  PyObject* const values[3] = {n, Py_False, st.tpb};
  for (int f = 0; f < 3; ++f) {
    Py_INCREF(values[f]);
    *(PyObject**)((char*)o + st.fields[f]) = values[f];
  }
  return o;
}

static PyObject* fast_threads(PyObject* self, PyObject* const* a, Py_ssize_t n, PyObject* names) {
  (void)self;
  if (n == 1 && !names && PyLong_CheckExact(a[0])) return plain_threads(a[0]);
  return PyObject_Vectorcall(st.threads, a, (size_t)n, names);
}

static int plain_mapping(PyObject* p) {
  if (!PyDict_CheckExact(p)) return 0;
  PyObject *k, *v;
  Py_ssize_t at = 0;
  while (PyDict_Next(p, &at, &k, &v))
    if (!PyUnicode_CheckExact(k) || Py_TYPE(v) != st.par_type) return 0;
  return 1;
}

static PyObject* fast_par(PyObject* self, PyObject* const* a, Py_ssize_t n, PyObject* names) {
  (void)self;
  if (n != 1 || names || !plain_mapping(a[0])) return PyObject_Vectorcall(st.par, a, (size_t)n, names);
  PyObject* copy = PyDict_Copy(a[0]);
  if (!copy) return NULL;
  PyObject* o = PyObject_CallNoArgs(st.options_type);
  if (o && PyObject_SetAttr(o, st.parallelize, copy) < 0) Py_CLEAR(o);
  Py_DECREF(copy);
  return o;
}

static PyMethodDef made[] = {
    {"threads", (PyCFunction)(void (*)(void))fast_threads, METH_FASTCALL | METH_KEYWORDS,
     "threads(n)\n--\n\nA LoopPar describing a parallel operation over `n` threads."},
    {"par", (PyCFunction)(void (*)(void))fast_par, METH_FASTCALL | METH_KEYWORDS,
     "par(p)\n--\n\nDefault options carrying the parallelisation mapping `p`."}};

// functions(LoopPar, its default threads per block, CompileOptions, threads, par) -> the two functions
static PyObject* functions(PyObject* self, PyObject* args) {
  (void)self;
  PyObject *par_type, *tpb, *options_type, *threads, *par;
  if (!PyArg_ParseTuple(args, "O!OO!OO", &PyType_Type, &par_type, &tpb, &PyType_Type, &options_type, &threads, &par)) return NULL;
  if (st.par_type) { PyErr_SetString(PyExc_RuntimeError, "functions: made already"); return NULL; }
  static const char* const names[3] = {"nthreads", "reduction", "_tpb"};
  Py_ssize_t fields[3];
  for (int f = 0; f < 3; ++f) {
    PyObject* slot = PyObject_GetAttrString(par_type, names[f]);
    if (!slot) return NULL;
    const int object = Py_TYPE(slot) == &PyMemberDescr_Type && ((PyMemberDescrObject*)slot)->d_member->type == T_OBJECT_EX;
    fields[f] = object ? ((PyMemberDescrObject*)slot)->d_member->offset : 0;
    Py_DECREF(slot);
    if (!object) { PyErr_SetString(PyExc_TypeError, "functions: the fields of the first type are not slots"); return NULL; }
  }
  PyObject* name = PyUnicode_InternFromString("parallelize");
  PyObject* modules[2] = {PyObject_GetAttrString(threads, "__module__"), PyObject_GetAttrString(par, "__module__")};
  PyObject* both[2] = {NULL, NULL};
  for (int q = 0; name && q < 2 && modules[q]; ++q) both[q] = PyCFunction_NewEx(&made[q], NULL, modules[q]);
  Py_XDECREF(modules[0]);
  Py_XDECREF(modules[1]);
  if (!name || !both[0] || !both[1]) {
    Py_XDECREF(name);
    Py_XDECREF(both[0]);
    Py_XDECREF(both[1]);
    return NULL;
  }
  PyObject* const kept[] = {par_type, tpb, options_type, threads, par};
  for (int q = 0; q < 5; ++q) Py_INCREF(kept[q]);
  st = (State){(PyTypeObject*)par_type, {fields[0], fields[1], fields[2]}, tpb, options_type, threads, par, name};
  return Py_BuildValue("(NN)", both[0], both[1]);
}

static PyMethodDef methods[] = {{"functions", functions, METH_VARARGS, "functions(LoopPar, tpb, CompileOptions, threads, par) -> (threads, par)"}, {NULL, NULL, 0, NULL}};
static PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_fastopts", "Options of a call, built without the interpreter.", -1, methods, NULL, NULL, NULL, NULL};

PyMODINIT_FUNC PyInit__fastopts(void) { return PyModule_Create(&module_def); }
