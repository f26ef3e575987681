// The short path of a warm call: a CPython extension that recognises a call seen before and runs its launch plan.
//
// What a call specialises on -- element types and shapes of device tensors, values of scalars, 16-byte alignment, the
// settings of the options object -- is written into a byte string, looked up, and the plan runs on the tensors' device
// pointers.  The Python statement of the same key (a tuple per argument, hashed) took 4.5 of the 7.2 us that a call
// with two tensors costs, the launch itself the rest; this file takes 0.4 us.  What it does not recognise (host arrays,
// sliced or gradient-tracking tensors, tensors without memory of their own, unusual option values) it leaves to the Python path, which decides everything
// and adds what it compiled.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <cstring>
#include <new>
#include <string>
#include <unordered_map>
#include <vector>

namespace {

using RunFn = int32_t (*)(void*, void* const*, int32_t);

struct Entry {
  void* plan;
  std::vector<int32_t> order;   // plan pointer k is the order[k]-th tensor of the call
};

struct Table {
  PyObject_HEAD
  std::unordered_map<std::string, Entry>* entries;
  std::string* key;             // built per call; calls hold the interpreter lock while they use it
  PyObject* opts_type;
  PyObject* loop_par_type;
  Py_ssize_t par_fields[3];     // where a LoopPar keeps nthreads, reduction and _tpb: slots, read without a look-up by name
  RunFn run;
};

constexpr size_t MAX_ENTRIES = 256;
constexpr size_t MAX_POINTERS = 64;

PyObject *s_opts, *s_parallelize, *s_nthreads, *s_reduction, *s_tpb, *s_member_names;

void put(std::string& k, const void* p, size_t n) { k.append((const char*)p, n); }
void put_tag(std::string& k, char c) { k.push_back(c); }
void put_i64(std::string& k, int64_t v) { put(k, &v, sizeof v); }
bool put_str(std::string& k, PyObject* s) {
  if (!PyUnicode_CheckExact(s)) return false;
  Py_ssize_t n = 0;
  const char* t = PyUnicode_AsUTF8AndSize(s, &n);
  if (!t) { PyErr_Clear(); return false; }
  put_i64(k, n);
  put(k, t, (size_t)n);
  return true;
}
bool put_long(std::string& k, PyObject* v) {
  int overflow = 0;
  long long x = PyLong_AsLongLongAndOverflow(v, &overflow);
  if (overflow || (x == -1 && PyErr_Occurred())) { PyErr_Clear(); return false; }
  put_i64(k, x);
  return true;
}

struct Pointers {
  void* p[MAX_POINTERS];
  size_t n = 0;
  bool aligned = true;
};

// one value of the call; false: not for this path
bool put_value(std::string& k, PyObject* v, Pointers& ps) {
  if (Py_TYPE(v) == (PyTypeObject*)THPVariableClass) {
    const at::Tensor& t = THPVariable_Unpack(v);
    if (t.is_neg() || t.is_conj()) return false;   // (what stands in memory is not the value)
    if (t.dim() == 0) {
      if (t.is_cuda() || t.layout() != c10::kStrided || !t.device().is_cpu()) return false;
      put_tag(k, 's');
      put_tag(k, (char)t.scalar_type());
      put(k, t.const_data_ptr(), t.element_size());
      return true;
    }
    if (!t.is_cuda() || t.layout() != c10::kStrided || !t.is_contiguous() || t.requires_grad()) return false;
    if (ps.n == MAX_POINTERS) return false;
    void* p = t.mutable_data_ptr();   // (a tensor that shares its memory until it is written gets its own, as `data_ptr()` does)
    ps.p[ps.n++] = p;
    ps.aligned = ps.aligned && (uintptr_t)p % 16 == 0;
    put_tag(k, 't');
    put_tag(k, (char)t.scalar_type());
    put_tag(k, (char)t.dim());
    for (int64_t d : t.sizes()) put_i64(k, d);
    return true;
  }
  if (PyBool_Check(v)) {
    put_tag(k, v == Py_True ? 'T' : 'F');
    return true;
  }
  if (PyLong_CheckExact(v)) {
    put_tag(k, 'i');
    return put_long(k, v);
  }
  if (PyFloat_CheckExact(v)) {
    double d = PyFloat_AS_DOUBLE(v);
    put_tag(k, 'f');
    put(k, &d, sizeof d);
    return true;
  }
  return false;
}

bool put_args(std::string& k, PyObject* args, Pointers& ps) {
  const Py_ssize_t n = PyTuple_GET_SIZE(args);
  for (Py_ssize_t a = 0; a < n; ++a) {
    PyObject* v = PyTuple_GET_ITEM(args, a);
    if (PyDict_CheckExact(v)) {
      put_tag(k, '{');
      put_i64(k, PyDict_GET_SIZE(v));
      PyObject *name, *field;
      Py_ssize_t pos = 0;
      while (PyDict_Next(v, &pos, &name, &field)) {
        if (!put_str(k, name) || PyDict_CheckExact(field) || !put_value(k, field, ps)) return false;
      }
    } else if (!put_value(k, v, ps)) {
      return false;
    }
  }
  return true;
}

// settings of an options object: the fields that its own dictionary holds (a field that is not there has its default)
bool put_options(std::string& k, PyObject* opts, PyObject* loop_par_type, const Py_ssize_t* par_fields) {
  PyObject* d = PyObject_GenericGetDict(opts, nullptr);   // new reference
  if (!d) { PyErr_Clear(); return false; }
  bool ok = PyDict_CheckExact(d);
  PyObject *name, *v;
  Py_ssize_t pos = 0;
  while (ok && PyDict_Next(d, &pos, &name, &v)) {
    if (PyList_CheckExact(v)) {
      ok = PyList_GET_SIZE(v) == 0;   // (include paths and the like: Python's business)
      continue;
    }
    ok = put_str(k, name);
    if (!ok) break;
    if (name == s_parallelize || PyUnicode_Compare(name, s_parallelize) == 0) {
      ok = PyDict_CheckExact(v);
      if (!ok) break;
      put_i64(k, PyDict_GET_SIZE(v));
      PyObject *label, *par;
      Py_ssize_t q = 0;
      while (ok && PyDict_Next(v, &q, &label, &par)) {
        ok = (PyObject*)Py_TYPE(par) == loop_par_type && put_str(k, label);
        for (int f = 0; ok && f < 3; ++f) {
          PyObject* x = *(PyObject**)((char*)par + par_fields[f]);   // (null: deleted)
          ok = x && PyLong_Check(x) && put_long(k, x);
        }
      }
    } else if (v == Py_None || PyBool_Check(v)) {
      put_tag(k, v == Py_None ? 'N' : v == Py_True ? 'T' : 'F');
    } else if (PyLong_CheckExact(v)) {
      put_tag(k, 'i');
      ok = put_long(k, v);
    } else if (!PyFloat_Check(v) && !PyUnicode_Check(v) && !PyDict_Check(v) && !PyTuple_Check(v) && PyObject_HasAttr(v, s_member_names)) {
      // members of an enumeration live as long as the module: their address is their identity
      put_tag(k, 'e');
      put(k, &v, sizeof v);
    } else {
      ok = false;
    }
  }
  Py_DECREF(d);
  return ok;
}

// What is asked of a tensor throws where it has no memory to point at (inside torch.vmap and the like the type is
// torch.Tensor all the same), and nothing may be thrown through the interpreter's frames: such a call is not for this
// path, the Python path asks again and reports it.
bool make_key(Table* self, PyObject* args, PyObject* opts, Pointers& ps) noexcept {
  try {
    std::string& k = *self->key;
    k.clear();
    if (!put_args(k, args, ps)) return false;
    put_tag(k, ps.aligned ? '|' : '!');
    return put_options(k, opts, self->loop_par_type, self->par_fields);
  } catch (...) {
    PyErr_Clear();   // (an exception that Python code under the tensor raised)
    return false;
  }
}

// run(args, kwargs) -> None: a call this table does not know; else the status of the run
PyObject* table_run(PyObject* o, PyObject* const* a, Py_ssize_t na) {
  Table* self = (Table*)o;
  if (na != 2 || !PyTuple_CheckExact(a[0]) || !PyDict_CheckExact(a[1])) { PyErr_SetString(PyExc_TypeError, "run(args, kwargs)"); return nullptr; }
  if (PyDict_GET_SIZE(a[1]) != 1) Py_RETURN_NONE;
  PyObject* opts = PyDict_GetItemWithError(a[1], s_opts);
  if (!opts || (PyObject*)Py_TYPE(opts) != self->opts_type) { PyErr_Clear(); Py_RETURN_NONE; }
  Pointers ps;
  if (!make_key(self, a[0], opts, ps)) Py_RETURN_NONE;
  auto it = self->entries->find(*self->key);
  if (it == self->entries->end()) Py_RETURN_NONE;
  const Entry& e = it->second;
  void* p[MAX_POINTERS];
  const size_t n = e.order.size();
  for (size_t q = 0; q < n; ++q) p[q] = ps.p[e.order[q]];
  void* plan = e.plan;
  RunFn run = self->run;
  int32_t rc;
  Py_BEGIN_ALLOW_THREADS
  rc = run(plan, p, (int32_t)n);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// add(args, opts, plan, order): remember the plan for this call; order[k] = which tensor of the call is plan pointer k
PyObject* table_add(PyObject* o, PyObject* const* a, Py_ssize_t na) {
  Table* self = (Table*)o;
  if (na != 4 || !PyTuple_CheckExact(a[0]) || !PyTuple_CheckExact(a[3])) { PyErr_SetString(PyExc_TypeError, "add(args, opts, plan, order)"); return nullptr; }
  if ((PyObject*)Py_TYPE(a[1]) != self->opts_type) Py_RETURN_FALSE;
  Pointers ps;
  if (!make_key(self, a[0], a[1], ps)) Py_RETURN_FALSE;
  void* plan = PyLong_AsVoidPtr(a[2]);
  if (PyErr_Occurred()) return nullptr;
  if ((size_t)PyTuple_GET_SIZE(a[3]) != ps.n) Py_RETURN_FALSE;
  int32_t order[MAX_POINTERS];
  for (size_t q = 0; q < ps.n; ++q) {
    long v = PyLong_AsLong(PyTuple_GET_ITEM(a[3], q));
    if (v < 0 || (size_t)v >= ps.n) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "order out of range");
      return nullptr;
    }
    order[q] = (int32_t)v;
  }
  try {
    if (self->entries->size() >= MAX_ENTRIES) self->entries->clear();
    Entry e{plan, {order, order + ps.n}};
    (*self->entries)[*self->key] = std::move(e);
  } catch (...) {
    return PyErr_NoMemory();
  }
  Py_RETURN_TRUE;
}

PyObject* table_clear(PyObject* o, PyObject*) {
  ((Table*)o)->entries->clear();
  Py_RETURN_NONE;
}

PyObject* table_new(PyTypeObject* type, PyObject* args, PyObject*) {
  PyObject *opts_type, *loop_par_type, *run;
  if (!PyArg_ParseTuple(args, "OOO", &opts_type, &loop_par_type, &run)) return nullptr;
  void* fn = PyLong_AsVoidPtr(run);
  if (PyErr_Occurred()) return nullptr;
  Py_ssize_t fields[3];
  PyObject* const names[3] = {s_nthreads, s_reduction, s_tpb};
  for (int f = 0; f < 3; ++f) {
    PyObject* slot = PyObject_GetAttr(loop_par_type, names[f]);
    if (!slot) return nullptr;
    const bool object = Py_TYPE(slot) == &PyMemberDescr_Type && ((PyMemberDescrObject*)slot)->d_member->type == T_OBJECT_EX;
    fields[f] = object ? ((PyMemberDescrObject*)slot)->d_member->offset : 0;
    Py_DECREF(slot);
    if (!object) { PyErr_SetString(PyExc_TypeError, "CallTable: the fields of the second type are not slots"); return nullptr; }
  }
  Table* self = (Table*)type->tp_alloc(type, 0);
  if (!self) return nullptr;
  std::copy(fields, fields + 3, self->par_fields);
  self->entries = new (std::nothrow) std::unordered_map<std::string, Entry>();
  self->key = new (std::nothrow) std::string();
  if (!self->entries || !self->key) { Py_DECREF(self); return PyErr_NoMemory(); }
  Py_INCREF(opts_type);
  Py_INCREF(loop_par_type);
  self->opts_type = opts_type;
  self->loop_par_type = loop_par_type;
  self->run = (RunFn)fn;
  return (PyObject*)self;
}

void table_dealloc(PyObject* o) {
  Table* self = (Table*)o;
  delete self->entries;
  delete self->key;
  Py_XDECREF(self->opts_type);
  Py_XDECREF(self->loop_par_type);
  Py_TYPE(o)->tp_free(o);
}

PyMethodDef table_methods[] = {
    {"run", (PyCFunction)(void (*)(void))table_run, METH_FASTCALL, "run(args, kwargs): status of the run, None for a call that is not known"},
    {"add", (PyCFunction)(void (*)(void))table_add, METH_FASTCALL, "add(args, opts, plan, order): remember a compiled call"},
    {"clear", table_clear, METH_NOARGS, "forget all calls"},
    {nullptr, nullptr, 0, nullptr}};

PyTypeObject table_type = {PyVarObject_HEAD_INIT(nullptr, 0)};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_fastcall", "Warm calls of jitted functions.", -1, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fastcall(void) {
  table_type.tp_name = "parpy_amd._fastcall.CallTable";
  table_type.tp_basicsize = sizeof(Table);
  table_type.tp_flags = Py_TPFLAGS_DEFAULT;
  table_type.tp_new = table_new;
  table_type.tp_dealloc = table_dealloc;
  table_type.tp_methods = table_methods;
  if (PyType_Ready(&table_type) < 0) return nullptr;
  s_opts = PyUnicode_InternFromString("opts");
  s_parallelize = PyUnicode_InternFromString("parallelize");
  s_nthreads = PyUnicode_InternFromString("nthreads");
  s_reduction = PyUnicode_InternFromString("reduction");
  s_tpb = PyUnicode_InternFromString("_tpb");
  s_member_names = PyUnicode_InternFromString("_member_names_");
  PyObject* m = PyModule_Create(&module_def);
  if (!m) return nullptr;
  Py_INCREF(&table_type);
  if (PyModule_AddObject(m, "CallTable", (PyObject*)&table_type) < 0) {
    Py_DECREF(&table_type);
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
