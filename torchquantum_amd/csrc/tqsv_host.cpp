// The host path between two launches, as a CPython extension: recording gates
// on a device's tape and turning a tape into its plan's key and its parameter
// pointers.  A circuit of 820 gates passes here on every call of a model, so
// what costs microseconds per gate in Python (attribute look-ups on modules
// and tensors, one tuple per gate) is done on the objects directly.
//
// The tape is a Python list of engine.TapeOp instances (a dataclass with
// slots); their slots are read and written at the offsets of its member
// descriptors.  Every function here does what the Python code it stands in
// for does, and where an argument is not of the plain kind it returns "not
// handled" and that Python code runs.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <structmember.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <string>
#include <vector>

namespace {

enum Slot { S_NAME, S_WIRES, S_PARAMS, S_INVERSE, S_VERSION, S_CONJ, S_NONUNITARY, N_SLOTS };
const char* const kSlotNames[N_SLOTS] = {"name", "wires", "params", "inverse", "version", "conj", "nonunitary"};

PyTypeObject* g_op_type = nullptr;       // engine.TapeOp
Py_ssize_t g_off[N_SLOTS];

PyObject *g_s_params, *g_s_parameters, *g_s_wires, *g_s_inverse, *g_s_hooks[4], *g_s_forward, *g_s_func, *g_s_compiled;
PyObject* g_zero;

PyObject*& slot(PyObject* op, Slot s) { return *reinterpret_cast<PyObject**>(reinterpret_cast<char*>(op) + g_off[s]); }

// a C++ exception (torch) as a Python one
template <class F>
PyObject* guarded(F f) {
  try {
    return f();
  } catch (const c10::Error& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
  }
  return nullptr;
}

// bind(TapeOp): the class whose instances the other functions make and read
PyObject* h_bind(PyObject*, PyObject* cls) {
  if (!PyType_Check(cls)) {
    PyErr_SetString(PyExc_TypeError, "bind: a class is needed");
    return nullptr;
  }
  Py_ssize_t off[N_SLOTS];
  for (int i = 0; i < N_SLOTS; ++i) {
    PyObject* d = PyDict_GetItemString(reinterpret_cast<PyTypeObject*>(cls)->tp_dict, kSlotNames[i]);
    if (!d || !Py_IS_TYPE(d, &PyMemberDescr_Type)) {
      PyErr_Format(PyExc_TypeError, "bind: %s is not a slot of the class", kSlotNames[i]);
      return nullptr;
    }
    off[i] = reinterpret_cast<PyMemberDescrObject*>(d)->d_member->offset;
  }
  std::memcpy(g_off, off, sizeof off);
  Py_INCREF(cls);
  Py_XDECREF(reinterpret_cast<PyObject*>(g_op_type));
  g_op_type = reinterpret_cast<PyTypeObject*>(cls);
  Py_RETURN_NONE;
}

bool bound() {
  if (g_op_type) return true;
  PyErr_SetString(PyExc_RuntimeError, "bind() has not been called");
  return false;
}

// a TapeOp; steals `wires`
PyObject* new_op(PyObject* name, PyObject* wires, PyObject* params, bool inverse, PyObject* version) {
  PyObject* op = g_op_type->tp_alloc(g_op_type, 0);
  if (!op) {
    Py_DECREF(wires);
    return nullptr;
  }
  PyObject* inv = inverse ? Py_True : Py_False;
  Py_INCREF(name);
  Py_INCREF(params);
  Py_INCREF(inv);
  Py_INCREF(version);
  Py_INCREF(Py_False);
  Py_INCREF(Py_False);
  slot(op, S_NAME) = name;
  slot(op, S_WIRES) = wires;
  slot(op, S_PARAMS) = params;
  slot(op, S_INVERSE) = inv;
  slot(op, S_VERSION) = version;
  slot(op, S_CONJ) = Py_False;
  slot(op, S_NONUNITARY) = Py_False;
  return op;
}

// The plain form of a gate's arguments: int wires in range and all different,
// as many as the gate has, and no parameter or a real [rows, npar] tensor.
// 1: *out is the new TapeOp, 0: not the plain form, -1: a Python error.
int plain_op(PyObject* name, long nw, long npar, PyObject* wires, PyObject* params, bool inverse, long n,
             PyObject** out) {
  long w[8];
  long k = 0;
  if (nw > 8) return 0;
  if (PyLong_CheckExact(wires)) {
    w[k++] = PyLong_AsLong(wires);
  } else if (PyList_CheckExact(wires) || PyTuple_CheckExact(wires)) {
    const Py_ssize_t len = PySequence_Fast_GET_SIZE(wires);
    if (len != nw) return 0;
    PyObject** items = PySequence_Fast_ITEMS(wires);
    for (Py_ssize_t i = 0; i < len; ++i) {
      if (!PyLong_CheckExact(items[i])) return 0;
      w[k++] = PyLong_AsLong(items[i]);
    }
  } else {
    return 0;
  }
  if (PyErr_Occurred()) {
    PyErr_Clear();
    return 0;
  }
  if (k != nw) return 0;
  for (long i = 0; i < k; ++i) {
    if (w[i] < 0 || w[i] >= n) return 0;
    for (long j = 0; j < i; ++j)
      if (w[j] == w[i]) return 0;
  }
  PyObject* version = g_zero;
  PyObject* made = nullptr;
  if (npar > 0) {
    if (!THPVariable_Check(params)) return 0;
    const at::Tensor& t = THPVariable_Unpack(params);
    if (t.dim() != 2 || t.size(1) != npar || t.is_complex()) return 0;
    made = version = PyLong_FromLongLong((long long)t._version());
    if (!version) return -1;
  } else {
    params = Py_None;
  }
  PyObject* tup = PyTuple_New(k);
  if (!tup) {
    Py_XDECREF(made);
    return -1;
  }
  for (long i = 0; i < k; ++i) PyTuple_SET_ITEM(tup, i, PyLong_FromLong(w[i]));
  *out = new_op(name, tup, params, inverse, version);
  Py_XDECREF(made);
  return *out ? 1 : -1;
}

// make(name, num_wires, num_params, wires, params, inverse, n_wires): the
// TapeOp of a gate called with arguments of the plain form, else None
PyObject* h_make(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 7 || !bound()) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "make: 7 arguments");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    const long nw = PyLong_AsLong(a[1]), npar = PyLong_AsLong(a[2]), n = PyLong_AsLong(a[6]);
    const int inv = PyObject_IsTrue(a[5]);
    if (PyErr_Occurred() || inv < 0) return nullptr;
    PyObject* op = nullptr;
    const int r = plain_op(a[0], nw, npar, a[3], a[4], inv != 0, n, &op);
    if (r < 0) return nullptr;
    if (r == 0) Py_RETURN_NONE;
    return op;
  });
}

bool empty_or_missing(PyObject* dict, PyObject* key) {
  PyObject* v = PyDict_GetItemWithError(dict, key);
  if (!v) return !PyErr_Occurred();
  if (v == Py_None) return true;
  return PyDict_Check(v) && PyDict_GET_SIZE(v) == 0;
}

// operator_op(op, spec, wires, n_wires): the TapeOp that op(q_device,
// wires=wires) would record, op an Operator module whose class has the plain
// forward, spec = (gate name, num_wires, num_params).  Sets op.wires as that
// call does.  None where a hook, a compiled or replaced forward or an
// argument that is not plain makes the call itself necessary.
PyObject* h_operator_op(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 4 || !bound()) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "operator_op: 4 arguments");
    return nullptr;
  }
  return guarded([&]() -> PyObject* {
    PyObject** dp = _PyObject_GetDictPtr(a[0]);
    if (!dp || !*dp || !PyTuple_CheckExact(a[1]) || PyTuple_GET_SIZE(a[1]) != 3) Py_RETURN_NONE;
    PyObject* d = *dp;
    for (PyObject* h : g_s_hooks)
      if (!empty_or_missing(d, h)) Py_RETURN_NONE;
    if (PyDict_GetItemWithError(d, g_s_forward) || PyDict_GetItemWithError(d, g_s_func)) Py_RETURN_NONE;
    if (!empty_or_missing(d, g_s_compiled)) Py_RETURN_NONE;
    PyObject* pd = PyDict_GetItemWithError(d, g_s_parameters);
    PyObject* p = pd && PyDict_Check(pd) ? PyDict_GetItemWithError(pd, g_s_params) : nullptr;
    PyObject* own = PyDict_GetItemWithError(d, g_s_params);
    if (own) p = own;                     // a plain attribute hides a parameter
    PyObject* inv = PyDict_GetItemWithError(d, g_s_inverse);
    if (PyErr_Occurred()) return nullptr;
    if (!p || !inv || !PyBool_Check(inv)) Py_RETURN_NONE;
    const long nw = PyLong_AsLong(PyTuple_GET_ITEM(a[1], 1)), npar = PyLong_AsLong(PyTuple_GET_ITEM(a[1], 2));
    const long n = PyLong_AsLong(a[3]);
    if (PyErr_Occurred()) return nullptr;
    PyObject* op = nullptr;
    const int r = plain_op(PyTuple_GET_ITEM(a[1], 0), nw, npar, a[2], p, inv == Py_True, n, &op);
    if (r < 0) return nullptr;
    if (r == 0) Py_RETURN_NONE;
    PyObject* w = PyLong_CheckExact(a[2]) ? PyList_New(1) : nullptr;
    if (w) {
      Py_INCREF(a[2]);
      PyList_SET_ITEM(w, 0, a[2]);
    } else if (PyErr_Occurred()) {
      Py_DECREF(op);
      return nullptr;
    } else {
      w = a[2];
      Py_INCREF(w);
    }
    const int e = PyDict_SetItem(d, g_s_wires, w);
    Py_DECREF(w);
    if (e) {
      Py_DECREF(op);
      return nullptr;
    }
    return op;
  });
}

bool tape_ok(PyObject* tape) {
  if (!bound()) return false;
  if (!PyList_CheckExact(tape)) {
    PyErr_SetString(PyExc_TypeError, "a tape is a list of TapeOp");
    return false;
  }
  const Py_ssize_t n = PyList_GET_SIZE(tape);
  for (Py_ssize_t i = 0; i < n; ++i) {
    if (!Py_IS_TYPE(PyList_GET_ITEM(tape, i), g_op_type)) {
      PyErr_SetString(PyExc_TypeError, "a tape is a list of TapeOp");
      return false;
    }
  }
  return true;
}

// stale(tape): index of the first op whose parameter tensor was modified in
// place since it was recorded, or -1
PyObject* h_stale(PyObject*, PyObject* tape) {
  if (!tape_ok(tape)) return nullptr;
  return guarded([&]() -> PyObject* {
    const Py_ssize_t n = PyList_GET_SIZE(tape);
    for (Py_ssize_t i = 0; i < n; ++i) {
      PyObject* op = PyList_GET_ITEM(tape, i);
      PyObject* p = slot(op, S_PARAMS);
      if (p == Py_None || !THPVariable_Check(p)) continue;
      const long long v = PyLong_AsLongLong(slot(op, S_VERSION));
      if (v == -1 && PyErr_Occurred()) return nullptr;
      if ((long long)THPVariable_Unpack(p)._version() != v) return PyLong_FromSsize_t(i);
    }
    return PyLong_FromLong(-1);
  });
}

void put(std::string& s, int64_t v) { s.append(reinterpret_cast<const char*>(&v), sizeof v); }

// structure(tape): the circuit's structure as bytes -- every op's gate, wires,
// flags and, of its parameter, the shape, type, place and whether it wants a
// gradient.  Two tapes have equal bytes exactly if a plan fits both.
PyObject* h_structure(PyObject*, PyObject* tape) {
  if (!tape_ok(tape)) return nullptr;
  return guarded([&]() -> PyObject* {
    const Py_ssize_t n = PyList_GET_SIZE(tape);
    std::string s;
    s.reserve((size_t)n * 72);
    for (Py_ssize_t i = 0; i < n; ++i) {
      PyObject* op = PyList_GET_ITEM(tape, i);
      Py_ssize_t len = 0;
      const char* name = PyUnicode_AsUTF8AndSize(slot(op, S_NAME), &len);
      if (!name) return nullptr;
      put(s, (int64_t)len);
      s.append(name, (size_t)len);
      PyObject* w = slot(op, S_WIRES);
      if (!PyTuple_CheckExact(w)) {
        PyErr_SetString(PyExc_TypeError, "TapeOp.wires is a tuple");
        return nullptr;
      }
      const Py_ssize_t k = PyTuple_GET_SIZE(w);
      put(s, (int64_t)k);
      for (Py_ssize_t q = 0; q < k; ++q) {
        const long long v = PyLong_AsLongLong(PyTuple_GET_ITEM(w, q));
        if (v == -1 && PyErr_Occurred()) return nullptr;
        put(s, v);
      }
      const int inv = PyObject_IsTrue(slot(op, S_INVERSE)), cj = PyObject_IsTrue(slot(op, S_CONJ));
      if (inv < 0 || cj < 0) return nullptr;
      PyObject* p = slot(op, S_PARAMS);
      if (p == Py_None) {
        put(s, inv | cj << 1);
        continue;
      }
      if (!THPVariable_Check(p)) {
        PyErr_SetString(PyExc_TypeError, "TapeOp.params is a tensor or None");
        return nullptr;
      }
      const at::Tensor& t = THPVariable_Unpack(p);
      const bool cplx = t.is_complex();
      // a matrix: its shape only, as its values are fetched to the host
      const int64_t meta = cplx ? 0 : (int64_t)t.requires_grad() << 4 | (int64_t)t.is_cuda() << 5 |
                                          (int64_t)t.scalar_type() << 8;
      put(s, inv | cj << 1 | 4 | (int64_t)cplx << 3 | meta);
      put(s, t.dim());
      for (int64_t q = 0; q < t.dim(); ++q) put(s, t.size(q));
    }
    return PyBytes_FromStringAndSize(s.data(), (Py_ssize_t)s.size());
  });
}

// pointers(tape, index, out): out[j] = (data pointer, row stride or 0 for one
// row, column stride) of tape[index[j]].params; index int32, out int64 [len, 3]
PyObject* h_pointers(PyObject*, PyObject* const* a, Py_ssize_t na) {
  if (na != 3) {
    PyErr_SetString(PyExc_TypeError, "pointers: 3 arguments");
    return nullptr;
  }
  if (!tape_ok(a[0])) return nullptr;
  Py_buffer idx, out;
  if (PyObject_GetBuffer(a[1], &idx, PyBUF_CONTIG_RO)) return nullptr;
  if (PyObject_GetBuffer(a[2], &out, PyBUF_CONTIG)) {
    PyBuffer_Release(&idx);
    return nullptr;
  }
  PyObject* r = guarded([&]() -> PyObject* {
    const Py_ssize_t n = idx.len / 4, len = PyList_GET_SIZE(a[0]);
    if (idx.itemsize != 4 || out.itemsize != 8 || out.len < n * 24) {
      PyErr_SetString(PyExc_ValueError, "pointers: index int32, out int64 [len, 3]");
      return nullptr;
    }
    const int32_t* ix = static_cast<const int32_t*>(idx.buf);
    int64_t* o = static_cast<int64_t*>(out.buf);
    for (Py_ssize_t j = 0; j < n; ++j) {
      PyObject* p = ix[j] >= 0 && ix[j] < len ? slot(PyList_GET_ITEM(a[0], ix[j]), S_PARAMS) : Py_None;
      if (!THPVariable_Check(p)) {
        PyErr_SetString(PyExc_ValueError, "pointers: an op without a parameter tensor");
        return nullptr;
      }
      const at::Tensor& t = THPVariable_Unpack(p);
      if (t.dim() != 2) {
        PyErr_SetString(PyExc_ValueError, "pointers: parameters are [rows, P]");
        return nullptr;
      }
      o[3 * j] = reinterpret_cast<int64_t>(t.data_ptr());
      o[3 * j + 1] = t.size(0) > 1 ? t.stride(0) : 0;
      o[3 * j + 2] = t.stride(1);
    }
    Py_RETURN_NONE;
  });
  PyBuffer_Release(&idx);
  PyBuffer_Release(&out);
  return r;
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyCFunction fast() { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F)); }

PyMethodDef kMethods[] = {
    {"bind", h_bind, METH_O, "bind(TapeOp)"},
    {"make", fast<h_make>(), METH_FASTCALL, "make(name, num_wires, num_params, wires, params, inverse, n_wires)"},
    {"operator_op", fast<h_operator_op>(), METH_FASTCALL, "operator_op(op, spec, wires, n_wires)"},
    {"stale", h_stale, METH_O, "stale(tape)"},
    {"structure", h_structure, METH_O, "structure(tape)"},
    {"pointers", fast<h_pointers>(), METH_FASTCALL, "pointers(tape, index, out)"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_tqhost", "Tape recording and plan keys.", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__tqhost(void) {
  g_s_params = PyUnicode_InternFromString("params");
  g_s_parameters = PyUnicode_InternFromString("_parameters");
  g_s_wires = PyUnicode_InternFromString("wires");
  g_s_inverse = PyUnicode_InternFromString("inverse");
  g_s_forward = PyUnicode_InternFromString("forward");
  g_s_func = PyUnicode_InternFromString("func");
  g_s_compiled = PyUnicode_InternFromString("_compiled_call_impl");
  const char* hooks[4] = {"_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks"};
  for (int i = 0; i < 4; ++i) g_s_hooks[i] = PyUnicode_InternFromString(hooks[i]);
  g_zero = PyLong_FromLong(0);
  if (PyErr_Occurred()) return nullptr;
  return PyModule_Create(&kModule);
}
