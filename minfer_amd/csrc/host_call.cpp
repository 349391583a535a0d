// The host side of a launch, for `kernels/ops.py`: checking an operand and calling a library's entry point.  (Both are a few
// hundred nanoseconds of work; through ctypes and torch's Python attributes they were 13 us a launch, which is more than most
// kernels of a short prompt take: the 0.5B prompt of 37 tokens, 150 launches, spent 1.9 ms of 2.5 on them.)
//
//   need(t, name, dtype=None, shape=None)   nothing where `t` is a contiguous tensor on the GPU of that type (one, or a tuple of
//                                           them) and shape; anything else goes to the function given to `otherwise`, which
//                                           names what is wrong
//   Launch(address, kinds)(...)             calls the C function at `address`; kinds, a letter an argument: p pointer (a tensor:
//                                           its data; None; a number; a ctypes array: its place; a ctypes pointer: its value),
//                                           i int, q 64 bits, f float, d double.  Returns its int.  The call runs without the
//                                           interpreter's lock.
//   Record()                                the launches that a thread makes between `with record:` and its end (those of Launches
//                                           whose `recorded` is set and that returned 0), to be made again with other tensors
//                                           in some places: `bind(olds)`, then `run(news)` for each set.  It holds the objects
//                                           that the launches were given, so their memory stays theirs.  A pointer is replaced
//                                           where it is a tensor's first address; a launch that was given a number as a pointer
//                                           (other than its last, the stream) may have an address inside one, and does not bind.
#include <Python.h>
#include <stdint.h>
#include <string.h>

#include <exception>
#include <new>
#include <vector>

#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#if !defined(__x86_64__) || !defined(__linux__)
#error "the call below is written for the System V convention of x86-64"
#endif

namespace {

constexpr int MAX_INT = 44, MAX_FP = 8;

struct Call {
  void* fn;
  uint64_t w[MAX_INT];
  double f[MAX_FP];
  uint64_t pointers;                                 // bit i: w[i] is one
  bool numbers;                                      // one of them, not the last argument, came as a number
};
struct Place { int call, word, tensor; };
struct Recorded {
  std::vector<Call> calls;
  std::vector<PyObject*> held;
  std::vector<Place> places;
  std::vector<at::Tensor> olds;
};
thread_local Recorded* t_recording = nullptr;

struct Launch {
  PyObject_HEAD
  vectorcallfunc call;
  void* fn;
  int n;
  char recorded;
  char kinds[MAX_INT + MAX_FP + 1];
};

// Whole numbers and pointers go into registers and onto the stack in their order, floating ones into registers of their own in
// theirs (all of them: at most eight), so one call with room for the most of each serves every signature: a function takes its
// own and does not see the rest.  A float lies in the low half of its register.
#define MF_I4(x) w[x], w[x + 1], w[x + 2], w[x + 3]
int call_any(void* fn, const uint64_t* w, const double* f) {
  using U = uint64_t;
  using Fn = int (*)(U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U, U,
                     U, U, U, U, double, double, double, double, double, double, double, double);
  return reinterpret_cast<Fn>(fn)(MF_I4(0), MF_I4(4), MF_I4(8), MF_I4(12), MF_I4(16), MF_I4(20), MF_I4(24), MF_I4(28), MF_I4(32), MF_I4(36),
                                  MF_I4(40), f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7]);
}

PyObject* wrong_kind(const char* what, Py_ssize_t at, PyObject* got) {
  PyErr_Format(PyExc_TypeError, "argument %zd: %s expected instead of %s", at + 1, what, Py_TYPE(got)->tp_name);
  return nullptr;
}

PyObject *g_array = nullptr, *g_pointer = nullptr;   // ctypes.Array and ctypes.c_void_p

// The address that a ctypes array lies at or a ctypes pointer holds; false (and no error): it is neither.  Nothing else with a
// buffer is taken: the array of a numerical library is host memory, which no kernel may be given by mistake.  The caller holds
// the object, and with it the memory.
bool ctypes_address(PyObject* a, uint64_t& address) {
  const int array = PyObject_IsInstance(a, g_array), pointer = array == 0 ? PyObject_IsInstance(a, g_pointer) : 0;
  Py_buffer b;
  if ((array <= 0 && pointer <= 0) || PyObject_GetBuffer(a, &b, PyBUF_SIMPLE) != 0) {
    PyErr_Clear();
    return false;
  }
  if (array > 0) address = reinterpret_cast<uint64_t>(b.buf);
  else memcpy(&address, b.buf, sizeof address);
  PyBuffer_Release(&b);
  return true;
}

// a whole number, or what says which one it is (`__index__`); false: neither, with the error set
bool whole(PyObject* a, Py_ssize_t at, uint64_t& v) {
  PyObject* n = PyNumber_Index(a);
  if (!n) {
    PyErr_Clear();
    wrong_kind("int", at, a);
    return false;
  }
  v = PyLong_AsUnsignedLongLongMask(n);
  Py_DECREF(n);
  return true;
}

PyObject* launch_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  Launch* l = reinterpret_cast<Launch*>(self);
  const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
  if (n != l->n || (kwnames && PyTuple_GET_SIZE(kwnames))) {
    PyErr_Format(PyExc_TypeError, "%d arguments expected, %zd given", l->n, n);
    return nullptr;
  }
  uint64_t w[MAX_INT] = {};
  double f[MAX_FP] = {};
  uint64_t pointers = 0;
  bool numbers = false;
  int nw = 0, nf = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* a = args[i];
    if (l->kinds[i] == 'p') pointers |= uint64_t(1) << nw;
    switch (l->kinds[i]) {
      case 'p':
        if (a == Py_None) {
          w[nw++] = 0;
        } else if (THPVariable_Check(a)) {
          try {
            w[nw++] = reinterpret_cast<uint64_t>(THPVariable_Unpack(a).data_ptr());
          } catch (const std::exception& e) {
            PyErr_SetString(PyExc_RuntimeError, e.what());
            return nullptr;
          }
        } else if (PyLong_Check(a)) {
          w[nw] = PyLong_AsUnsignedLongLongMask(a);
          numbers |= w[nw++] != 0 && i + 1 < n;
        } else if (ctypes_address(a, w[nw])) {
          ++nw;
        } else {
          return wrong_kind("a tensor, a number, None or a ctypes array or pointer", i, a);
        }
        break;
      case 'i':
        if (!whole(a, i, w[nw])) return nullptr;
        w[nw] = static_cast<uint32_t>(w[nw]);
        ++nw;
        break;
      case 'q':
        if (!whole(a, i, w[nw++])) return nullptr;
        break;
      default: {
        const double v = PyFloat_AsDouble(a);
        if (v == -1.0 && PyErr_Occurred()) return nullptr;
        if (l->kinds[i] == 'd') {
          f[nf++] = v;
        } else {
          const float s = static_cast<float>(v);
          memcpy(&f[nf++], &s, sizeof s);
        }
      }
    }
    if (PyErr_Occurred()) return nullptr;
  }
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = call_any(l->fn, w, f);
  Py_END_ALLOW_THREADS
  if (t_recording && l->recorded && rc == 0) {
    try {
      Call c;
      c.fn = l->fn;
      memcpy(c.w, w, sizeof w);
      memcpy(c.f, f, sizeof f);
      c.pointers = pointers;
      c.numbers = numbers;
      for (Py_ssize_t i = 0; i < n; ++i)
        if (l->kinds[i] == 'p') {
          t_recording->held.push_back(args[i]);
          Py_INCREF(args[i]);
        }
      t_recording->calls.push_back(c);
    } catch (const std::exception& e) {
      PyErr_SetString(PyExc_RuntimeError, e.what());
      return nullptr;
    }
  }
  return PyLong_FromLong(rc);
}

PyObject* launch_new(PyTypeObject* type, PyObject* args, PyObject*) {
  unsigned long long address;
  const char* kinds;
  int recorded = 0;
  if (!PyArg_ParseTuple(args, "Ks|p", &address, &kinds, &recorded)) return nullptr;
  int nw = 0, nf = 0;
  for (const char* k = kinds; *k; ++k) {
    if (*k == 'f' || *k == 'd') ++nf;
    else if (*k == 'p' || *k == 'i' || *k == 'q') ++nw;
    else nw = MAX_INT + 1;
  }
  if (!address || nw > MAX_INT || nf > MAX_FP) {
    PyErr_Format(PyExc_ValueError, "Launch: arguments \"%s\" (at most %d and %d floating ones)", kinds, MAX_INT, MAX_FP);
    return nullptr;
  }
  Launch* l = reinterpret_cast<Launch*>(type->tp_alloc(type, 0));
  if (!l) return nullptr;
  l->call = launch_call;
  l->fn = reinterpret_cast<void*>(static_cast<uintptr_t>(address));
  l->n = nw + nf;
  l->recorded = recorded != 0;
  strcpy(l->kinds, kinds);
  return reinterpret_cast<PyObject*>(l);
}

PyTypeObject LaunchType = {PyVarObject_HEAD_INIT(nullptr, 0)};

struct Record {
  PyObject_HEAD
  Recorded* r;
};

PyObject* record_new(PyTypeObject* type, PyObject*, PyObject*) {
  Record* self = reinterpret_cast<Record*>(type->tp_alloc(type, 0));
  if (!self) return nullptr;
  self->r = new (std::nothrow) Recorded;
  if (!self->r) {
    Py_DECREF(self);
    return PyErr_NoMemory();
  }
  return reinterpret_cast<PyObject*>(self);
}

void record_free(PyObject* o) {
  Record* self = reinterpret_cast<Record*>(o);
  if (self->r) {
    if (t_recording == self->r) t_recording = nullptr;
    for (PyObject* h : self->r->held) Py_DECREF(h);
    delete self->r;
  }
  Py_TYPE(o)->tp_free(o);
}

PyObject* record_enter(PyObject* self, PyObject*) {
  if (t_recording) {
    PyErr_SetString(PyExc_RuntimeError, "Record: this thread is recording already");
    return nullptr;
  }
  t_recording = reinterpret_cast<Record*>(self)->r;
  Py_INCREF(self);
  return self;
}

PyObject* record_exit(PyObject*, PyObject*) {
  t_recording = nullptr;
  Py_RETURN_NONE;
}

// the tensor of a place, or nothing where it is None
bool place_tensor(PyObject* o, at::Tensor& t) {
  if (o == Py_None) return true;
  if (!THPVariable_Check(o)) return false;
  t = THPVariable_Unpack(o);
  return t.is_contiguous();
}

// bind(olds): the places at which these tensors (None: no such tensor) begin.  False where two of them begin at the same address,
// or where a launch was given a pointer as a number.
PyObject* record_bind(PyObject* self, PyObject* olds) {
  Recorded& r = *reinterpret_cast<Record*>(self)->r;
  if (!PyTuple_Check(olds)) {
    PyErr_SetString(PyExc_TypeError, "bind: a tuple of tensors");
    return nullptr;
  }
  try {
    r.places.clear();
    r.olds.clear();
    for (const Call& c : r.calls)
      if (c.numbers) Py_RETURN_FALSE;
    for (Py_ssize_t j = 0; j < PyTuple_GET_SIZE(olds); ++j) {
      at::Tensor t;
      if (!place_tensor(PyTuple_GET_ITEM(olds, j), t)) Py_RETURN_FALSE;
      for (const at::Tensor& u : r.olds)
        if (t.defined() && u.defined() && t.data_ptr() == u.data_ptr()) Py_RETURN_FALSE;
      r.olds.push_back(t);
      if (!t.defined()) continue;
      const uint64_t at = reinterpret_cast<uint64_t>(t.data_ptr());
      for (size_t c = 0; c < r.calls.size(); ++c)
        for (int w = 0; w < MAX_INT; ++w)
          if ((r.calls[c].pointers >> w & 1) && r.calls[c].w[w] == at) r.places.push_back(Place{(int)c, w, (int)j});
    }
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
  Py_RETURN_TRUE;
}

// run(news): the launches with these tensors in the places of the bound ones.  None, nothing launched, where one is not like
// the one whose place it takes (type, shape, device, alignment); else the first code that is not 0, or 0.
PyObject* record_run(PyObject* self, PyObject* news) {
  Recorded& r = *reinterpret_cast<Record*>(self)->r;
  if (!PyTuple_Check(news) || (size_t)PyTuple_GET_SIZE(news) != r.olds.size()) {
    PyErr_SetString(PyExc_TypeError, "run: as many tensors as were bound");
    return nullptr;
  }
  int rc = 0;
  try {
    std::vector<uint64_t> at(r.olds.size(), 0);
    for (size_t j = 0; j < at.size(); ++j) {
      at::Tensor t;
      const at::Tensor& u = r.olds[j];
      if (!place_tensor(PyTuple_GET_ITEM(news, j), t) || t.defined() != u.defined()) Py_RETURN_NONE;
      if (!t.defined()) continue;
      at[j] = reinterpret_cast<uint64_t>(t.data_ptr());
      if (t.scalar_type() != u.scalar_type() || t.sizes() != u.sizes() || t.device() != u.device() ||
          (at[j] ^ reinterpret_cast<uint64_t>(u.data_ptr())) % 16)
        Py_RETURN_NONE;
    }
    std::vector<Call> calls = r.calls;
    for (const Place& p : r.places) calls[p.call].w[p.word] = at[p.tensor];
    Py_BEGIN_ALLOW_THREADS
    for (size_t c = 0; c < calls.size() && rc == 0; ++c) rc = call_any(calls[c].fn, calls[c].w, calls[c].f);
    Py_END_ALLOW_THREADS
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
  return PyLong_FromLong(rc);
}

PyMethodDef record_methods[] = {{"__enter__", record_enter, METH_NOARGS, "this thread's launches are recorded from here"},
                                {"__exit__", record_exit, METH_VARARGS, "... to here"},
                                {"bind", record_bind, METH_O, "the tensors that others are to take the place of"},
                                {"run", record_run, METH_O, "the launches with other tensors"},
                                {nullptr, nullptr, 0, nullptr}};
PyTypeObject RecordType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* g_otherwise = nullptr;

bool same_type(PyObject* dtype, at::ScalarType type) { return THPDtype_Check(dtype) && reinterpret_cast<THPDtype*>(dtype)->scalar_type == type; }

bool is_right(PyObject* t, PyObject* dtype, PyObject* shape) {
  if (!THPVariable_Check(t)) return false;
  const at::Tensor& x = THPVariable_Unpack(t);
  if (!x.is_cuda() || !x.is_contiguous()) return false;
  if (dtype != Py_None) {
    bool found = false;
    if (PyTuple_CheckExact(dtype))
      for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(dtype) && !found; ++i) found = same_type(PyTuple_GET_ITEM(dtype, i), x.scalar_type());
    else
      found = same_type(dtype, x.scalar_type());
    if (!found) return false;
  }
  if (shape != Py_None) {
    if (!PyTuple_Check(shape) || PyTuple_GET_SIZE(shape) != x.dim()) return false;
    for (Py_ssize_t i = 0; i < x.dim(); ++i) {
      PyObject* s = PyTuple_GET_ITEM(shape, i);
      if (!PyLong_Check(s) || PyLong_AsLongLong(s) != x.size(i)) return false;
    }
  }
  return true;
}

PyObject* need(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n < 2 || n > 4) {
    PyErr_SetString(PyExc_TypeError, "need(t, name, dtype=None, shape=None)");
    return nullptr;
  }
  PyObject* dtype = n > 2 ? args[2] : Py_None;
  PyObject* shape = n > 3 ? args[3] : Py_None;
  bool right = false;
  try {
    right = is_right(args[0], dtype, shape);
  } catch (const std::exception&) {                  // (a tensor without sizes or storage of its own: the general check)
  }
  if (PyErr_Occurred()) PyErr_Clear();
  if (right) Py_RETURN_NONE;
  if (!g_otherwise) {
    PyErr_SetString(PyExc_RuntimeError, "need: no function was given to `otherwise`");
    return nullptr;
  }
  return PyObject_CallFunctionObjArgs(g_otherwise, args[0], args[1], dtype, shape, nullptr);
}

PyObject* otherwise(PyObject*, PyObject* fn) {
  Py_INCREF(fn);
  Py_XSETREF(g_otherwise, fn);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"need", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(need)), METH_FASTCALL, "check an operand"},
                         {"otherwise", otherwise, METH_O, "the general check, called for what `need` does not pass"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "mf_host_call", "operand checks and calls of the kernel libraries", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit_mf_host_call() {
  LaunchType.tp_name = "mf_host_call.Launch";
  LaunchType.tp_basicsize = sizeof(Launch);
  LaunchType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  LaunchType.tp_vectorcall_offset = offsetof(Launch, call);
  LaunchType.tp_call = PyVectorcall_Call;
  LaunchType.tp_new = launch_new;
  RecordType.tp_name = "mf_host_call.Record";
  RecordType.tp_basicsize = sizeof(Record);
  RecordType.tp_flags = Py_TPFLAGS_DEFAULT;
  RecordType.tp_new = record_new;
  RecordType.tp_dealloc = record_free;
  RecordType.tp_methods = record_methods;
  if (PyType_Ready(&LaunchType) < 0 || PyType_Ready(&RecordType) < 0) return nullptr;
  PyObject* ctypes = PyImport_ImportModule("ctypes");
  if (!ctypes) return nullptr;
  Py_XSETREF(g_array, PyObject_GetAttrString(ctypes, "Array"));
  Py_XSETREF(g_pointer, PyObject_GetAttrString(ctypes, "c_void_p"));
  Py_DECREF(ctypes);
  if (!g_array || !g_pointer) return nullptr;
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  Py_INCREF(&LaunchType);
  if (PyModule_AddObject(m, "Launch", reinterpret_cast<PyObject*>(&LaunchType)) < 0) return nullptr;
  Py_INCREF(&RecordType);
  if (PyModule_AddObject(m, "Record", reinterpret_cast<PyObject*>(&RecordType)) < 0) return nullptr;
  return m;
}
