// Calls of the kernel launchers (`int ome_xxx(..., hipStream_t)`) from Python without ctypes, which converts each argument through an object
// of its own: a launcher of 21 arguments takes 4.5 us that way and 0.8 so.
//
// bind(name, address, kinds): `kinds` has a letter an argument: p a pointer (or None), i a 32-bit, l a 64-bit integer, f a float.  call(name, *args) calls it
// and raises by `fail(name, code)` if it returns anything but 0; a name that is not bound, arguments of any other number or type and keywords go to
// `other(name, *args, ...)`, which calls by ctypes.
//
// One prototype serves every launcher: by the System V calling convention of x86-64 integers and pointers fill six registers and then eight
// bytes each of the stack, floats the low halves of eight vector registers, both in their own order, and a callee does not
// look at what lies beyond its own arguments.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <cstring>

#if !defined(__x86_64__) || !defined(__linux__)
#error "the calling convention of x86-64 Linux"
#endif

namespace {

constexpr int REGS = 6, FLOATS = 8, SHORT = 18, LONG = 58;   // integers in registers, floats, integers on the stack

struct Launcher {
  void* f;
  int n;
  char kinds[REGS + LONG + FLOATS + 1];
};

PyObject *g_bound, *g_other, *g_fail;

void release(PyObject* capsule) { delete static_cast<Launcher*>(PyCapsule_GetPointer(capsule, nullptr)); }

#define OME_S6(k) uint64_t, uint64_t, uint64_t, uint64_t, uint64_t, uint64_t
#define OME_F8 float, float, float, float, float, float, float, float
typedef int (*ShortCall)(OME_S6(0), OME_F8, OME_S6(0), OME_S6(1), OME_S6(2));
typedef int (*LongCall)(OME_S6(0), OME_F8, OME_S6(0), OME_S6(1), OME_S6(2), OME_S6(3), OME_S6(4), OME_S6(5), OME_S6(6), OME_S6(7), OME_S6(8), uint64_t, uint64_t,
                        uint64_t, uint64_t);

int invoke(const Launcher& l, const uint64_t* a, const float* x, int integers) {
  const uint64_t* s = a + REGS;
#define OME_A6(b, k) b[6 * k], b[6 * k + 1], b[6 * k + 2], b[6 * k + 3], b[6 * k + 4], b[6 * k + 5]
#define OME_X8 x[0], x[1], x[2], x[3], x[4], x[5], x[6], x[7]
  if (integers <= REGS + SHORT)
    return reinterpret_cast<ShortCall>(l.f)(OME_A6(a, 0), OME_X8, OME_A6(s, 0), OME_A6(s, 1), OME_A6(s, 2));
  return reinterpret_cast<LongCall>(l.f)(OME_A6(a, 0), OME_X8, OME_A6(s, 0), OME_A6(s, 1), OME_A6(s, 2), OME_A6(s, 3), OME_A6(s, 4), OME_A6(s, 5), OME_A6(s, 6),
                                         OME_A6(s, 7), OME_A6(s, 8), s[54], s[55], s[56], s[57]);
}

PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* names) {
  PyObject* const capsule = nargs > 0 && !names ? PyDict_GetItem(g_bound, args[0]) : nullptr;   // (borrowed)
  const Launcher* const bound = capsule ? static_cast<const Launcher*>(PyCapsule_GetPointer(capsule, nullptr)) : nullptr;
  if (bound && bound->n == nargs - 1) {
    const Launcher l = *bound;
    uint64_t a[REGS + LONG];
    float x[FLOATS] = {};
    int ints = 0, floats = 0;
    bool known = true;
    for (int i = 0; i < l.n && known; ++i) {
      PyObject* const o = args[1 + i];
      if (l.kinds[i] == 'f') {
        if (PyFloat_Check(o)) x[floats++] = (float)PyFloat_AS_DOUBLE(o);
        else known = false;
      } else if (PyLong_Check(o)) {
        const uint64_t v = PyLong_AsUnsignedLongLongMask(o);
        a[ints++] = l.kinds[i] == 'i' ? (uint64_t)(int64_t)(int32_t)v : v;
      } else if (o == Py_None && l.kinds[i] == 'p') {
        a[ints++] = 0;
      } else {
        known = false;
      }
    }
    if (known && !PyErr_Occurred()) {
      for (int i = ints; i < REGS + (ints <= REGS + SHORT ? SHORT : LONG); ++i) a[i] = 0;
      int code;
      Py_BEGIN_ALLOW_THREADS;
      code = invoke(l, a, x, ints);
      Py_END_ALLOW_THREADS;
      if (code == 0) Py_RETURN_NONE;
      PyObject* const why = PyLong_FromLong(code);
      if (!why) return nullptr;
      PyObject* const r = PyObject_CallFunctionObjArgs(g_fail, args[0], why, nullptr);
      Py_DECREF(why);
      return r;
    }
    PyErr_Clear();
  }
  return PyObject_Vectorcall(g_other, args, (size_t)nargs, names);
}

PyObject* bind(PyObject*, PyObject* args) {
  PyObject* name;
  unsigned long long address;
  const char* kinds;
  if (!PyArg_ParseTuple(args, "UKs", &name, &address, &kinds)) return nullptr;
  const size_t n = strlen(kinds);
  size_t floats = 0;
  for (size_t i = 0; i < n; ++i) {
    if (!strchr("pilf", kinds[i])) return PyErr_Format(PyExc_ValueError, "unknown kind '%c'", kinds[i]);
    floats += kinds[i] == 'f';
  }
  if (floats > FLOATS || n - floats > REGS + LONG || !address) Py_RETURN_FALSE;   // (left to `other`)
  Launcher* const l = new Launcher;
  l->f = reinterpret_cast<void*>(address);
  l->n = (int)n;
  memcpy(l->kinds, kinds, n + 1);
  PyObject* const capsule = PyCapsule_New(l, nullptr, release);
  if (!capsule) {
    delete l;
    return nullptr;
  }
  const int rc = PyDict_SetItem(g_bound, name, capsule);
  Py_DECREF(capsule);
  if (rc) return nullptr;
  Py_RETURN_TRUE;
}

PyObject* hooks(PyObject*, PyObject* args) {
  PyObject *other, *fail;
  if (!PyArg_ParseTuple(args, "OO", &other, &fail)) return nullptr;
  Py_INCREF(other);
  Py_INCREF(fail);
  Py_XSETREF(g_other, other);
  Py_XSETREF(g_fail, fail);
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {{"call", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(call)), METH_FASTCALL | METH_KEYWORDS, "call(name, *args, lib)"},
                         {"bind", bind, METH_VARARGS, "bind(name, address, kinds)"},
                         {"hooks", hooks, METH_VARARGS, "hooks(other, fail)"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "ome_call", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_ome_call() {
  g_bound = PyDict_New();
  return g_bound ? PyModule_Create(&module) : nullptr;
}
