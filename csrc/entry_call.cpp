// Calls of the mixer kernels' C entry points from Python.
//
// An entry point takes some 30 pointers, sizes and floats. Through ctypes each of
// them is an object first: of the 42 us that the host took for a recurrence of four
// launches, 14 were the launches. Here tensors are handed over as they are and
// read in C++: entry(address, result, name) returns a callable whose arguments are
// tensors or None (a pointer), integers and booleans, and floats (single precision).
//
// The call itself relies on the x86-64 System V convention: integers and pointers, in
// order, take registers and then the stack, floats registers of their own (up to
// eight), and a callee does not see what lies behind its own arguments. So one
// prototype with the most of both serves all entry points.
#include <Python.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <string>
#include <utility>

#if !defined(__x86_64__) || defined(_WIN32)
#error "entry points are called by the x86-64 System V convention"
#endif

namespace {

constexpr int kInts = 48, kFloats = 8;

struct Entry {
  void* fn;
  int result;  // 0: none, 1: int, 2: long
  std::string name;
};

template <size_t>
using Int = int64_t;
template <size_t>
using Float = float;

template <size_t... I, size_t... F>
int64_t invoke(void* fn, const int64_t* a, const float* f,
               std::index_sequence<I...>, std::index_sequence<F...>) {
  using Fn = int64_t (*)(Int<I>..., Float<F>...);
  return reinterpret_cast<Fn>(fn)(a[I]..., f[F]...);
}

void free_entry(PyObject* capsule) {
  delete static_cast<Entry*>(PyCapsule_GetPointer(capsule, nullptr));
}

PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  const Entry* e =
      static_cast<const Entry*>(PyCapsule_GetPointer(self, nullptr));
  if (e == nullptr) return nullptr;
  int64_t a[kInts] = {};
  float f[kFloats] = {};
  int na = 0, nf = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = args[i];
    if (PyFloat_Check(o)) {
      if (nf == kFloats) {
        PyErr_Format(PyExc_TypeError, "%s: too many floats", e->name.c_str());
        return nullptr;
      }
      f[nf++] = static_cast<float>(PyFloat_AS_DOUBLE(o));
      continue;
    }
    if (na == kInts) {
      PyErr_Format(PyExc_TypeError, "%s: too many arguments", e->name.c_str());
      return nullptr;
    }
    if (o == Py_None) {
      a[na++] = 0;
    } else if (PyLong_Check(o)) {
      const long long v = PyLong_AsLongLong(o);
      if (v == -1 && PyErr_Occurred()) return nullptr;
      a[na++] = v;
    } else if (THPVariable_Check(o)) {
      a[na++] = reinterpret_cast<int64_t>(THPVariable_Unpack(o).data_ptr());
    } else {
      PyErr_Format(PyExc_TypeError, "%s: argument %zd is a %s",
                   e->name.c_str(), i, Py_TYPE(o)->tp_name);
      return nullptr;
    }
  }
  int64_t r;
  Py_BEGIN_ALLOW_THREADS
  r = invoke(e->fn, a, f, std::make_index_sequence<kInts>{},
             std::make_index_sequence<kFloats>{});
  Py_END_ALLOW_THREADS
  if (e->result == 0) Py_RETURN_NONE;
  return PyLong_FromLongLong(e->result == 1 ? static_cast<int32_t>(r) : r);
  END_HANDLE_TH_ERRORS
}

PyMethodDef kCall = {"entry_point", reinterpret_cast<PyCFunction>(
                                        reinterpret_cast<void (*)()>(call)),
                     METH_FASTCALL, nullptr};

PyObject* entry(PyObject*, PyObject* args) {
  unsigned long long address;
  int result;
  const char* name;
  if (!PyArg_ParseTuple(args, "Kis", &address, &result, &name)) return nullptr;
  if (address == 0) {
    PyErr_SetString(PyExc_ValueError, "entry: no address");
    return nullptr;
  }
  auto* e = new Entry{reinterpret_cast<void*>(address), result, name};
  PyObject* capsule = PyCapsule_New(e, nullptr, free_entry);
  if (capsule == nullptr) {
    delete e;
    return nullptr;
  }
  PyObject* fn = PyCFunction_New(&kCall, capsule);
  Py_DECREF(capsule);
  return fn;
}

// Row stride (elements) of a 2-D view whose rows are contiguous.
PyObject* row_stride(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !THPVariable_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "row_stride(tensor, name)");
    return nullptr;
  }
  const at::Tensor& t = THPVariable_Unpack(args[0]);
  if (t.dim() != 2 || t.stride(1) != 1) {
    PyErr_Format(PyExc_ValueError,
                 "%S: need a 2-D view with unit inner stride", args[1]);
    return nullptr;
  }
  return PyLong_FromLongLong(t.stride(0));
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"entry", entry, METH_VARARGS, "entry(address, result, name)"},
    {"row_stride",
     reinterpret_cast<PyCFunction>(
         reinterpret_cast<void (*)()>(row_stride)),
     METH_FASTCALL, "row_stride(tensor, name)"},
    {nullptr, nullptr, 0, nullptr}};

}  // namespace

void register_entry_calls(PyObject* module) {
  if (PyModule_AddFunctions(module, kMethods) != 0) throw python_error();
}
