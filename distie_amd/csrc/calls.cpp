// Calls of the libraries' C functions from Python, with tensors as arguments, and the two other things that every launch does: the
// allocation of its result and the look whether its tensors are on the device and contiguous.
//
// A step that is launched kernel by kernel makes 120 to 260 such calls, and where prompts are short the host is what it waits for: 11 us
// a launch, of which ctypes took 2.0 for a function of 21 arguments, `data_ptr()` of ten tensors 1.0, `torch.empty` 1.8 and the looks at
// the tensors 0.8. Here they take 0.3, 0.05, 0.8 and 0.15 us.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>
#include <ATen/ATen.h>

#include <cstring>
#include <exception>

#if !defined(__x86_64__)
#error "arguments are laid out as the calls of x86-64 Linux have them"
#endif

namespace {

// On x86-64 Linux the whole-number arguments of a call go to six registers and then, in order, to the stack, eight bytes each, and its
// floating-point arguments to eight registers of their own, whatever the order of the two kinds. So a call with all fourteen registers
// and enough of the stack filled is a call of every function with at most that many arguments: it looks at those that are its own.
constexpr int WHOLE_REGISTERS = 6, FLOAT_REGISTERS = 8, STACK = 34;
typedef int64_t W;
typedef int (*Any)(W, W, W, W, W, W, double, double, double, double, double, double, double, double,
                   W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W, W);

int call_any(void* function, const W* w, const double* f) {
  const W* s = w + WHOLE_REGISTERS;
  return reinterpret_cast<Any>(function)(w[0], w[1], w[2], w[3], w[4], w[5], f[0], f[1], f[2], f[3], f[4], f[5], f[6], f[7],
                                         s[0], s[1], s[2], s[3], s[4], s[5], s[6], s[7], s[8], s[9], s[10], s[11], s[12], s[13], s[14],
                                         s[15], s[16], s[17], s[18], s[19], s[20], s[21], s[22], s[23], s[24], s[25], s[26], s[27],
                                         s[28], s[29], s[30], s[31], s[32], s[33]);
}

struct Function {
  PyObject_HEAD
  vectorcallfunc vectorcall;
  PyObject* slow;                // the same as ctypes has it, for arguments that are no tensors, numbers or None
  void* address;
  int count;
  char kinds[WHOLE_REGISTERS + STACK + FLOAT_REGISTERS + 1];     // an argument each: 'p' pointer, 'w' whole number, 'f' float
};

bool failed(const std::exception& e) {
  if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, e.what());
  return false;
}

// A tensor's address; false, with Python's error set, if it has none.
bool address_of(PyObject* o, W* out) {
  try {
    *out = reinterpret_cast<W>(THPVariable_Unpack(o).data_ptr());
    return true;
  } catch (const std::exception& e) {
    return failed(e);
  }
}

PyObject* call_slowly(Function* f, PyObject* const* args, Py_ssize_t n) {
  THPObjectPtr tuple(PyTuple_New(n));
  if (!tuple) return nullptr;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* item;
    if (THPVariable_Check(args[i])) {
      W at = 0;
      if (!address_of(args[i], &at)) return nullptr;
      item = PyLong_FromUnsignedLongLong(static_cast<unsigned long long>(at));
      if (item == nullptr) return nullptr;
    } else {
      item = args[i];
      Py_INCREF(item);
    }
    PyTuple_SET_ITEM(tuple.get(), i, item);
  }
  return PyObject_Call(f->slow, tuple.get(), nullptr);
}

PyObject* function_call(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* names) {
  Function* f = reinterpret_cast<Function*>(self);
  const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
  if (n != f->count || (names != nullptr && PyTuple_GET_SIZE(names) != 0)) {
    PyErr_Format(PyExc_TypeError, "this function takes %d positional arguments, not %zd", f->count, n);
    return nullptr;
  }
  W whole[WHOLE_REGISTERS + STACK];
  double floats[FLOAT_REGISTERS] = {};
  int w = 0, fl = 0;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* const a = args[i];
    switch (f->kinds[i]) {
      case 'f': {
        const double v = PyFloat_AsDouble(a);
        if (v == -1.0 && PyErr_Occurred()) return nullptr;
        const float single = static_cast<float>(v);
        std::memcpy(&floats[fl++], &single, sizeof(single));       // the low half of its register
        break;
      }
      case 'w':
        whole[w] = static_cast<W>(PyLong_AsUnsignedLongLongMask(a));
        if (whole[w] == -1 && PyErr_Occurred()) return nullptr;
        ++w;
        break;
      default:
        if (a == Py_None) {
          whole[w++] = 0;
        } else if (THPVariable_Check(a)) {
          if (!address_of(a, &whole[w++])) return nullptr;
        } else if (PyLong_Check(a)) {
          whole[w] = static_cast<W>(PyLong_AsUnsignedLongLongMask(a));
          if (whole[w] == -1 && PyErr_Occurred()) return nullptr;
          ++w;
        } else {
          return call_slowly(f, args, n);
        }
    }
  }
  for (; w < WHOLE_REGISTERS + STACK; ++w) whole[w] = 0;
  int status;
  Py_BEGIN_ALLOW_THREADS
  status = call_any(f->address, whole, floats);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(status);
}

PyObject* function_new(PyTypeObject* type, PyObject* args, PyObject*) {
  PyObject* slow;
  unsigned long long address;
  const char* kinds;
  if (!PyArg_ParseTuple(args, "OKs", &slow, &address, &kinds)) return nullptr;
  int whole = 0, floats = 0;
  for (const char* k = kinds; *k; ++k) {
    if (*k == 'f') ++floats;
    else if (*k == 'w' || *k == 'p') ++whole;
    else floats = FLOAT_REGISTERS + 1;
  }
  if (whole > WHOLE_REGISTERS + STACK || floats > FLOAT_REGISTERS || address == 0 || !PyCallable_Check(slow)) {
    PyErr_SetString(PyExc_ValueError, "a function of too many arguments, or of kinds that are not known here");
    return nullptr;
  }
  PyObject* self = type->tp_alloc(type, 0);
  if (self == nullptr) return nullptr;
  Function* f = reinterpret_cast<Function*>(self);
  f->vectorcall = function_call;
  Py_INCREF(slow);
  f->slow = slow;
  f->address = reinterpret_cast<void*>(address);
  f->count = whole + floats;
  std::memcpy(f->kinds, kinds, f->count + 1);
  return self;
}

void function_dealloc(PyObject* self) {
  Py_XDECREF(reinterpret_cast<Function*>(self)->slow);
  Py_TYPE(self)->tp_free(self);
}

PyTypeObject function_type = [] {
  PyTypeObject t = {PyVarObject_HEAD_INIT(nullptr, 0)};
  t.tp_name = "distie_calls.Function";
  t.tp_basicsize = sizeof(Function);
  t.tp_dealloc = function_dealloc;
  t.tp_vectorcall_offset = offsetof(Function, vectorcall);
  t.tp_call = PyVectorcall_Call;
  t.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  t.tp_doc = "Function(ctypes function, address, kinds): a C function that returns an int";
  t.tp_new = function_new;
  return t;
}();

// owned(device index, tensor or None, ..) -> whether all of them are contiguous and on that GPU
PyObject* owned(PyObject*, PyObject* const* args, Py_ssize_t n) {
  const long index = n > 0 ? PyLong_AsLong(args[0]) : -1;
  if (index == -1 && PyErr_Occurred()) return nullptr;
  try {
    for (Py_ssize_t i = 1; i < n; ++i) {
      if (args[i] == Py_None) continue;
      if (!THPVariable_Check(args[i])) Py_RETURN_FALSE;
      const at::Tensor& t = THPVariable_Unpack(args[i]);
      if (!t.is_cuda() || t.get_device() != index || !t.is_contiguous()) Py_RETURN_FALSE;
    }
  } catch (const std::exception& e) {
    failed(e);
    return nullptr;
  }
  Py_RETURN_TRUE;
}

// empty(device index, shape, dtype) -> as torch.empty
PyObject* empty(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 3 || !(PyTuple_Check(args[1]) || PyLong_Check(args[1])) || !THPDtype_Check(args[2])) {
    PyErr_SetString(PyExc_TypeError, "empty(device index, shape, dtype)");
    return nullptr;
  }
  const long index = PyLong_AsLong(args[0]);
  if (index == -1 && PyErr_Occurred()) return nullptr;
  c10::SmallVector<int64_t, 6> sizes;
  const bool one = PyLong_Check(args[1]);
  for (Py_ssize_t i = 0; i < (one ? 1 : PyTuple_GET_SIZE(args[1])); ++i) {
    const long long size = PyLong_AsLongLong(one ? args[1] : PyTuple_GET_ITEM(args[1], i));
    if (size == -1 && PyErr_Occurred()) return nullptr;
    sizes.push_back(size);
  }
  const at::ScalarType dtype = reinterpret_cast<THPDtype*>(args[2])->scalar_type;
  try {
    at::Tensor t;
    {
      struct Released {
        PyThreadState* state = PyEval_SaveThread();
        ~Released() { PyEval_RestoreThread(state); }
      } released;
      t = at::empty(sizes, at::TensorOptions().dtype(dtype).device(at::Device(at::kCUDA, index)));
    }
    return THPVariable_Wrap(std::move(t));
  } catch (const c10::OutOfMemoryError& e) {
    // (its Python class is torch's own, by which callers know it)
    THPObjectPtr torch_module(PyImport_ImportModule("torch"));
    THPObjectPtr kind(torch_module ? PyObject_GetAttrString(torch_module.get(), "OutOfMemoryError") : nullptr);
    if (kind) PyErr_SetString(kind.get(), e.what_without_backtrace());
    return nullptr;
  } catch (const std::exception& e) {
    failed(e);
    return nullptr;
  }
}

PyMethodDef methods[] = {
    {"owned", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(owned)), METH_FASTCALL,
     "owned(device index, tensor or None, ..) -> whether all are contiguous and on that GPU"},
    {"empty", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(empty)), METH_FASTCALL,
     "empty(device index, shape, dtype) -> an uninitialised tensor on that GPU"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "distie_calls", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_distie_calls() {
  if (PyType_Ready(&function_type) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module);
  if (m == nullptr) return nullptr;
  Py_INCREF(&function_type);
  if (PyModule_AddObject(m, "Function", reinterpret_cast<PyObject*>(&function_type)) < 0) {
    Py_DECREF(&function_type);
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
