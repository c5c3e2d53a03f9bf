// Python extension _k3h_py: the per-call tensor checks of k3h.py, natively.  A typed
// call checks up to a dozen tensors before it launches; done in Python (device, dtype,
// contiguity, size and address, each an attribute call) they took longer than the
// launch itself: the fused op on 9 rows 10.9 -> 5.3 us per call (back to back, with the
// current stream's handle taken without a Stream object), the two calls of a KDA layer
// over 517 rows 25.8 -> 11.8 us.
//
//   dev(t, name, dtypes, numel=None, align=16): raises ValueError unless t is a
//     contiguous GPU tensor of one of `dtypes` (mask of the DT_* bits, 0 for any) with
//     at least numel elements at an address that is a multiple of align
//   ptr(t): data address of a tensor, None for None
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <exception>
#include <string>

namespace {

enum : long { DT_BF16 = 1, DT_F32 = 2, DT_U8 = 4, DT_E4M3 = 8, DT_I32 = 16, DT_I64 = 32 };

struct Dt {
  long bit;
  at::ScalarType type;
  const char* name;
};
const Dt kDts[] = {{DT_BF16, at::kBFloat16, "torch.bfloat16"}, {DT_F32, at::kFloat, "torch.float32"},
                   {DT_U8, at::kByte, "torch.uint8"},          {DT_E4M3, at::kFloat8_e4m3fn, "torch.float8_e4m3fn"},
                   {DT_I32, at::kInt, "torch.int32"},          {DT_I64, at::kLong, "torch.int64"}};

bool dtype_ok(at::ScalarType t, long mask) {
  if (mask == 0) return true;
  for (const Dt& d : kDts)
    if ((mask & d.bit) && d.type == t) return true;
  return false;
}

PyObject* reject(const char* name, const std::string& why) {
  PyErr_SetString(PyExc_ValueError, (std::string(name) + ": " + why).c_str());
  return nullptr;
}

// The Python-visible dtype ("torch.bfloat16") of a rejected tensor.
std::string dtype_name(PyObject* t) {
  std::string s = "?";
  if (PyObject* d = PyObject_GetAttrString(t, "dtype")) {
    if (PyObject* r = PyObject_Str(d)) {
      if (const char* c = PyUnicode_AsUTF8(r)) s = c;
      Py_DECREF(r);
    }
    Py_DECREF(d);
  }
  PyErr_Clear();
  return s;
}

bool is_int(PyObject* o, const char* what, long long* out) {
  *out = PyLong_AsLongLong(o);
  if (*out == -1 && PyErr_Occurred()) {
    PyErr_Format(PyExc_TypeError, "dev: %s must be an integer", what);
    return false;
  }
  return true;
}

PyObject* dev(PyObject*, PyObject* const* args, Py_ssize_t nargs, PyObject* kwnames) {
  PyObject *numel_o = nargs > 3 ? args[3] : Py_None, *align_o = nargs > 4 ? args[4] : nullptr;
  if (nargs < 3 || nargs > 5) {
    PyErr_SetString(PyExc_TypeError, "dev(t, name, dtypes, numel=None, align=16)");
    return nullptr;
  }
  for (Py_ssize_t k = 0; kwnames && k < PyTuple_GET_SIZE(kwnames); ++k) {
    PyObject* key = PyTuple_GET_ITEM(kwnames, k);
    if (!PyUnicode_CompareWithASCIIString(key, "align") && nargs < 5) {
      align_o = args[nargs + k];
    } else if (!PyUnicode_CompareWithASCIIString(key, "numel") && nargs < 4) {
      numel_o = args[nargs + k];
    } else {
      PyErr_Format(PyExc_TypeError, "dev: unexpected keyword %U", key);
      return nullptr;
    }
  }
  const char* name = PyUnicode_AsUTF8(args[1]);
  if (!name) return nullptr;
  long long mask = 0, numel = -1, align = 16;
  if (!is_int(args[2], "dtypes", &mask) || (numel_o != Py_None && !is_int(numel_o, "numel", &numel)) ||
      (align_o && !is_int(align_o, "align", &align)))
    return nullptr;
  try {
    if (!THPVariable_Check(args[0])) return reject(name, "expected a torch tensor");
    const at::Tensor& t = THPVariable_Unpack(args[0]);
    if (!t.is_cuda()) return reject(name, "must be a GPU tensor (got " + t.device().str() + ")");
    if (!dtype_ok(t.scalar_type(), (long)mask)) {
      std::string want;
      for (const Dt& d : kDts)
        if (mask & d.bit) want += (want.empty() ? "" : ", ") + std::string(d.name);
      return reject(name, "dtype " + dtype_name(args[0]) + " not in [" + want + "]");
    }
    if (!t.is_contiguous()) return reject(name, "must be contiguous");
    if (numel_o != Py_None && t.numel() < numel)
      return reject(name, "needs at least " + std::to_string(numel) + " elements, has " +
                              std::to_string(t.numel()));
    if (align > 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % (uintptr_t)align)
      return reject(name, "must be " + std::to_string(align) + "-byte aligned");
  } catch (const std::exception& e) {
    return reject(name, e.what());
  }
  Py_RETURN_NONE;
}

PyObject* ptr(PyObject*, PyObject* t) {
  if (t == Py_None) Py_RETURN_NONE;
  if (!THPVariable_Check(t)) {
    PyErr_SetString(PyExc_ValueError, "ptr: expected a torch tensor or None");
    return nullptr;
  }
  try {
    return PyLong_FromVoidPtr(THPVariable_Unpack(t).data_ptr());
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_ValueError, e.what());
    return nullptr;
  }
}

PyMethodDef kMethods[] = {
    {"dev", (PyCFunction)(void (*)(void))dev, METH_FASTCALL | METH_KEYWORDS,
     "dev(t, name, dtypes, numel=None, align=16): check a kernel argument"},
    {"ptr", ptr, METH_O, "ptr(t): data address, None for None"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_k3h_py", nullptr, -1, kMethods, nullptr, nullptr,
                       nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__k3h_py() {
  PyObject* m = PyModule_Create(&kModule);
  if (!m) return nullptr;
  if (PyModule_AddIntConstant(m, "BF16", DT_BF16) || PyModule_AddIntConstant(m, "F32", DT_F32) ||
      PyModule_AddIntConstant(m, "U8", DT_U8 | DT_E4M3) || PyModule_AddIntConstant(m, "I32", DT_I32) ||
      PyModule_AddIntConstant(m, "I64", DT_I64) || PyModule_AddIntConstant(m, "ANY", 0)) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
