// CPython module dsmoe._host: the per-tensor part of a layer call's host work.
// A layer holds 3 (E + S) expert weights; checking their shapes and taking their
// addresses one by one in Python cost about 1 us each (E 64: 0.2 ms per call).
//
// scan(weights, masters, x, gate_w, gate_bias, E, S, k) checks everything that
// dsmoe.ops.check_layer_args and moe_layer check (gate_bias None: not there, in a
// backward).  It returns None when anything
// is not exactly what the kernels take from an eager call (a tensor subclass,
// another device, a stride, a wrong shape): the caller then goes through those
// Python checks, which name the fault or handle the case.  Else it returns
// (inter width, shared inter width, whether anything requires grad, the six host
// arrays of weight addresses as bytes).
// addresses(tensors) returns the data pointers of a list of tensors as bytes.
// empty_like(tensors, float32) returns new tensors of their shapes (contiguous, on
// their device, in their dtype or float32).
#include <Python.h>

#include <cstdint>
#include <cstring>
#include <utility>
#include <vector>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

namespace {

PyTypeObject* g_parameter = nullptr;

// An ordinary strided device tensor: no subclass, no lazy conjugate, negation or
// zero, no wrapper of a functional transform.
bool plain(PyObject* o, const at::Tensor** out) {
  if (Py_TYPE(o) != g_parameter && Py_TYPE(o) != reinterpret_cast<PyTypeObject*>(THPVariableClass)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  static const c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot,
                                        c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                        c10::DispatchKey::ZeroTensor, c10::DispatchKey::Functionalize,
                                        c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper});
  if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || t.key_set().has_any(odd)) return false;
  *out = &t;
  return true;
}

bool matrix(const at::Tensor& t, c10::ScalarType dtype, const c10::Device& dev, int64_t rows, int64_t cols) {
  return t.scalar_type() == dtype && t.device() == dev && t.dim() == 2 && t.size(0) == rows && t.size(1) == cols &&
         t.is_contiguous();
}

PyObject* scan(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject *weights, *masters, *ox, *ogw, *ogb;
  int E, S;
  long k;
  if (!PyArg_ParseTuple(args, "O!O!OOOiil", &PyList_Type, &weights, &PyList_Type, &masters, &ox, &ogw, &ogb, &E, &S, &k))
    return nullptr;
  const at::Tensor *x, *gw, *gb;
  const Py_ssize_t n = PyList_GET_SIZE(weights), nm = PyList_GET_SIZE(masters);
  if (E < 1 || S < 0 || n != 3 * ((Py_ssize_t)E + S) || (nm != 0 && nm != n) || k < 1 || k > E) Py_RETURN_NONE;
  if (!plain(ox, &x) || !plain(ogw, &gw) || (ogb != Py_None && !plain(ogb, &gb))) Py_RETURN_NONE;
  const c10::ScalarType dt = x->scalar_type();
  const c10::Device dev = x->device();
  if ((dt != at::kFloat && dt != at::kBFloat16) || x->dim() != 2 || !x->is_contiguous()) Py_RETURN_NONE;
  if (nm && dt != at::kBFloat16) Py_RETURN_NONE;
  const int64_t D = x->size(1);
  if (!matrix(*gw, at::kFloat, dev, E, D)) Py_RETURN_NONE;
  if (ogb != Py_None && (gb->scalar_type() != at::kFloat || gb->device() != dev || gb->dim() != 1 ||
                         gb->size(0) != E || !gb->is_contiguous()))
    Py_RETURN_NONE;
  bool grad = x->requires_grad() || gw->requires_grad();
  int64_t inter[2] = {0, 0};
  const int count[2] = {E, S};
  PyObject* arrays[6] = {};
  Py_ssize_t at = 0;
  bool ok = true;
  for (int grp = 0; grp < 2 && ok; ++grp) {
    for (int w = 0; w < 3 && ok; ++w) {
      PyObject* b = PyBytes_FromStringAndSize(nullptr, count[grp] * (Py_ssize_t)sizeof(void*));
      if (!b) {
        for (PyObject* a : arrays) Py_XDECREF(a);
        return nullptr;
      }
      arrays[3 * grp + w] = b;
      char* dst = PyBytes_AS_STRING(b);
      for (int i = 0; i < count[grp] && ok; ++i, ++at) {
        const at::Tensor* t;
        ok = plain(PyList_GET_ITEM(weights, at), &t);
        if (!ok) break;
        if (w == 0 && i == 0 && t->dim() == 2) inter[grp] = t->size(0);
        ok = w == 1 ? matrix(*t, dt, dev, D, inter[grp]) : matrix(*t, dt, dev, inter[grp], D);
        if (!ok) break;
        grad = grad || t->requires_grad();
        if (nm) {
          const at::Tensor* mt;
          ok = plain(PyList_GET_ITEM(masters, at), &mt) && mt->scalar_type() == at::kFloat &&
               mt->sizes() == t->sizes() && mt->device() == dev;
          if (!ok) break;
          grad = grad || mt->requires_grad();
        }
        const void* p = t->const_data_ptr();
        std::memcpy(dst + (size_t)i * sizeof(void*), &p, sizeof(void*));
      }
    }
  }
  if (!ok) {
    for (PyObject* a : arrays) Py_XDECREF(a);
    Py_RETURN_NONE;
  }
  return Py_BuildValue("LLN(NNNNNN)", (long long)inter[0], (long long)inter[1], PyBool_FromLong(grad), arrays[0],
                       arrays[1], arrays[2], arrays[3], arrays[4], arrays[5]);
  END_HANDLE_TH_ERRORS
}

PyObject* addresses(PyObject*, PyObject* list) {
  HANDLE_TH_ERRORS
  if (!PyList_Check(list)) {
    PyErr_SetString(PyExc_TypeError, "addresses: a list of tensors");
    return nullptr;
  }
  const Py_ssize_t n = PyList_GET_SIZE(list);
  PyObject* b = PyBytes_FromStringAndSize(nullptr, n * (Py_ssize_t)sizeof(void*));
  if (!b) return nullptr;
  char* dst = PyBytes_AS_STRING(b);
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = PyList_GET_ITEM(list, i);
    if (!THPVariable_Check(o)) {
      Py_DECREF(b);
      PyErr_SetString(PyExc_TypeError, "addresses: a list of tensors");
      return nullptr;
    }
    const void* p = THPVariable_Unpack(o).unsafeGetTensorImpl()->data();
    std::memcpy(dst + (size_t)i * sizeof(void*), &p, sizeof(void*));
  }
  return b;
  END_HANDLE_TH_ERRORS
}

PyObject* empty_like(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  PyObject* list;
  int f32;
  if (!PyArg_ParseTuple(args, "O!p", &PyList_Type, &list, &f32)) return nullptr;
  const Py_ssize_t n = PyList_GET_SIZE(list);
  for (Py_ssize_t i = 0; i < n; ++i)
    if (!THPVariable_Check(PyList_GET_ITEM(list, i))) {
      PyErr_SetString(PyExc_TypeError, "empty_like: a list of tensors");
      return nullptr;
    }
  std::vector<at::Tensor> made;
  made.reserve(n);
  for (Py_ssize_t i = 0; i < n; ++i) {
    const at::Tensor& t = THPVariable_Unpack(PyList_GET_ITEM(list, i));
    made.push_back(at::empty(t.sizes(), t.options().dtype(f32 ? at::kFloat : t.scalar_type()).requires_grad(false)));
  }
  PyObject* out = PyList_New(n);
  if (!out) return nullptr;
  for (Py_ssize_t i = 0; i < n; ++i) {
    PyObject* o = THPVariable_Wrap(std::move(made[i]));
    if (!o) {
      Py_DECREF(out);
      return nullptr;
    }
    PyList_SET_ITEM(out, i, o);
  }
  return out;
  END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {{"scan", scan, METH_VARARGS, nullptr}, {"addresses", addresses, METH_O, nullptr},
                         {"empty_like", empty_like, METH_VARARGS, nullptr}, {}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  PyObject* nn = PyImport_ImportModule("torch.nn.parameter");
  if (!nn) return nullptr;
  g_parameter = reinterpret_cast<PyTypeObject*>(PyObject_GetAttrString(nn, "Parameter"));
  Py_DECREF(nn);
  if (!g_parameter) return nullptr;
  return PyModule_Create(&module);
}
