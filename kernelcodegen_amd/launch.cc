// The operators' calls in native code: one object per bound kernel that takes the operand tensors, allocates the result and
// launches on torch's current stream.
//
// A small call is as long as its host code.  Of the 5 us that a call took from Python (softmax of 64 x 512 4.9 us), the HIP
// launch itself is 2.4; the rest was the allocation through torch's argument parser (0.9 to 1.4 us), packing the arguments, the
// foreign-function call and two look-ups of the stream.  This does them in one step.
//
//   Launch(entry, handle, dims, num_pointers, num_scalars, fail, keep)
//       entry      address of kcg_hip_launch_packed (include/kcg_hip.h): the library itself is not linked
//       handle     kernel handle
//       dims       seven whole numbers: grid, block, LDS bytes
//       fail       called with a status that is not 0; raises
//       keep       any object that has to live as long
//   launch(pointer, ..., number, ...)      pointers as whole numbers or tensors; numbers as fp32
//   launch.result(shape, dtype)            a Launch whose call leaves the last pointer out: call(tensor, ..., number, ...)
//                                          allocates it on the first tensor's device and returns it
//   launch.result(None, None)              the result is like the first tensor
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>

#include <cmath>
#include <cstdint>
#include <cstring>
#include <vector>

namespace {

typedef int (*Entry)(void* handle, const uint32_t* dims, void* stream, const void* slots, int num_args);
constexpr int MAX_ARGS = 16;      // as many as the entry takes

struct Launch {
  PyObject_HEAD
  vectorcallfunc call;
  Entry entry;
  void* handle;
  uint32_t dims[7];
  int pointers, scalars;
  int result;                     // 0: no result, 1: shape and dtype, 2: like the first tensor
  std::vector<int64_t>* shape;
  at::ScalarType dtype;
  PyObject *fail, *keep;
};

// The launch on the current stream, without the GIL; the status of the entry.
int launch(const Launch* self, const uint64_t* slots) {
  void* stream = (void*)c10::hip::getCurrentHIPStream().stream();
  return self->entry(self->handle, self->dims, stream, slots, self->pointers + self->scalars);
}

bool scalar(PyObject* o, uint64_t& slot) {
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) return false;
  // a number beyond the fp32 range is an infinity, as the conversion to a C float gives it
  const float f = v > 3.4028235677973366e38 ? INFINITY : v < -3.4028235677973366e38 ? -INFINITY : (float)v;
  slot = 0;
  memcpy(&slot, &f, sizeof f);
  return true;
}

PyObject* failed(Launch* self, int rc) {
  PyObject* r = PyObject_CallFunction(self->fail, "i", rc);
  if (r) {
    Py_DECREF(r);
    PyErr_Format(PyExc_RuntimeError, "kernel launch failed with status %d", rc);
  }
  return nullptr;
}

PyObject* callLaunch(PyObject* me, PyObject* const* args, size_t nargsf, PyObject* kwnames) {
  HANDLE_TH_ERRORS
  Launch* self = (Launch*)me;
  const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
  const int given = self->pointers - (self->result ? 1 : 0);
  if ((kwnames && PyTuple_GET_SIZE(kwnames)) || n != given + self->scalars) {
    PyErr_Format(PyExc_TypeError, "a launch of this kernel takes %d pointers and %d numbers", given, self->scalars);
    return nullptr;
  }
  uint64_t slots[MAX_ARGS];
  for (int i = 0; i < given; ++i) {
    if (THPVariable_Check(args[i])) {
      slots[i] = (uint64_t)(uintptr_t)THPVariable_Unpack(args[i]).data_ptr();
    } else {
      PyObject* whole = PyNumber_Index(args[i]);
      if (!whole) return nullptr;
      slots[i] = PyLong_AsUnsignedLongLong(whole);
      Py_DECREF(whole);
      if (slots[i] == (uint64_t)-1 && PyErr_Occurred()) return nullptr;
    }
  }
  for (int i = 0; i < self->scalars; ++i)
    if (!scalar(args[given + i], slots[self->pointers + i])) return nullptr;
  int rc;
  if (!self->result) {
    {
      pybind11::gil_scoped_release unlocked;      // (an exception takes it back)
      rc = launch(self, slots);
    }
    if (rc) return failed(self, rc);
    Py_RETURN_NONE;
  }
  if (!given || !THPVariable_Check(args[0])) {
    PyErr_SetString(PyExc_TypeError, "the first operand must be a tensor");
    return nullptr;
  }
  at::Tensor out;
  {
    const at::Tensor& like = THPVariable_Unpack(args[0]);
    pybind11::gil_scoped_release unlocked;
    out = self->result == 2 ? at::empty_like(like) : at::empty(*self->shape, like.options().dtype(self->dtype).requires_grad(false));
    slots[given] = (uint64_t)(uintptr_t)out.data_ptr();
    rc = launch(self, slots);
  }
  if (rc) return failed(self, rc);
  return THPVariable_Wrap(out);
  END_HANDLE_TH_ERRORS
}

PyTypeObject LaunchType = {PyVarObject_HEAD_INIT(nullptr, 0)};

PyObject* newLaunch(PyTypeObject* type, PyObject* args, PyObject* kwargs) {
  HANDLE_TH_ERRORS
  unsigned long long entry, handle;
  unsigned int d[7];
  int pointers, scalars;
  PyObject *fail, *keep;
  if ((kwargs && PyDict_GET_SIZE(kwargs)) ||
      !PyArg_ParseTuple(args, "KK(IIIIIII)iiOO", &entry, &handle, &d[0], &d[1], &d[2], &d[3], &d[4], &d[5], &d[6], &pointers, &scalars, &fail, &keep)) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "Launch takes no keyword arguments");
    return nullptr;
  }
  if (!entry || !handle || pointers < 1 || scalars < 0 || pointers + scalars > MAX_ARGS) {
    PyErr_SetString(PyExc_ValueError, "Launch: no entry, no kernel, or not 1 to 16 arguments");
    return nullptr;
  }
  Launch* self = (Launch*)type->tp_alloc(type, 0);
  if (!self) return nullptr;
  self->call = callLaunch;
  self->entry = (Entry)(uintptr_t)entry;
  self->handle = (void*)(uintptr_t)handle;
  memcpy(self->dims, d, sizeof d);
  self->pointers = pointers;
  self->scalars = scalars;
  self->result = 0;
  self->shape = nullptr;
  Py_INCREF(fail);
  self->fail = fail;
  Py_INCREF(keep);
  self->keep = keep;
  return (PyObject*)self;
  END_HANDLE_TH_ERRORS
}

PyObject* withResult(PyObject* me, PyObject* args) {
  HANDLE_TH_ERRORS
  Launch* self = (Launch*)me;
  PyObject *shape, *dtype;
  if (!PyArg_ParseTuple(args, "OO", &shape, &dtype)) return nullptr;
  std::vector<int64_t> sizes;
  if (shape != Py_None) {
    PyObject* seq = PySequence_Fast(shape, "the shape is a sequence of whole numbers");
    if (!seq) return nullptr;
    for (Py_ssize_t i = 0; i < PySequence_Fast_GET_SIZE(seq); ++i) {
      const long long v = PyLong_AsLongLong(PySequence_Fast_GET_ITEM(seq, i));
      if (v == -1 && PyErr_Occurred()) {
        Py_DECREF(seq);
        return nullptr;
      }
      sizes.push_back(v);
    }
    Py_DECREF(seq);
    if (!THPDtype_Check(dtype)) {
      PyErr_SetString(PyExc_TypeError, "a shape needs a torch dtype");
      return nullptr;
    }
  }
  Launch* made = (Launch*)LaunchType.tp_alloc(&LaunchType, 0);
  if (!made) return nullptr;
  made->call = callLaunch;
  made->entry = self->entry;
  made->handle = self->handle;
  memcpy(made->dims, self->dims, sizeof made->dims);
  made->pointers = self->pointers;
  made->scalars = self->scalars;
  made->result = shape == Py_None ? 2 : 1;
  made->shape = nullptr;
  if (shape != Py_None) {
    made->shape = new std::vector<int64_t>(std::move(sizes));
    made->dtype = ((THPDtype*)dtype)->scalar_type;
  }
  Py_INCREF(self->fail);
  made->fail = self->fail;
  Py_INCREF(self->keep);
  made->keep = self->keep;
  return (PyObject*)made;
  END_HANDLE_TH_ERRORS
}

void freeLaunch(PyObject* me) {
  Launch* self = (Launch*)me;
  delete self->shape;
  Py_XDECREF(self->fail);
  Py_XDECREF(self->keep);
  Py_TYPE(me)->tp_free(me);
}

PyMethodDef methods[] = {{"result", withResult, METH_VARARGS, "result(shape, dtype): a Launch that allocates and returns its last pointer's tensor"},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", "bound kernel launches on torch tensors", -1, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__launch(void) {
  LaunchType.tp_name = "kernelcodegen_amd._launch.Launch";
  LaunchType.tp_basicsize = sizeof(Launch);
  LaunchType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  LaunchType.tp_vectorcall_offset = offsetof(Launch, call);
  LaunchType.tp_call = PyVectorcall_Call;
  LaunchType.tp_new = newLaunch;
  LaunchType.tp_dealloc = freeLaunch;
  LaunchType.tp_methods = methods;
  if (PyType_Ready(&LaunchType) < 0) return nullptr;
  PyObject* m = PyModule_Create(&module);
  if (!m) return nullptr;
  Py_INCREF(&LaunchType);
  if (PyModule_AddObject(m, "Launch", (PyObject*)&LaunchType) < 0) {
    Py_DECREF(&LaunchType);
    Py_DECREF(m);
    return nullptr;
  }
  // the version whose headers this was built on (torch.__version__), for the importer to compare
  if (PyModule_AddStringConstant(m, "torch_version", KCG_TORCH_VERSION) < 0) {
    Py_DECREF(m);
    return nullptr;
  }
  return m;
}
