// OperationInvocation.submit's way into hyle_hip_plan_launch: a CPython extension, because a small launch is bound by
// what the host spends on it.  Converting eight arguments and two binding arrays through ctypes takes 1.3 us of the 2.4 us
// that a submit of two inputs spends in Python, here it is 0.2 (a layer of one token in six submits is as long as its
// submits).  The GIL is released for the launch, which may wait for room in the queue.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include "hyle_hip.h"

namespace {

constexpr Py_ssize_t kMostInputs = HYLE_HIP_MAX_INPUTS, kMostOutputs = HYLE_HIP_MAX_OUTPUTS;

PyObject *pointer_type = nullptr;  // ctypes.c_void_p

// An address: an int, None for null, or a c_void_p of either.  Anything else is refused here; the caller then asks ctypes.
bool address_of(PyObject *object, void **out) {
  if (PyLong_Check(object)) {
    *out = reinterpret_cast<void *>(PyLong_AsUnsignedLongLongMask(object));
    return !PyErr_Occurred();
  }
  *out = nullptr;
  if (object == Py_None) return true;
  const int pointer = PyObject_IsInstance(object, pointer_type);
  if (pointer < 0) return false;
  if (pointer == 0) {
    PyErr_Format(PyExc_TypeError, "cannot be converted to pointer: %.100s", Py_TYPE(object)->tp_name);
    return false;
  }
  PyObject *value = PyObject_GetAttrString(object, "value");
  if (value == nullptr) return false;
  if (value != Py_None) *out = reinterpret_cast<void *>(PyLong_AsUnsignedLongLongMask(value));
  Py_DECREF(value);
  return !PyErr_Occurred();
}

bool addresses_of(PyObject *sequence, void **out, Py_ssize_t most, uint32_t *count) {
  if (PyObject_Size(sequence) < 0) return false;  // an iterator is no sequence
  PyObject *items = PySequence_Fast(sequence, "a sequence of device addresses is expected");
  if (items == nullptr) return false;
  const Py_ssize_t size = PySequence_Fast_GET_SIZE(items);
  bool fine = size <= most;
  if (!fine) PyErr_SetString(PyExc_IndexError, "more bindings than an operation can have");
  for (Py_ssize_t i = 0; fine && i < size; ++i) fine = address_of(PySequence_Fast_GET_ITEM(items, i), &out[i]);
  Py_DECREF(items);
  *count = static_cast<uint32_t>(size);
  return fine;
}

// launch(function, plan, inputs, outputs, workspace, workspace size, stream) -> status code
PyObject *launch(PyObject *, PyObject *const *args, Py_ssize_t count) {
  if (count != 7) {
    PyErr_SetString(PyExc_TypeError, "launch takes seven arguments");
    return nullptr;
  }
  void *function, *plan, *workspace, *stream, *inputs[kMostInputs], *outputs[kMostOutputs];
  uint32_t input_count, output_count;
  if (!address_of(args[0], &function) || !address_of(args[1], &plan) || !addresses_of(args[2], inputs, kMostInputs, &input_count) ||
      !addresses_of(args[3], outputs, kMostOutputs, &output_count) || !address_of(args[4], &workspace) || !address_of(args[6], &stream))
    return nullptr;
  const size_t size = PyLong_AsSize_t(args[5]);
  if (size == static_cast<size_t>(-1) && PyErr_Occurred()) return nullptr;
  hyle_hip_status status;
  Py_BEGIN_ALLOW_THREADS
  status = reinterpret_cast<decltype(&hyle_hip_plan_launch)>(function)(static_cast<const hyle_hip_plan *>(plan), inputs, input_count, outputs,
                                                                       output_count, workspace, size, stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(static_cast<long>(status));
}

PyObject *data_ptr_name = nullptr;  // "data_ptr"

// The addresses of a list or tuple of tensors: what their data_ptr() answers.
bool storage_of(PyObject *tensors, void **out, Py_ssize_t most, uint32_t *count) {
  const Py_ssize_t size = PySequence_Fast_GET_SIZE(tensors);
  if (size > most) {
    PyErr_SetString(PyExc_IndexError, "more bindings than an operation can have");
    return false;
  }
  for (Py_ssize_t i = 0; i < size; ++i) {
    // (data_ptr() of a tensor subclass is Python: it may change the list)
    if (i >= PySequence_Fast_GET_SIZE(tensors)) {
      PyErr_SetString(PyExc_RuntimeError, "bindings changed while they were read");
      return false;
    }
    PyObject *tensor = PySequence_Fast_GET_ITEM(tensors, i);
    Py_INCREF(tensor);
    PyObject *address = PyObject_CallMethodNoArgs(tensor, data_ptr_name);
    Py_DECREF(tensor);
    if (address == nullptr) return false;
    const bool fine = address_of(address, &out[i]);
    Py_DECREF(address);
    if (!fine) return false;
  }
  *count = static_cast<uint32_t>(size);
  return true;
}

// launch_tensors(function, current device, current stream of a device, plan, inputs, outputs, workspace, workspace size)
// -> status code: launch with lists or tuples of tensors, on the current device's current stream.
PyObject *launch_tensors(PyObject *, PyObject *const *args, Py_ssize_t count) {
  if (count != 8 || !(PyList_Check(args[4]) || PyTuple_Check(args[4])) || !(PyList_Check(args[5]) || PyTuple_Check(args[5]))) {
    PyErr_SetString(PyExc_TypeError, "launch_tensors takes eight arguments, bindings as lists or tuples");
    return nullptr;
  }
  void *function, *plan, *workspace, *stream, *inputs[kMostInputs], *outputs[kMostOutputs];
  uint32_t input_count, output_count;
  PyObject *device = PyObject_CallNoArgs(args[1]);
  if (device == nullptr) return nullptr;
  PyObject *handle = PyObject_CallOneArg(args[2], device);
  Py_DECREF(device);
  if (handle == nullptr) return nullptr;
  const bool found = address_of(handle, &stream);
  Py_DECREF(handle);
  if (!found || !address_of(args[0], &function) || !address_of(args[3], &plan) || !storage_of(args[4], inputs, kMostInputs, &input_count) ||
      !storage_of(args[5], outputs, kMostOutputs, &output_count) || !address_of(args[6], &workspace))
    return nullptr;
  const size_t size = PyLong_AsSize_t(args[7]);
  if (size == static_cast<size_t>(-1) && PyErr_Occurred()) return nullptr;
  hyle_hip_status status;
  Py_BEGIN_ALLOW_THREADS
  status = reinterpret_cast<decltype(&hyle_hip_plan_launch)>(function)(static_cast<const hyle_hip_plan *>(plan), inputs, input_count, outputs,
                                                                       output_count, workspace, size, stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(static_cast<long>(status));
}

PyMethodDef methods[] = {{"launch_tensors", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(launch_tensors)), METH_FASTCALL, nullptr},
                         {"launch", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(launch)), METH_FASTCALL, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_submit", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__submit() {
  PyObject *ctypes = PyImport_ImportModule("ctypes");
  if (ctypes == nullptr) return nullptr;
  pointer_type = PyObject_GetAttrString(ctypes, "c_void_p");
  Py_DECREF(ctypes);
  data_ptr_name = PyUnicode_InternFromString("data_ptr");
  return pointer_type == nullptr || data_ptr_name == nullptr ? nullptr : PyModule_Create(&module);
}
