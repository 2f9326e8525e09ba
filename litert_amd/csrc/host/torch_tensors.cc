// Output tensors and scratch for the Python ops, allocated without torch.empty's argument parsing: a small
// call's host part was 6.0 us, 1.7 of it that one function (the launch 3.1), and its kernel takes 3 to 5.
// Built against the installed torch and loaded by its version only; without it ops call torch.empty.
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Exceptions.h>

#include <ATen/ATen.h>
#include <c10/core/Allocator.h>
#include <c10/core/DeviceGuard.h>
#include <pybind11/pybind11.h>

#include <memory>
#include <utility>

namespace {

// empty(like, rows, columns): rows x columns on like's device, one value of `type` each.
template <c10::ScalarType kType>
PyObject* Empty(PyObject*, PyObject* const* args, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  if (count != 3) return PyErr_Format(PyExc_TypeError, "expected 3 arguments, got %zd", count);
  if (!THPVariable_Check(args[0])) return PyErr_Format(PyExc_TypeError, "expected a tensor");
  const long long rows = PyLong_AsLongLong(args[1]);
  const long long columns = PyLong_AsLongLong(args[2]);
  if (PyErr_Occurred()) return nullptr;
  const c10::Device device = THPVariable_Unpack(args[0]).device();
  at::Tensor out;
  {
    // As torch.empty does: an allocation that has to ask the device, or wait for it, stops no other thread.
    pybind11::gil_scoped_release unlocked;
    out = at::empty({rows, columns}, at::TensorOptions().dtype(kType).device(device));
  }
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

constexpr const char* kMemoryName = "litert_amd.memory";

void FreeMemory(PyObject* capsule) {
  delete static_cast<at::DataPtr*>(PyCapsule_GetPointer(capsule, kMemoryName));
}

// scratch(like, bytes): (address, what holds the memory), from like's device's allocator on its current
// stream. No tensor around it: 0.55 us, 0.95 with one.
PyObject* Scratch(PyObject*, PyObject* const* args, Py_ssize_t count) {
  HANDLE_TH_ERRORS
  if (count != 2) return PyErr_Format(PyExc_TypeError, "expected 2 arguments, got %zd", count);
  if (!THPVariable_Check(args[0])) return PyErr_Format(PyExc_TypeError, "expected a tensor");
  const size_t bytes = PyLong_AsSize_t(args[1]);
  if (PyErr_Occurred()) return nullptr;
  const c10::Device device = THPVariable_Unpack(args[0]).device();
  std::unique_ptr<at::DataPtr> memory;
  {
    pybind11::gil_scoped_release unlocked;
    c10::DeviceGuard guard(device);
    memory = std::make_unique<at::DataPtr>(c10::GetAllocator(device.type())->allocate(bytes));
  }
  PyObject* address = PyLong_FromVoidPtr(memory->get());
  if (!address) return nullptr;
  PyObject* holder = PyCapsule_New(memory.get(), kMemoryName, FreeMemory);
  if (!holder) {
    Py_DECREF(address);
    return nullptr;
  }
  memory.release();  // the capsule's
  PyObject* both = PyTuple_Pack(2, address, holder);
  Py_DECREF(address);
  Py_DECREF(holder);
  return both;
  END_HANDLE_TH_ERRORS
}

#define LRTFC_METHOD(name, ...) \
  {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&__VA_ARGS__)), METH_FASTCALL, nullptr}

PyMethodDef kMethods[] = {
    LRTFC_METHOD("empty_int8", Empty<c10::ScalarType::Char>),
    LRTFC_METHOD("empty_float32", Empty<c10::ScalarType::Float>),
    LRTFC_METHOD("scratch", Scratch),
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "litert_amd_tensors", nullptr, -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_litert_amd_tensors() { return PyModule_Create(&kModule); }
