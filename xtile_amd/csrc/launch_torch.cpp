// The Python module `_launch`: xt.launch over torch tensors in one native call.
//
// A launch through the Python checks (signature JSON, six attribute reads and
// a size product a tensor, a device context manager, ctypes arrays) took 12-16
// us of host time, several times what a small kernel runs; this call takes the
// tensors' fields from their C++ objects and hands them to xt_gpu_run_buffers.
//
//   bind(run, free, type)                xt_gpu_run_buffers and xt_free of the library
//                                        that owns the module handles, as addresses,
//                                        and the handles' type (None: capsules)
//   launch(handle, buffers, func, stream) True when the program was enqueued.
//                                        False when anything is not the plain
//                                        case: the caller then takes the checked
//                                        path, which launches it or raises.
//
// The plain case: every buffer exactly a torch.Tensor with storage of its own
// (no subclass, no functorch or functionalisation wrapper), contiguous, of its
// memref's type and shape, all on one GPU.  Only a HIP error after the launch
// was tried raises here.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdint>
#include <exception>
#include <string>

#include "xtile_amd.h"

namespace {

typedef int (*RunFn)(xt_module*, const char*, const xt_buffer*, int, void*, char**);
typedef void (*FreeFn)(void*);
RunFn g_run = nullptr;
FreeFn g_free = nullptr;
PyTypeObject* g_handle = nullptr;  // the ctypes binding's NativeModule; nullptr: capsules
PyObject* g_ptr_name = nullptr;    // "_ptr"

constexpr const char* kCapsuleName = "xtile_amd.xt_module";
constexpr int kMost = 16;

// The module behind a handle of the binding in use; nullptr for anything else,
// whatever attributes it has.
xt_module* module_of(PyObject* handle) {
  if (!g_handle)
    return PyCapsule_IsValid(handle, kCapsuleName)
               ? static_cast<xt_module*>(PyCapsule_GetPointer(handle, kCapsuleName))
               : nullptr;
  if (!PyObject_TypeCheck(handle, g_handle)) return nullptr;
  PyObject* p = PyObject_GetAttr(handle, g_ptr_name);
  if (!p) {
    PyErr_Clear();
    return nullptr;
  }
  void* v = PyLong_Check(p) ? PyLong_AsVoidPtr(p) : nullptr;
  Py_DECREF(p);
  if (PyErr_Occurred()) PyErr_Clear();
  return static_cast<xt_module*>(v);
}

int dtype_of(c10::ScalarType t) {
  switch (t) {
    case c10::ScalarType::Float: return XT_F32;
    case c10::ScalarType::Half: return XT_F16;
    case c10::ScalarType::BFloat16: return XT_BF16;
    case c10::ScalarType::Char: return XT_I8;
    case c10::ScalarType::Int: return XT_I32;
    default: return -1;
  }
}

// What only the checked path handles: wrappers whose data is elsewhere.
const c10::DispatchKeySet kWrapped =
    c10::DispatchKeySet({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                         c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::FuncTorchGradWrapper,
                         c10::DispatchKey::Functionalize, c10::DispatchKey::Batched});

// Makes `device` current and puts back the one that was.
struct OnDevice {
  c10::DeviceIndex was, now;
  explicit OnDevice(c10::DeviceIndex d) : was(c10::hip::current_device()), now(d) {
    if (was != now) c10::hip::set_device(now);
  }
  ~OnDevice() {
    try {
      if (was != now) c10::hip::set_device(was);
    } catch (const std::exception&) {  // the launch's own status stands
    }
  }
};

PyObject* launch_plain(PyObject* const* args) {
  xt_module* m = g_run ? module_of(args[0]) : nullptr;
  if (!m || !PyTuple_CheckExact(args[1])) Py_RETURN_FALSE;
  const char* func = "";
  if (args[2] != Py_None) {
    func = PyUnicode_Check(args[2]) ? PyUnicode_AsUTF8(args[2]) : nullptr;
    if (!func) {
      PyErr_Clear();
      Py_RETURN_FALSE;
    }
  }
  const Py_ssize_t n = PyTuple_GET_SIZE(args[1]);
  if (n < 1 || n > kMost) Py_RETURN_FALSE;
  xt_buffer b[kMost];
  c10::DeviceIndex device = -1;
  for (Py_ssize_t k = 0; k < n; ++k) {
    PyObject* o = PyTuple_GET_ITEM(args[1], k);
    if (!THPVariable_CheckExact(o)) Py_RETURN_FALSE;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || !t.has_storage() ||
        t.key_set().has_any(kWrapped) || t.unsafeGetTensorImpl()->has_symbolic_sizes_strides() || !t.is_contiguous())
      Py_RETURN_FALSE;
    if (k == 0) device = t.get_device();
    else if (t.get_device() != device) Py_RETURN_FALSE;
    static_assert(sizeof(long long) == sizeof(int64_t), "shapes are passed as they are");
    b[k].ptr = t.data_ptr();
    b[k].shape = reinterpret_cast<const long long*>(t.sizes().data());
    b[k].rank = static_cast<int>(t.dim());
    b[k].dtype = dtype_of(t.scalar_type());
  }
  OnDevice on(device);
  void* stream;
  if (args[3] == Py_None) {
    stream = c10::hip::getCurrentHIPStream(device).stream();
  } else {
    stream = PyLong_Check(args[3]) ? PyLong_AsVoidPtr(args[3]) : nullptr;
    if (!PyLong_Check(args[3]) || PyErr_Occurred()) {
      PyErr_Clear();
      Py_RETURN_FALSE;
    }
  }
  char* err = nullptr;
  int st = XT_ERR_ARGUMENT;
  Py_BEGIN_ALLOW_THREADS;
  try {
    st = g_run(m, func, b, static_cast<int>(n), stream, &err);
  } catch (const std::exception&) {  // out of memory while planning
  }
  Py_END_ALLOW_THREADS;
  const std::string text = err ? err : "launch failed";
  if (err) g_free(err);
  if (st == XT_OK) Py_RETURN_TRUE;
  if (st == XT_ERR_DEVICE) {
    PyErr_SetString(PyExc_RuntimeError, text.c_str());
    return nullptr;
  }
  Py_RETURN_FALSE;  // refused before any launch: the checked path says why
}

PyObject* launch(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  if (nargs != 4) {
    PyErr_SetString(PyExc_TypeError, "launch(handle, buffers, func, stream)");
    return nullptr;
  }
  try {
    return launch_plain(args);
  } catch (const std::exception&) {
    if (PyErr_Occurred()) PyErr_Clear();
    Py_RETURN_FALSE;  // a tensor without data: the checked path raises what torch says
  }
}

PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  void* run = nargs == 3 && PyLong_Check(args[0]) ? PyLong_AsVoidPtr(args[0]) : nullptr;
  void* release = nargs == 3 && PyLong_Check(args[1]) ? PyLong_AsVoidPtr(args[1]) : nullptr;
  if (PyErr_Occurred()) return nullptr;
  if (!run || !release || (args[2] != Py_None && !PyType_Check(args[2]))) {
    PyErr_SetString(PyExc_ValueError, "bind(address of xt_gpu_run_buffers, address of xt_free, handle type or None)");
    return nullptr;
  }
  PyObject* const was = reinterpret_cast<PyObject*>(g_handle);
  g_handle = nullptr;
  if (args[2] != Py_None) {
    Py_INCREF(args[2]);
    g_handle = reinterpret_cast<PyTypeObject*>(args[2]);
  }
  Py_XDECREF(was);
  g_run = reinterpret_cast<RunFn>(run);
  g_free = reinterpret_cast<FreeFn>(release);
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {
    {"launch", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(launch)), METH_FASTCALL,
     "launch(handle, buffers, func, stream) -> bool: whether the program was enqueued"},
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(bind)), METH_FASTCALL,
     "bind(xt_gpu_run_buffers, xt_free, type): the library's functions, as addresses, and its handles' type"},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_launch", "xt.launch over torch tensors", -1, kMethods,
                       nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__launch(void) {
  g_ptr_name = PyUnicode_InternFromString("_ptr");
  return g_ptr_name ? PyModule_Create(&kModule) : nullptr;
}
