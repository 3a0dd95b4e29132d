// The call of a kernel object in native code: what KernelAdapter.__call__ (adapter.py) does for a good call on the current
// device and torch's current stream: look at every operand, allocate the output and the workspace, call the C entry point.
// Whatever it does not settle (another device, a stream of the caller's, a CPU tensor, a subclass, a wrong shape, ...) it
// hands back as NotImplemented, and the adapter's own code carries it out or says what is wrong.
//
// Why: at one row the kernel takes 4.4 us and the call took the interpreter 17 (W4A16, N = K = 4096, through a layer) and 12
// (MXFP4): five attribute look-ups and comparisons an operand, a ctypes conversion an argument.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/Dtype.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/core/impl/DeviceGuardImplInterface.h>
#include <dlfcn.h>

#include <vector>

#include "../../include/dqgemm.h"

namespace {

constexpr int kMaxDevices = 64;
constexpr int kMaxPointers = 8;
bool g_initialised[kMaxDevices];  // the library's init() ran there; written and read under the interpreter's lock
const char* (*g_last_error)() = nullptr;
PyObject* g_raw_stream = nullptr;  // torch's private call for the current stream of a GPU
void* g_library = nullptr;

struct Args {
  void* p[kMaxPointers];
  const int* i;
  float f;
  size_t ws;
  void* stream;
};
using Invoke = int (*)(void*, const Args&);

// One line per entry point that a kernel object of a layer or of a decode loop calls: its arguments in order.
struct Entry {
  const char* name;
  int pointers, ints;
  Invoke invoke;
};
#define DQ_CALL(NAME) reinterpret_cast<decltype(&NAME)>(fn)
const Entry kEntries[] = {
    {"call_dequantize_gemv_w4a16", 5, 7,
     [](void* fn, const Args& a) {
       return DQ_CALL(call_dequantize_gemv_w4a16)(a.p[0], a.p[1], a.p[2], a.p[3], a.p[4], a.i[0], a.i[1], a.i[2], a.i[3], a.i[4], a.i[5], a.i[6], a.stream);
     }},
    {"call_dequantize_gemv_w4a16_ws", 6, 7,
     [](void* fn, const Args& a) {
       return DQ_CALL(call_dequantize_gemv_w4a16_ws)(a.p[0], a.p[1], a.p[2], a.p[3], a.p[4], a.p[5], a.ws, a.i[0], a.i[1], a.i[2], a.i[3], a.i[4], a.i[5], a.i[6], a.stream);
     }},
    {"call_dequant_gemm_bf16_mxfp4", 5, 6,
     [](void* fn, const Args& a) {
       return DQ_CALL(call_dequant_gemm_bf16_mxfp4)(a.p[0], a.p[1], a.p[2], a.p[3], a.p[4], a.i[0], a.i[1], a.i[2], a.i[3], a.i[4], a.i[5], a.stream);
     }},
    {"call_dequant_gemm_bf16_mxfp4_ws", 6, 7,
     [](void* fn, const Args& a) {
       return DQ_CALL(call_dequant_gemm_bf16_mxfp4_ws)(a.p[0], a.p[1], a.p[2], a.p[3], a.p[4], a.p[5], a.ws, a.i[0], a.i[1], a.i[2], a.i[3], a.i[4], a.i[5], a.i[6], a.stream);
     }},
    {"call_bitlinear_fp16", 4, 4,
     [](void* fn, const Args& a) {
       return DQ_CALL(call_bitlinear_fp16)(a.p[0], a.p[1], a.p[2], a.p[3], a.ws, a.i[0], a.i[1], a.i[2], a.i[3], a.f, a.stream);
     }},
    {"call_gemm_int8xint4", 3, 6,
     [](void* fn, const Args& a) {
       return DQ_CALL(call_gemm_int8xint4)(a.p[0], a.p[1], a.p[2], a.i[0], a.i[1], a.i[2], a.i[3], a.i[4], a.i[5], a.stream);
     }},
};
#undef DQ_CALL

struct Param {
  at::ScalarType dtype;
  bool packed;
  std::vector<int64_t> shape;
  int role;  // 0: the caller's; 1: allocated and returned; 2: workspace
};

struct Call {
  PyObject_HEAD
  const Entry* entry;
  void* fn;
  std::vector<Param>* params;
  int inputs;                 // parameters of role 0
  int returned;               // the one that is returned, or -1
  int slot[kMaxPointers];     // pointer argument -> parameter, -1: NULL
  std::vector<int>* ints;
  float f;
  size_t ws;
};

PyObject* not_settled() { Py_RETURN_NOTIMPLEMENTED; }

// Other threads run while blocks are allocated and the kernel is launched, either of which may have to wait.
struct WithoutInterpreter {
  PyThreadState* const state = PyEval_SaveThread();
  ~WithoutInterpreter() { PyEval_RestoreThread(state); }
};

// call(*inputs): the caller's parameters in order
PyObject* call_call(PyObject* self_, PyObject* args, PyObject* kwargs) {
  HANDLE_TH_ERRORS
  Call* const self = reinterpret_cast<Call*>(self_);
  if ((kwargs && PyDict_GET_SIZE(kwargs)) || PyTuple_GET_SIZE(args) != self->inputs || !g_library) return not_settled();
  // a mode that sees torch's calls is to see the ones that the adapter makes
  if (at::impl::PythonTorchFunctionTLS::stack_len() != 0 || c10::impl::TorchDispatchModeTLS::any_modes_set()) return not_settled();
  const size_t n = self->params->size();
  void* pointers[16] = {};
  int device = -1;
  size_t at_input = 0;
  for (size_t k = 0; k < n; ++k) {
    const Param& p = (*self->params)[k];
    if (p.role != 0) continue;
    PyObject* const o = PyTuple_GET_ITEM(args, at_input++);
    if (o == Py_None) continue;
    if (!THPVariable_CheckExact(o)) return not_settled();
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.device().is_cuda() || t.layout() != at::kStrided || !t.has_storage()) return not_settled();
    if (device < 0) device = t.device().index();
    const at::ScalarType dtype = t.scalar_type();
    if (t.device().index() != device || !(dtype == p.dtype || (p.packed && (dtype == at::kChar || dtype == at::kByte))) ||
        t.sizes() != at::IntArrayRef(p.shape) || t.numel() == 0 || !t.is_contiguous())
      return not_settled();
    pointers[k] = t.data_ptr();
  }
  if (device < 0 || device >= kMaxDevices || !g_initialised[device]) return not_settled();
  const auto* const guard = c10::impl::getDeviceGuardImpl(at::kCUDA);
  if (guard->getDevice().index() != device) return not_settled();
  // torch's current stream, which the blocks below are allocated under
  PyObject* const index = PyLong_FromLong(device);
  PyObject* const raw = index ? PyObject_CallOneArg(g_raw_stream, index) : nullptr;
  Py_XDECREF(index);
  if (!raw) return nullptr;
  void* const stream = reinterpret_cast<void*>(PyLong_AsUnsignedLongLong(raw));
  Py_DECREF(raw);
  if (PyErr_Occurred()) return nullptr;
  at::Tensor returned, scratch;
  int rc;
  {
    const WithoutInterpreter released;
    const at::Device dev(at::kCUDA, static_cast<c10::DeviceIndex>(device));
    for (size_t k = 0; k < n; ++k) {
      const Param& p = (*self->params)[k];
      if (p.role == 0) continue;
      at::Tensor t = at::empty(p.shape, at::TensorOptions().dtype(p.dtype).device(dev));
      pointers[k] = t.data_ptr();
      (p.role == 1 ? returned : scratch) = std::move(t);
    }
    Args a;
    for (int s = 0; s < self->entry->pointers; ++s) a.p[s] = self->slot[s] < 0 ? nullptr : pointers[self->slot[s]];
    a.i = self->ints->data();
    a.f = self->f;
    a.ws = self->ws;
    a.stream = stream;
    rc = self->entry->invoke(self->fn, a);
  }
  if (rc != 0) {
    PyErr_Format(PyExc_RuntimeError, "Kernel call failed: %s", g_last_error());
    return nullptr;
  }
  if (self->returned < 0) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(returned));
  END_HANDLE_TH_ERRORS
}

void call_dealloc(PyObject* self_) {
  Call* const self = reinterpret_cast<Call*>(self_);
  delete self->params;
  delete self->ints;
  Py_TYPE(self_)->tp_free(self_);
}

PyTypeObject CallType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// bind(entry, ((dtype, packed, shape, role), ...), slots, ints, f, ws) -> callable, or None where there is no such entry
PyObject* bind(PyObject*, PyObject* args) {
  HANDLE_TH_ERRORS
  const char* name;
  PyObject *params, *slots, *ints;
  float f;
  Py_ssize_t ws;
  if (!PyArg_ParseTuple(args, "sO!O!O!fn", &name, &PyTuple_Type, &params, &PyTuple_Type, &slots, &PyTuple_Type, &ints, &f, &ws)) return nullptr;
  const Entry* entry = nullptr;
  for (const Entry& e : kEntries)
    if (!strcmp(e.name, name)) entry = &e;
  void* const fn = entry && g_library ? dlsym(g_library, name) : nullptr;
  const Py_ssize_t n = PyTuple_GET_SIZE(params);
  if (!fn || PyTuple_GET_SIZE(slots) != entry->pointers || PyTuple_GET_SIZE(ints) != entry->ints || n > 16) Py_RETURN_NONE;
  Call* const self = PyObject_New(Call, &CallType);
  if (!self) return nullptr;
  self->entry = entry;
  self->fn = fn;
  self->params = new std::vector<Param>();
  self->ints = new std::vector<int>();
  self->inputs = 0;
  self->returned = -1;
  self->f = f;
  self->ws = static_cast<size_t>(ws);
  bool good = true;
  int workspaces = 0;
  for (Py_ssize_t k = 0; k < n && good; ++k) {
    PyObject *dtype, *shape;
    int packed, role;
    if (!PyArg_ParseTuple(PyTuple_GET_ITEM(params, k), "OpO!i", &dtype, &packed, &PyTuple_Type, &shape, &role) || !THPDtype_Check(dtype)) {
      good = false;
      break;
    }
    Param p{reinterpret_cast<THPDtype*>(dtype)->scalar_type, packed != 0, {}, role};
    for (Py_ssize_t d = 0; d < PyTuple_GET_SIZE(shape); ++d) p.shape.push_back(PyLong_AsLongLong(PyTuple_GET_ITEM(shape, d)));
    self->inputs += role == 0;
    workspaces += role == 2;
    if (role == 1) {
      good = self->returned < 0;
      self->returned = static_cast<int>(k);
    }
    self->params->push_back(std::move(p));
  }
  good = good && workspaces <= 1;
  for (int s = 0; s < entry->pointers && good; ++s) {
    self->slot[s] = static_cast<int>(PyLong_AsLong(PyTuple_GET_ITEM(slots, s)));
    good = self->slot[s] < n;
  }
  for (int s = 0; s < entry->ints; ++s) self->ints->push_back(static_cast<int>(PyLong_AsLong(PyTuple_GET_ITEM(ints, s))));
  if (good && !PyErr_Occurred()) return reinterpret_cast<PyObject*>(self);
  Py_DECREF(self);
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
  END_HANDLE_TH_ERRORS
}

// open(path of libdqgemm.so, torch's call for the current stream)
PyObject* open_library(PyObject*, PyObject* args) {
  const char* path;
  PyObject* raw_stream;
  if (!PyArg_ParseTuple(args, "sO", &path, &raw_stream)) return nullptr;
  if (!g_library && PyCallable_Check(raw_stream)) {
    void* const library = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    g_last_error = library ? reinterpret_cast<decltype(g_last_error)>(dlsym(library, "get_last_error")) : nullptr;
    if (g_last_error) {
      Py_INCREF(raw_stream);
      g_raw_stream = raw_stream;
      g_library = library;
    }
  }
  return PyBool_FromLong(g_library != nullptr);
}

PyObject* initialised(PyObject*, PyObject* args) {
  int device;
  if (!PyArg_ParseTuple(args, "i", &device)) return nullptr;
  if (device >= 0 && device < kMaxDevices) g_initialised[device] = true;
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {{"bind", bind, METH_VARARGS, nullptr},
                          {"open", open_library, METH_VARARGS, nullptr},
                          {"initialised", initialised, METH_VARARGS, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_hostcall", nullptr, -1, kMethods};

}  // namespace

#define DQ_TEXT_OF(X) #X
#define DQ_TEXT(X) DQ_TEXT_OF(X)

PyMODINIT_FUNC PyInit__hostcall(void) {
  CallType.tp_name = "tilelang_amd._hostcall.Call";
  CallType.tp_basicsize = sizeof(Call);
  CallType.tp_flags = Py_TPFLAGS_DEFAULT;
  CallType.tp_dealloc = call_dealloc;
  CallType.tp_call = call_call;
  if (PyType_Ready(&CallType) < 0) return nullptr;
  PyObject* const module = PyModule_Create(&kModule);
  // the torch whose headers this was compiled against, which the caller compares before it makes a call
  if (module && PyModule_AddStringConstant(module, "built_for", DQ_TEXT(DQ_BUILT_FOR)) < 0) {
    Py_DECREF(module);
    return nullptr;
  }
  return module;
}
