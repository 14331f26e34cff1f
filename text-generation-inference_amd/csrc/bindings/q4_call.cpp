// Host path of one eager linear call: y[..., N] = x[..., K] @ dequant(W) (+ bias) in one C call from Python.
//
// A call for a few tokens is bound by the host: 4096 x 4096 for one token runs 4.3 us on the GPU, and the checks, the output's
// allocation and a ctypes call with ten arguments took 7.6 us in Python, 5.6 us here.  A handle does the same steps and nothing else, on
// the same state: it reads the plans of the weight and the workspaces of the process where the Python code
// keeps them (the two dicts it is given) and holds no pointer of a call.  Whatever is not the plain case (a tensor
// subclass, a transform or a mode that watches operators, gradients to record, a strided or unaligned x, another
// device, no workspace yet, act-order calls that may be regrouped) is handed back as None:
// the Python code then decides, with its own errors.
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <stddef.h>
#include <string.h>

#include <algorithm>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include "q4_linear.h"

namespace {

using LinearFn = int (*)(const q4_weight*, const void*, const void*, void*, int, int, void*, size_t, int, void*);
using TunedFn = int (*)(const q4_weight*, const void*, const void*, void*, int, int, void*, size_t, int, int, int, int, void*);

LinearFn g_linear = nullptr;      // q4_linear_ex of the loaded library
TunedFn g_tuned = nullptr;        // q4_gemv_tuned
PyObject* g_workspaces = nullptr; // ops._workspaces
PyObject* g_check = nullptr;      // _lib.check: raises for a negative status

// What a weight's calls need.  The weight's tensors are kept alive by the PackedWeight that owns the object.
struct Call {
  PyObject_HEAD
  vectorcallfunc vectorcall;
  q4_weight weight;
  PyObject* plans;  // PackedWeight._plans
  int device;
  long first_regrouped_row;  // rows from which Python asks whether the call is regrouped
};

void call_dealloc(PyObject* self) {
  Py_XDECREF(((Call*)self)->plans);
  Py_TYPE(self)->tp_free(self);
}

bool watched() {
  if (c10::impl::dispatch_mode_enabled() || at::impl::torch_function_mode_enabled() || torch::jit::tracer::isTracing()) return true;
  static constexpr c10::DispatchKeySet kTransforms(
      {c10::DispatchKey::FuncTorchDynamicLayerFrontMode, c10::DispatchKey::FuncTorchDynamicLayerBackMode, c10::DispatchKey::Functionalize});
  return c10::impl::tls_local_dispatch_key_set().included_.has_any(kTransforms);
}

// a dense tensor of this GPU that operators would meet as it is; asked before anything else of a tensor (sizes of a nested one throw)
bool plain(const at::Tensor& t, int device) {
  const c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                 c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate, c10::DispatchKey::Negative,
                                 c10::DispatchKey::ZeroTensor, c10::DispatchKey::NestedTensor, c10::DispatchKey::AutogradNestedTensor});
  return t.is_cuda() && t.layout() == c10::kStrided && !t.key_set().has_any(odd) && t.get_device() == device && t.is_contiguous();
}

// An integer of a tuple.
bool item(PyObject* tuple, Py_ssize_t i, long* out) {
  if (i >= PyTuple_GET_SIZE(tuple)) return false;
  *out = PyLong_AsLong(PyTuple_GET_ITEM(tuple, i));
  if (*out != -1 || PyErr_Occurred() == nullptr) return true;
  PyErr_Clear();
  return false;
}

PyObject* find(PyObject* dict, unsigned long long a, long long b) {
  PyObject* key = Py_BuildValue("(KL)", a, b);
  if (key == nullptr) return nullptr;
  PyObject* got = PyDict_GetItemWithError(dict, key);
  Py_DECREF(key);
  return got;
}

PyObject* call(Call* self, PyObject* x_obj, PyObject* bias_obj, PyObject* owner) {
  if (!THPVariable_CheckExact(x_obj) || watched()) Py_RETURN_NONE;
  const at::Tensor& x = THPVariable_Unpack(x_obj);
  const q4_weight& w = self->weight;
  const auto type = x.scalar_type();
  if ((type != at::kHalf && type != at::kBFloat16) || !plain(x, self->device) || x.dim() < 2 || x.size(-1) != w.K) Py_RETURN_NONE;
  if (x.requires_grad() && c10::GradMode::is_enabled()) Py_RETURN_NONE;
  const void* bias = nullptr;
  if (bias_obj != Py_None) {
    if (!THPVariable_Check(bias_obj)) Py_RETURN_NONE;
    const at::Tensor& b = THPVariable_Unpack(bias_obj);
    if (b.scalar_type() != type || !plain(b, self->device) || b.numel() != w.N || (b.requires_grad() && c10::GradMode::is_enabled()))
      Py_RETURN_NONE;
    bias = b.const_data_ptr();
  }
  const void* xp = x.const_data_ptr();
  const long M = w.K > 0 ? (long)(x.numel() / w.K) : 0;
  if (M < 1 || M > INT32_MAX || M >= self->first_regrouped_row || w.N < 1 || (uintptr_t)xp % 16 != 0) Py_RETURN_NONE;
  if (c10::hip::current_device() != self->device) Py_RETURN_NONE;
  const int dtype = type == at::kHalf ? Q4_DTYPE_F16 : Q4_DTYPE_BF16;

  PyObject* plan = find(self->plans, (unsigned long long)M, dtype);  // (path, workspace bytes, decode configuration or None)
  if (plan == nullptr && !PyErr_Occurred() && owner != nullptr) {  // a row count not met before: the weight asks the library and keeps it
    PyObject* made = PyObject_CallMethod(owner, "plan", "li", M, dtype);
    if (made == nullptr) return nullptr;
    Py_DECREF(made);
    plan = find(self->plans, (unsigned long long)M, dtype);
  }
  if (plan == nullptr) return PyErr_Occurred() ? nullptr : Py_NewRef(Py_None);
  if (!PyTuple_Check(plan) || PyTuple_GET_SIZE(plan) != 3) Py_RETURN_NONE;
  long need = -1;
  if (!item(plan, 1, &need) || need < 0) Py_RETURN_NONE;
  PyObject* tuned = PyTuple_GET_ITEM(plan, 2);
  long cfg[4] = {0, 0, 0, 4};
  if (tuned != Py_None) {
    if (!PyTuple_Check(tuned)) Py_RETURN_NONE;
    for (int i = 0; i < 4; ++i) {
      if (i == 3 && PyTuple_GET_SIZE(tuned) == 3) break;
      if (!item(tuned, i, &cfg[i])) Py_RETURN_NONE;
    }
    need = std::max(need, (long)Q4_WORKSPACE_COUNTER_BYTES + cfg[2] * M * w.N * 4);
  }
  void* stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)self->device).stream();
  PyObject* ws_obj = find(g_workspaces, (unsigned long long)self->device, (long long)(intptr_t)stream);
  if (ws_obj == nullptr) return PyErr_Occurred() ? nullptr : Py_NewRef(Py_None);
  if (!THPVariable_Check(ws_obj)) Py_RETURN_NONE;
  const at::Tensor workspace = THPVariable_Unpack(ws_obj);  // (its own reference: the dict may change while the lock is released)
  if (workspace.numel() < need) Py_RETURN_NONE;

  c10::SmallVector<int64_t, 4> sizes(x.sizes().begin(), x.sizes().end());
  sizes.back() = w.N;
  at::Tensor y = at::empty(sizes, x.options());
  int rc;
  void* ws = workspace.data_ptr();
  void* yp = y.data_ptr();
  const size_t ws_bytes = (size_t)workspace.numel();
  Py_BEGIN_ALLOW_THREADS
  if (tuned != Py_None)
    rc = g_tuned(&w, xp, bias, yp, (int)M, dtype, ws, ws_bytes, (int)cfg[0], (int)cfg[1], (int)cfg[2], (int)cfg[3], stream);
  else
    rc = g_linear(&w, xp, bias, yp, (int)M, dtype, ws, ws_bytes, Q4_PATH_AUTO, stream);
  Py_END_ALLOW_THREADS
  if (rc < 0) {
    PyObject* ok = PyObject_CallFunction(g_check, "i", rc);
    if (ok == nullptr) return nullptr;
    Py_DECREF(ok);
  }
  return THPVariable_Wrap(std::move(y));
}

PyTypeObject CallType = {PyVarObject_HEAD_INIT(nullptr, 0)};

// handle(x, bias[, weight]) -> y, or None where the Python code has to do it.  With its PackedWeight at hand a row count that
// has no plan yet is planned and run here, the Python code behind it left out: 4096 x 4096, first call at one row 5.8 us on the host,
// 8.8 with it, 8.7 all in Python; first pass of one layer (4096 / 14336) at 301 rows 191, 195 and 195 us.
PyObject* call_vector(PyObject* self, PyObject* const* args, size_t nargsf, PyObject* names) {
  const Py_ssize_t count = PyVectorcall_NARGS(nargsf);
  if ((count != 2 && count != 3) || (names != nullptr && PyTuple_GET_SIZE(names) != 0)) {
    PyErr_SetString(PyExc_TypeError, "x, bias and, if at hand, the weight");
    return nullptr;
  }
  Py_INCREF(self);  // (the lock is released during the launch)
  PyObject* y;
  try {
    y = call((Call*)self, args[0], args[1], count == 3 ? args[2] : nullptr);
  } catch (...) {  // out of memory, say: no exception may leave a C function, and the Python code meets the cause again and raises
    y = PyErr_Occurred() ? nullptr : Py_NewRef(Py_None);
  }
  Py_DECREF(self);
  return y;
}

// handle(struct bytes, plans, device index, first regrouped row)
PyObject* py_handle(PyObject*, PyObject* args) {
  const char* bytes;
  Py_ssize_t size;
  PyObject* plans;
  int device;
  long first;
  if (!PyArg_ParseTuple(args, "y#O!il", &bytes, &size, &PyDict_Type, &plans, &device, &first)) return nullptr;
  if (size != (Py_ssize_t)sizeof(q4_weight)) {
    PyErr_SetString(PyExc_ValueError, "not a q4_weight");
    return nullptr;
  }
  Call* h = (Call*)CallType.tp_alloc(&CallType, 0);
  if (h == nullptr) return nullptr;
  h->vectorcall = call_vector;
  memcpy(&h->weight, bytes, sizeof(q4_weight));
  h->plans = Py_NewRef(plans);
  h->device = device;
  h->first_regrouped_row = first;
  return (PyObject*)h;
}

// bind(address of q4_linear_ex, address of q4_gemv_tuned, workspaces, check)
PyObject* py_bind(PyObject*, PyObject* args) {
  unsigned long long linear, tuned;
  PyObject *workspaces, *check;
  if (!PyArg_ParseTuple(args, "KKO!O", &linear, &tuned, &PyDict_Type, &workspaces, &check)) return nullptr;
  g_linear = (LinearFn)(uintptr_t)linear;
  g_tuned = (TunedFn)(uintptr_t)tuned;
  Py_XSETREF(g_workspaces, Py_NewRef(workspaces));
  Py_XSETREF(g_check, Py_NewRef(check));
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {{"handle", py_handle, METH_VARARGS, nullptr},
                          {"bind", py_bind, METH_VARARGS, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_q4call", nullptr, -1, kMethods};

}  // namespace

PyMODINIT_FUNC PyInit__q4call(void) {
  CallType.tp_name = "_q4call.Call";
  CallType.tp_basicsize = sizeof(Call);
  CallType.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL;
  CallType.tp_vectorcall_offset = offsetof(Call, vectorcall);
  CallType.tp_call = PyVectorcall_Call;
  CallType.tp_dealloc = call_dealloc;
  if (PyType_Ready(&CallType) < 0) return nullptr;
  PyObject* module = PyModule_Create(&kModule);
  // the torch whose classes are compiled in
  if (module != nullptr && PyModule_AddStringConstant(module, "torch_version", Q4_TORCH_VERSION) < 0) Py_CLEAR(module);
  return module;
}
