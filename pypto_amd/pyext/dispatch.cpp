// The argument side of a program call in native code: torch tensors -> ChipTensor descriptors -> pto_hip_run.
//
// A registered program called on resident tensors is what a serving loop does for every step and layer
// (RegistrationHandle.__call__, python/pypto/runtime/worker.py:675-773), and for small calls the time is the issue of
// the call: descriptors built field by field through ctypes take about a microsecond a tensor, longer than the launches.
// Per call from Python, us: paged attention of one sequence (7 tensors) 16.6 -> 8.0, decoder layer (20 tensors) 57 -> 32
//
// Only the plain case is taken: exact torch tensors (or parameters), contiguous, on the GPU - or on the CPU where the signature
// says that the launcher reads the tensor on the host.  For anything else `run` returns None and launches nothing, and the
// caller goes through its general path, which stages host tensors and words the errors.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstring>
#include <cstdint>
#include <limits>

#include "pto_hip.h"

namespace {

typedef int (*RunFn)(int, const PtoHipChipTensor*, int, const uint64_t*, int, void*);
constexpr int kMaxArgs = 64;

// DataType code of a torch type, 0 where the target has none (as runtime.py's table)
uint32_t dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kChar: return PTO_HIP_INT8;
    case at::kInt: return PTO_HIP_INT32;
    case at::kLong: return PTO_HIP_INT64;
    case at::kFloat8_e4m3fn: return PTO_HIP_FP8E4M3FN;
    case at::kHalf: return PTO_HIP_FP16;
    case at::kFloat: return PTO_HIP_FP32;
    case at::kBFloat16: return PTO_HIP_BF16;
    default: return 0;
  }
}

// False: not the plain case.
bool describe(PyObject* o, bool host_ok, PtoHipChipTensor* d) {
  PyTypeObject* type = Py_TYPE(o);
  if (type != reinterpret_cast<PyTypeObject*>(THPVariableClass) && type != reinterpret_cast<PyTypeObject*>(ParameterClass)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (t.layout() != at::kStrided || !t.is_contiguous() || t.dim() > PTO_HIP_MAX_DIMS) return false;
  const bool cuda = t.is_cuda();
  if (!cuda && !(host_ok && t.is_cpu())) return false;
  const uint32_t code = dtype_code(t.scalar_type());
  if (!code) return false;
  uint64_t addr = reinterpret_cast<uint64_t>(t.data_ptr());
  if (cuda && !addr) addr = 1;  // an empty tensor
  *d = PtoHipChipTensor{};
  d->buffer.addr = addr;
  d->buffer.size = (uint64_t)t.numel() * (uint64_t)t.element_size();
  const auto sizes = t.sizes();
  for (size_t i = 0; i < sizes.size(); ++i) d->shapes[i] = (uint32_t)sizes[i];
  d->ndims = (uint32_t)sizes.size();
  d->dtype = code;
  return true;
}

// Raw 64-bit pattern of a scalar argument; floats travel as fp32 bits (runner.py:948-953).
bool scalar_bits(PyObject* o, uint64_t* out) {
  if (PyLong_Check(o)) {  // bool among them
    *out = (uint64_t)PyLong_AsUnsignedLongLongMask(o);
    return true;
  }
  if (!PyFloat_Check(o)) return false;
  const double v = PyFloat_AS_DOUBLE(o);
  if (std::isfinite(v) && std::fabs(v) > (double)std::numeric_limits<float>::max()) return false;  // an error of the general path
  const float f = (float)v;
  uint32_t bits;
  std::memcpy(&bits, &f, 4);
  *out = bits;
  return true;
}

// run(address of pto_hip_run, callable id, host flags (a byte per tensor of the signature), optional tensors, scalars, args, stream)
// -> status, or None where the call is not the plain case
PyObject* run(PyObject*, PyObject* const* argv, Py_ssize_t argc) {
  if (argc != 7 || !PyLong_Check(argv[0]) || !PyLong_Check(argv[1]) || !PyBytes_Check(argv[2]) || !PyLong_Check(argv[3]) ||
      !PyLong_Check(argv[4]) || !PyTuple_Check(argv[5])) {
    PyErr_SetString(PyExc_TypeError, "run(run_address, cid, host_flags, optional, n_scalars, args, stream)");
    return nullptr;
  }
  const RunFn fn = reinterpret_cast<RunFn>(PyLong_AsVoidPtr(argv[0]));
  const long cid = PyLong_AsLong(argv[1]), optional = PyLong_AsLong(argv[3]), n_scalars = PyLong_AsLong(argv[4]);
  const Py_ssize_t most = PyBytes_GET_SIZE(argv[2]), n_args = PyTuple_GET_SIZE(argv[5]), n_tensors = n_args - n_scalars;
  const char* host = PyBytes_AS_STRING(argv[2]);
  void* stream = nullptr;
  if (PyLong_Check(argv[6])) stream = PyLong_AsVoidPtr(argv[6]);
  else if (argv[6] != Py_None) Py_RETURN_NONE;
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  if (!fn || n_scalars < 0 || n_tensors > most || n_tensors < most - optional || n_tensors < 0 || n_args > kMaxArgs) Py_RETURN_NONE;
  PtoHipChipTensor tensors[kMaxArgs];
  uint64_t scalars[kMaxArgs];
  try {
    for (Py_ssize_t i = 0; i < n_tensors; ++i)
      if (!describe(PyTuple_GET_ITEM(argv[5], i), host[i] != 0, &tensors[i])) Py_RETURN_NONE;
  } catch (...) {  // a tensor without memory of its own (a transform's or a mode's): the general path words the error
    Py_RETURN_NONE;
  }
  for (Py_ssize_t i = 0; i < n_scalars; ++i)
    if (!scalar_bits(PyTuple_GET_ITEM(argv[5], n_tensors + i), &scalars[i])) Py_RETURN_NONE;
  int status;
  Py_BEGIN_ALLOW_THREADS  // the library's dispatch lock may be held by a thread that waits for the interpreter
  status = fn((int)cid, tensors, (int)n_tensors, scalars, (int)n_scalars, stream);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(status);
}

PyMethodDef methods[] = {
    {"run", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(run)), METH_FASTCALL, "pto_hip_run on torch tensors; None where not the plain case"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_dispatch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__dispatch(void) { return PyModule_Create(&module); }
