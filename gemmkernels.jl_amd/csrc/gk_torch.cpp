// The way of a call from Python to the library for callers that hold torch tensors: a module that does in C++ what the
// package's own Python does for a call that it has seen before.  It decides nothing: which launch a kind of operands gets is the Python side's,
// which registers it here (`remember`), and whatever is out of the ordinary -- a tensor subclass or a wrapper, a call not seen before, a workspace
// that is missing or too small, a stream that is being captured, a launch that the library refuses -- is handed back to it.
//
// What bounds a small product is the host: mul! at 51 x 17 x 23 in Float32 takes 3 us on the device and took 6.4 us a call, of
// which the HIP launch is 2.4, the checks of the library 1, ctypes 1 and reading three tensors and looking them up in a dictionary 1.8.  Through this module and
// gk_run 3.1 us a call; a plan 5.2 -> 3.3, matmul() on a diagonal A 7.3 -> 3.4, contract() 6.7 -> 4.3.
#include <Python.h>

#include <torch/csrc/autograd/python_variable.h>

#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <cstdint>
#include <cstring>
#include <string>
#include <unordered_map>

namespace {

typedef int (*MatmulFn)(const void*, const void*, const void*, const void*, void*, const void*, const void*, int32_t, void*);
typedef int (*SlicedFn)(const void*, const void*, const void*, const void*, void*, const void*, const void*, int32_t, void*, size_t, void*);
typedef int (*SplitFn)(const void*, const void*, const void*, const void*, void*, const void*, const void*, void*, size_t, void*);
typedef int (*CaptureFn)(void*, int32_t*, uint64_t*);
typedef int (*RunFn)(const void*, const void*, const void*, const void*, void*, void*);
RunFn g_run = nullptr;
MatmulFn g_matmul = nullptr;
SlicedFn g_sliced = nullptr;
SplitFn g_split = nullptr;
CaptureFn g_capture = nullptr;

enum : long { PLAIN = 0, SLICED = 1, SPLIT_K = 2, PREPARED = 3 };      // (PREPARED: `conf` is what gk_prepare gave)

// What tells one kind of call from another: as the Python side's key, without an address.
struct Kind {
  int64_t extent[6], stride[6];
  double alpha, beta;
  int8_t dtype[3], device;
  uint8_t transposed, aligned, pad[2];
  bool operator==(const Kind& o) const { return memcmp(this, &o, sizeof(Kind)) == 0; }
};
struct KindHash {
  size_t operator()(const Kind& k) const {
    uint64_t h = 1469598103934665603ull, w;
    static_assert(sizeof(Kind) % 8 == 0, "hashed in words");
    for (size_t i = 0; i < sizeof(Kind); i += 8) {
      memcpy(&w, (const char*)&k + i, 8);
      h = (h ^ w) * 1099511628211ull;
      h ^= h >> 29;
    }
    return (size_t)h;
  }
};
struct Launch {
  long form;
  const void* conf;
  const void* transforms;
  int32_t kernel;
  size_t workspace;
  PyObject* owner;          // keeps what conf and transforms point to
};
struct Workspace {
  void* address;
  size_t bytes;
  PyObject* owner;
};

// (touched with the GIL held only)
std::unordered_map<Kind, Launch, KindHash> g_launches;
std::unordered_map<uint64_t, Workspace> g_workspaces[16];     // per device: by stream
constexpr size_t kMaxLaunches = 1024;

// A plain matrix on a device; false: not for this module.
bool read_matrix(PyObject* obj, int which, Kind* kind, char** address) {
  if (!THPVariable_CheckExact(obj)) return false;
  const at::Tensor& t = THPVariable_Unpack(obj);
  const auto* impl = t.unsafeGetTensorImpl();
  if (impl->layout() != c10::kStrided || !impl->has_storage() || impl->dim() != 2 || !t.is_cuda() || impl->is_python_dispatch() ||
      impl->key_set().has(c10::DispatchKey::FuncTorchGradWrapper) || impl->key_set().has(c10::DispatchKey::FuncTorchBatched))
    return false;
  const auto sizes = impl->sizes(), strides = impl->strides();
  for (int i = 0; i < 2; ++i) { kind->extent[2 * which + i] = sizes[i]; kind->stride[2 * which + i] = strides[i]; }
  kind->dtype[which] = (int8_t)t.scalar_type();
  *address = (char*)t.data_ptr();
  kind->aligned |= (uint8_t)(((uintptr_t)*address % 16 == 0) << which);
  return true;
}

bool read_call(PyObject* const* args, Kind* kind, char** a, char** b, char** c) {
  memset(kind, 0, sizeof(*kind));
  if (!read_matrix(args[0], 0, kind, c) || !read_matrix(args[1], 1, kind, a) || !read_matrix(args[2], 2, kind, b)) return false;
  kind->transposed = (uint8_t)((args[3] == Py_True ? 1 : 0) | (args[4] == Py_True ? 2 : 0));
  kind->alpha = PyFloat_AS_DOUBLE(args[5]);
  kind->beta = PyFloat_AS_DOUBLE(args[6]);
  kind->device = (int8_t)c10::hip::current_device();
  return true;
}

// The buffer of eager launches on a stream of the current device; false where there is none of that size, or the stream is being captured.
bool find_workspace(void* stream, size_t bytes, Workspace* space) {
  int32_t capturing = 0;
  uint64_t id = 0;
  const int device = c10::hip::current_device();
  if (device >= 16 || g_capture(stream, &capturing, &id) != 0 || capturing != 0) return false;
  const auto found = g_workspaces[device].find((uint64_t)(uintptr_t)stream);
  if (found == g_workspaces[device].end() || found->second.bytes < bytes) return false;
  *space = found->second;
  return true;
}

PyObject* error_of(const std::exception& e) {
  PyErr_SetString(PyExc_RuntimeError, e.what());
  return nullptr;
}

// bind(gk_matmul, gk_matmul_sliced, gk_matmul_split_k, gk_stream_capture, gk_run): addresses of the library's entry points
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 5) { PyErr_SetString(PyExc_TypeError, "bind takes five addresses"); return nullptr; }
  g_matmul = (MatmulFn)PyLong_AsVoidPtr(args[0]);
  g_sliced = (SlicedFn)PyLong_AsVoidPtr(args[1]);
  g_split = (SplitFn)PyLong_AsVoidPtr(args[2]);
  g_capture = (CaptureFn)PyLong_AsVoidPtr(args[3]);
  g_run = (RunFn)PyLong_AsVoidPtr(args[4]);
  if (PyErr_Occurred()) return nullptr;
  Py_RETURN_NONE;
}

// remember(C, A, B, tA, tB, alpha, beta, form, conf, transforms, kernel, workspace, owner): the launch of a kind of call
PyObject* remember(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 13 || !PyFloat_CheckExact(args[5]) || !PyFloat_CheckExact(args[6])) { PyErr_SetString(PyExc_TypeError, "remember: wrong arguments"); return nullptr; }
  try {
    Kind kind;
    char *a, *b, *c;
    if (!read_call(args, &kind, &a, &b, &c)) Py_RETURN_FALSE;
    Launch launch{PyLong_AsLong(args[7]), PyLong_AsVoidPtr(args[8]), PyLong_AsVoidPtr(args[9]), (int32_t)PyLong_AsLong(args[10]), PyLong_AsSize_t(args[11]), args[12]};
    if (PyErr_Occurred()) return nullptr;
    if (g_launches.size() >= kMaxLaunches) {
      auto old = std::move(g_launches);
      g_launches.clear();
      for (auto& e : old) Py_DECREF(e.second.owner);
    }
    const auto put = g_launches.emplace(kind, launch);
    Py_INCREF(launch.owner);
    if (!put.second) {
      PyObject* before = put.first->second.owner;
      put.first->second = launch;
      Py_DECREF(before);
    }
    Py_RETURN_TRUE;
  } catch (const std::exception& e) { return error_of(e); }
}

// use_workspace(device, stream, address, bytes, owner): the buffer of eager launches on a stream
PyObject* use_workspace(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 5) { PyErr_SetString(PyExc_TypeError, "use_workspace: wrong arguments"); return nullptr; }
  const long device = PyLong_AsLong(args[0]);
  const uint64_t stream = (uint64_t)(uintptr_t)PyLong_AsVoidPtr(args[1]);
  const Workspace w{PyLong_AsVoidPtr(args[2]), PyLong_AsSize_t(args[3]), args[4]};
  if (PyErr_Occurred()) return nullptr;
  if (device < 0 || device >= 16) Py_RETURN_FALSE;
  try {
    auto put = g_workspaces[device].emplace(stream, w);
    Py_INCREF(w.owner);
    if (!put.second) {
      PyObject* before = put.first->second.owner;
      put.first->second = w;
      Py_DECREF(before);
    }
  } catch (const std::exception& e) { return error_of(e); }
  Py_RETURN_TRUE;
}

// mul(C, A, B, tA, tB, alpha, beta): True when the call is on its way, False when it is the Python side's
PyObject* mul(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 7 || !PyFloat_CheckExact(args[5]) || !PyFloat_CheckExact(args[6])) Py_RETURN_FALSE;
  try {
    Kind kind;
    char *a, *b, *c;
    if (g_launches.empty() || !read_call(args, &kind, &a, &b, &c)) Py_RETURN_FALSE;
    const auto hit = g_launches.find(kind);
    if (hit == g_launches.end()) Py_RETURN_FALSE;
    const Launch launch = hit->second;
    void* stream = (void*)c10::hip::getCurrentHIPStream().stream();
    Workspace space{nullptr, 0, nullptr};
    if (launch.workspace > 0 && !find_workspace(stream, launch.workspace, &space)) Py_RETURN_FALSE;
    // (other threads may forget the launch, or put a larger workspace in the place of this one, while the GIL is given up)
    Py_INCREF(launch.owner);
    Py_XINCREF(space.owner);
    int rc;
    Py_BEGIN_ALLOW_THREADS
    if (launch.form == PREPARED) rc = g_run(launch.conf, a, b, c, c, stream);
    else if (launch.form == PLAIN) rc = g_matmul(launch.conf, a, b, c, c, launch.transforms, nullptr, launch.kernel, stream);
    else if (launch.form == SLICED) rc = g_sliced(launch.conf, a, b, c, c, launch.transforms, nullptr, launch.kernel, space.address, space.bytes, stream);
    else rc = g_split(launch.conf, a, b, c, c, launch.transforms, nullptr, space.address, space.bytes, stream);
    Py_END_ALLOW_THREADS
    Py_XDECREF(space.owner);
    Py_DECREF(launch.owner);
    if (rc != 0) Py_RETURN_FALSE;           // (launched again over there, and refused with the library's message)
    Py_RETURN_TRUE;
  } catch (const std::exception&) {
    Py_RETURN_FALSE;
  }
}

// matmul(conf, a, b, c, d, transforms, epilogue, kernel, stream): gk_matmul on addresses; its status
PyObject* matmul(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 9) { PyErr_SetString(PyExc_TypeError, "matmul takes nine arguments"); return nullptr; }
  void* p[9];
  for (int i = 0; i < 9; ++i) p[i] = args[i] == Py_None ? nullptr : PyLong_AsVoidPtr(args[i]);
  if (PyErr_Occurred()) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_matmul(p[0], p[1], p[2], p[3], p[4], p[5], p[6], (int32_t)(intptr_t)p[7], p[8]);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// A plain strided tensor on a device, of any number of dimensions; false: not for this module.
bool read_tensor(PyObject* obj, const at::Tensor** tensor) {
  if (!THPVariable_CheckExact(obj)) return false;
  const at::Tensor& t = THPVariable_Unpack(obj);
  const auto* impl = t.unsafeGetTensorImpl();
  if (impl->layout() != c10::kStrided || !impl->has_storage() || !t.is_cuda() || impl->is_python_dispatch() ||
      impl->key_set().has(c10::DispatchKey::FuncTorchGradWrapper) || impl->key_set().has(c10::DispatchKey::FuncTorchBatched))
    return false;
  *tensor = &t;
  return true;
}

// leading_dims(forms, a, b, c, d): the leading dimensions of the operands of a configured launch as the Python side reads them, or None where it has to
// look for itself (an operand that it may refuse).  forms, one per operand: 0 no leading dimension, 1 a matrix, 2 interleaved, 3 planar complex numbers
PyObject* leading_dims(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 5 || !PyTuple_CheckExact(args[0]) || PyTuple_GET_SIZE(args[0]) != 4) Py_RETURN_NONE;
  try {
    long long ld[4] = {0, 0, 0, 0};
    for (int i = 0; i < 4; ++i) {
      const long form = PyLong_AsLong(PyTuple_GET_ITEM(args[0], i));
      PyObject* x = args[1 + i];
      if (x == Py_None || form == 0) continue;
      const at::Tensor* t;
      if (!read_tensor(x, &t)) Py_RETURN_NONE;
      const auto size = t->sizes(), stride = t->strides();
      if (form == 1 || (form == 2 && t->is_complex())) {
        if (size.size() != 2 || (size[0] > 1 && stride[0] != 1)) Py_RETURN_NONE;
        ld[i] = size[1] > 1 ? stride[1] : (size[0] > 1 ? size[0] : 1);
      } else if (form == 2) {
        if (size.size() != 3 || size[0] != 2 || stride[0] != 1 || (size[1] > 1 && stride[1] != 2)) Py_RETURN_NONE;
        ld[i] = size[2] > 1 ? stride[2] / 2 : (size[1] > 1 ? size[1] : 1);
      } else {
        if (size.size() != 3 || size[2] != 2 || (size[0] > 1 && stride[0] != 1) || stride[2] != stride[1] * size[1]) Py_RETURN_NONE;
        ld[i] = stride[1];
      }
    }
    return Py_BuildValue("(LLLL)", ld[0], ld[1], ld[2], ld[3]);
  } catch (const std::exception&) {
    Py_RETURN_NONE;
  }
}

// run(prepared, a, b, c, d): a prepared launch on torch's current stream; True when it is on its way, False when it is the Python side's
PyObject* run(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 5) Py_RETURN_FALSE;
  const void* prepared = PyLong_AsVoidPtr(args[0]);
  if (PyErr_Occurred()) return nullptr;
  try {
    void* p[4] = {nullptr, nullptr, nullptr, nullptr};
    for (int i = 0; i < 4; ++i) {
      if (args[1 + i] == Py_None) continue;
      const at::Tensor* t;
      if (!read_tensor(args[1 + i], &t)) Py_RETURN_FALSE;
      p[i] = t->data_ptr();
    }
    void* stream = (void*)c10::hip::getCurrentHIPStream().stream();
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = g_run(prepared, p[0], p[1], p[2], p[3], stream);
    Py_END_ALLOW_THREADS
    return PyBool_FromLong(rc == 0);
  } catch (const std::exception&) {
    Py_RETURN_FALSE;
  }
}

// run_at(prepared, a, b, c, d, stream): the same on addresses; its status
PyObject* run_at(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 6) { PyErr_SetString(PyExc_TypeError, "run_at takes six arguments"); return nullptr; }
  void* p[6];
  for (int i = 0; i < 6; ++i) p[i] = args[i] == Py_None ? nullptr : PyLong_AsVoidPtr(args[i]);
  if (PyErr_Occurred()) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_run(p[0], p[1], p[2], p[3], p[4], p[5]);
  Py_END_ALLOW_THREADS
  return PyLong_FromLong(rc);
}

// A launch in slices of K on the workspace of a stream, which other threads may replace by a larger one while the GIL is given up; -1: there is none.
int launch_sliced(const void* conf, void* const* p, const void* transforms, const void* epilogue, int32_t kernel, size_t bytes, void* stream) {
  Workspace space{nullptr, 0, nullptr};
  if (!find_workspace(stream, bytes, &space)) return -1;
  Py_INCREF(space.owner);
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = g_sliced(conf, p[0], p[1], p[2], p[3], transforms, epilogue, kernel, space.address, space.bytes, stream);
  Py_END_ALLOW_THREADS
  Py_DECREF(space.owner);
  return rc;
}

// sliced_at(conf, a, b, c, d, transforms, epilogue, kernel, workspace, stream): gk_matmul_sliced on addresses, with the workspace of that stream if it
// holds so many bytes; its status, or -1 where there is none and the Python side makes one
PyObject* sliced_at(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 10) { PyErr_SetString(PyExc_TypeError, "sliced_at takes ten arguments"); return nullptr; }
  void* p[10];
  for (int i = 0; i < 10; ++i) p[i] = args[i] == Py_None ? nullptr : PyLong_AsVoidPtr(args[i]);
  if (PyErr_Occurred()) return nullptr;
  try {
    return PyLong_FromLong(launch_sliced(p[0], p + 1, p[5], p[6], (int32_t)(intptr_t)p[7], (size_t)(uintptr_t)p[8], p[9]));
  } catch (const std::exception&) {
    return PyLong_FromLong(-1);
  }
}

// run_sliced(conf, kernel, workspace, a, b, c, d): the same without hooks on tensors at 16-byte boundaries and torch's current stream; True when it is on
// its way, False when it is the Python side's
PyObject* run_sliced(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 7) Py_RETURN_FALSE;
  const void* conf = PyLong_AsVoidPtr(args[0]);
  const long kernel = PyLong_AsLong(args[1]);
  const size_t bytes = PyLong_AsSize_t(args[2]);
  if (PyErr_Occurred()) return nullptr;
  try {
    void* p[4] = {nullptr, nullptr, nullptr, nullptr};
    for (int i = 0; i < 4; ++i) {
      if (args[3 + i] == Py_None) continue;
      const at::Tensor* t;
      if (!read_tensor(args[3 + i], &t)) Py_RETURN_FALSE;
      p[i] = t->data_ptr();
      if (((uintptr_t)p[i] & 15u) != 0) Py_RETURN_FALSE;
    }
    return PyBool_FromLong(launch_sliced(conf, p, nullptr, nullptr, (int32_t)kernel, bytes, (void*)c10::hip::getCurrentHIPStream().stream()) == 0);
  } catch (const std::exception&) {
    Py_RETURN_FALSE;
  }
}

// current_stream(): the handle of torch's current stream on the current device
PyObject* current_stream(PyObject*, PyObject*) {
  try {
    return PyLong_FromVoidPtr((void*)c10::hip::getCurrentHIPStream().stream());
  } catch (const std::exception& e) { return error_of(e); }
}

PyMethodDef g_methods[] = {{"bind", (PyCFunction)(void*)bind, METH_FASTCALL, nullptr},
                           {"remember", (PyCFunction)(void*)remember, METH_FASTCALL, nullptr},
                           {"use_workspace", (PyCFunction)(void*)use_workspace, METH_FASTCALL, nullptr},
                           {"mul", (PyCFunction)(void*)mul, METH_FASTCALL, nullptr},
                           {"matmul", (PyCFunction)(void*)matmul, METH_FASTCALL, nullptr},
                           {"leading_dims", (PyCFunction)(void*)leading_dims, METH_FASTCALL, nullptr},
                           {"run", (PyCFunction)(void*)run, METH_FASTCALL, nullptr},
                           {"run_at", (PyCFunction)(void*)run_at, METH_FASTCALL, nullptr},
                           {"sliced_at", (PyCFunction)(void*)sliced_at, METH_FASTCALL, nullptr},
                           {"run_sliced", (PyCFunction)(void*)run_sliced, METH_FASTCALL, nullptr},
                           {"current_stream", (PyCFunction)(void*)current_stream, METH_NOARGS, nullptr},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "gk_torch", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// The interpreter and the torch that this was built for: at::Tensor is read inline, so no other may load it (_native.py compares).
extern "C" const char gk_torch_built_for[] = GK_BUILT_FOR;

PyMODINIT_FUNC PyInit_gk_torch(void) { return PyModule_Create(&g_module); }
