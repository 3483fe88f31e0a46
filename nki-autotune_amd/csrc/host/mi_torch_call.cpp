// mi_torch_call.cpp -- the default call of every kernel_library operation,
// from torch tensors to the C ABI launch, in native code.
//
// A kernel_library call without a config checks its operands, finds the
// shape's config, allocates the output, reads the current stream and calls
// the C ABI.  In Python that takes 11.4 us of host time (10.9 with the
// output given; 13.7 for a split-K call's two launches), more than most
// small kernels run (3 to 8 us), so back-to-back calls of them ran at the
// host's pace.  call() below does the same steps for the ordinary call in
// 4.3 us (3.9; 7.4), of which the launch itself is 2.8.  It makes no
// decision of its own: whatever it does not
// recognise (another type, layout, device, shape, mode or an unknown config)
// it leaves undone and returns None, and the Python body of the operation
// runs, which checks everything, raises what is to be raised, and hands the
// shape's config to remember() for the next call.
//
// Nothing is kept between calls but the shapes' configs: no pointer, tensor
// or identity.  The GIL is held throughout except around the launch, as
// ctypes does, so the table needs no lock; nothing shared is read there.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <Python.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <climits>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <string>
#include <unordered_map>

#include "../../../include/mi_kernels.h"

namespace {

// What a call computes; the first argument of call() and remember().
enum Kind { kLhsTBf16 = 0, kLhsTF32 = 1, kRms = 2, kLhs = 3, kRmsNoGamma = 4 };

using MatmulFn = int (*)(const void*, const void*, void*, int, int, int, const mi_tile_cfg*, void*);
using RmsFn = int (*)(const void*, const void*, const void*, void*, int, int, int, float, const mi_tile_cfg*, void*);

struct Library {
  MatmulFn lhsT_bf16 = nullptr, lhsT_f32 = nullptr, lhs = nullptr;
  RmsFn rms = nullptr;
  std::string env;             // MI_KERNELS_LIB when the library was bound ("" if unset)
  PyObject* check_rc = nullptr;  // raises the error of a return code
} g_lib;

struct Shape {
  int64_t kind, M, N, K;
  bool operator==(const Shape& o) const { return kind == o.kind && M == o.M && N == o.N && K == o.K; }
};
struct ShapeHash {
  size_t operator()(const Shape& s) const {
    uint64_t h = (uint64_t)s.kind;
    for (const uint64_t v : {(uint64_t)s.M, (uint64_t)s.N, (uint64_t)s.K}) h = (h ^ v) * 0x9E3779B97F4A7C15ull, h ^= h >> 29;
    return (size_t)h;
  }
};
constexpr size_t kMaxShapes = 1 << 16;
std::unordered_map<Shape, mi_tile_cfg, ShapeHash> g_configs;

// A dense tensor on a HIP device that nothing intercepts: an exact Tensor or
// Parameter whose dispatch keys are the device's own, autograd's and
// autocast's (no conjugate or negative view, no functorch, Python or sparse
// key).
const at::Tensor* plain(PyObject* o, at::ScalarType dtype) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  static const uint64_t allowed =
      (c10::DispatchKeySet(c10::DispatchKey::CUDA) | c10::DispatchKeySet(c10::DispatchKey::AutogradCUDA) |
       c10::DispatchKeySet(c10::DispatchKey::ADInplaceOrView) | c10::autocast_dispatch_keyset).raw_repr();
  if (!t.defined() || (t.key_set().raw_repr() & ~allowed) != 0) return nullptr;
  if (!t.is_cuda() || t.scalar_type() != dtype || !t.is_contiguous()) return nullptr;
  return &t;
}

// No mode or transform is active on this thread.
bool no_mode() {
  if (at::impl::torch_function_mode_enabled() || c10::impl::dispatch_mode_enabled()) return false;
  static const uint64_t allowed = (c10::default_included_set | c10::autocast_dispatch_keyset).raw_repr();
  return (c10::impl::tls_local_dispatch_key_set().included_.raw_repr() & ~allowed) == 0;
}

bool disjoint(const at::Tensor& out, const at::Tensor& in) {
  const uintptr_t o = (uintptr_t)out.data_ptr(), i = (uintptr_t)in.data_ptr();
  return o + out.nbytes() <= i || i + in.nbytes() <= o;
}

// call(kind, a, b, gamma | None, eps, out | None): the output tensor, or
// None when the Python body has to run.  kind: 0 (bf16 or fp32 lhsT.rhs),
// 2 (rmsnorm_matmul, gamma or None), 3 (lhs.rhs).
PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 6) {
    PyErr_SetString(PyExc_TypeError, "call takes 6 arguments");
    return nullptr;
  }
  HANDLE_TH_ERRORS
  {
    if (!g_lib.check_rc || !no_mode()) Py_RETURN_NONE;
    int64_t kind = PyLong_AsLong(args[0]);
    PyObject *pa = args[1], *pb = args[2], *pg = args[3], *po = args[5];
    if (!THPVariable_CheckExact(pa)) Py_RETURN_NONE;
    const at::ScalarType dtype = THPVariable_Unpack(pa).scalar_type();
    if (dtype == at::kFloat && kind == kLhsTBf16) kind = kLhsTF32;
    else if (dtype != at::kBFloat16) Py_RETURN_NONE;
    const at::Tensor *a = plain(pa, dtype), *b = plain(pb, dtype);
    if (!a || !b || a->dim() != 2 || b->dim() != 2) Py_RETURN_NONE;
    const bool k_first = kind == kLhsTBf16 || kind == kLhsTF32;
    const int64_t M = a->size(k_first ? 1 : 0), K = a->size(k_first ? 0 : 1), N = b->size(1);
    if (b->size(0) != K || M < 1 || N < 1 || K < 1 || M > INT_MAX || N > INT_MAX || K > INT_MAX) Py_RETURN_NONE;
    const c10::Device dev = a->device();
    if (b->device() != dev) Py_RETURN_NONE;
    const at::Tensor* g = nullptr;
    float eps = 0.0f;
    if (kind == kRms) {
      const double e = PyFloat_AsDouble(args[4]);
      if (e == -1.0 && PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
      }
      eps = (float)e;
      if (pg == Py_None) {
        kind = kRmsNoGamma;
      } else {
        g = plain(pg, dtype);
        if (!g || g->dim() != 1 || g->size(0) != K || g->device() != dev) Py_RETURN_NONE;
      }
    }
    const at::Tensor* given = nullptr;
    if (po != Py_None) {
      given = plain(po, dtype);
      if (!given || given->dim() != 2 || given->size(0) != M || given->size(1) != N || given->device() != dev ||
          !disjoint(*given, *a) || !disjoint(*given, *b) || (g && !disjoint(*given, *g)))
        Py_RETURN_NONE;
    }
    const auto it = g_configs.find(Shape{kind, M, N, K});
    if (it == g_configs.end()) Py_RETURN_NONE;
    const mi_tile_cfg cfg = it->second;
    const char* env = std::getenv("MI_KERNELS_LIB");
    if (g_lib.env != (env ? env : "")) Py_RETURN_NONE;

    const c10::OptionalDeviceGuard guard(dev);
    at::Tensor made;
    if (!given) {
      made = at::empty({M, N}, a->options().requires_grad(false));
      given = &made;
    }
    void* stream = (void*)c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(dev.index()).stream();
    const void *ap = a->data_ptr(), *bp = b->data_ptr(), *gp = g ? g->data_ptr() : nullptr;
    void* op = given->data_ptr();
    // The entry point is read before the GIL is given up: another thread's
    // bind() may then put another library's in its place.
    const MatmulFn mm = kind == kLhs ? g_lib.lhs : kind == kLhsTF32 ? g_lib.lhsT_f32 : g_lib.lhsT_bf16;
    const RmsFn rms = g_lib.rms;
    int rc;
    Py_BEGIN_ALLOW_THREADS
    if (kind == kRms || kind == kRmsNoGamma) rc = rms(ap, gp, bp, op, (int)M, (int)N, (int)K, eps, &cfg, stream);
    else rc = mm(ap, bp, op, (int)M, (int)N, (int)K, &cfg, stream);
    Py_END_ALLOW_THREADS
    if (rc != 0) {
      static const char* const names[] = {"matmul_lhsT_rhs", "matmul_lhsT_rhs_f32", "rmsnorm_matmul", "matmul_lhs_rhs",
                                          "rmsnorm_matmul"};
      PyObject* r = PyObject_CallFunction(g_lib.check_rc, "is", rc, names[kind]);
      if (r) {  // check_rc raises for every code but 0
        Py_DECREF(r);
        PyErr_SetString(PyExc_RuntimeError, names[kind]);
      }
      return nullptr;
    }
    if (po != Py_None) {
      Py_INCREF(po);
      return po;
    }
    return THPVariable_Wrap(std::move(made));
  }
  END_HANDLE_TH_ERRORS
}

// bind(env, lhsT_bf16, lhsT_f32, rms, lhs, check_rc): the library's entry
// points (addresses), the value of MI_KERNELS_LIB they were found with, and
// the function that raises a return code's error.  Another library than the
// bound one drops every shape's config.
PyObject* bind(PyObject*, PyObject* args) {
  const char* env;
  unsigned long long p0, p1, p2, p3;
  PyObject* check_rc;
  if (!PyArg_ParseTuple(args, "sKKKKO", &env, &p0, &p1, &p2, &p3, &check_rc)) return nullptr;
  const MatmulFn lhsT_bf16 = (MatmulFn)(uintptr_t)p0, lhsT_f32 = (MatmulFn)(uintptr_t)p1, lhs = (MatmulFn)(uintptr_t)p3;
  const RmsFn rms = (RmsFn)(uintptr_t)p2;
  // The shapes' configs are the bound library's own.
  if (g_lib.env != env || g_lib.lhsT_bf16 != lhsT_bf16 || g_lib.lhsT_f32 != lhsT_f32 || g_lib.rms != rms ||
      g_lib.lhs != lhs)
    g_configs.clear();
  g_lib.env = env;
  g_lib.lhsT_bf16 = lhsT_bf16;
  g_lib.lhsT_f32 = lhsT_f32;
  g_lib.rms = rms;
  g_lib.lhs = lhs;
  Py_INCREF(check_rc);
  PyObject* const before = g_lib.check_rc;
  g_lib.check_rc = check_rc;
  Py_XDECREF(before);
  Py_RETURN_NONE;
}

// remember(kind, M, N, K, block_m, block_n, block_k, waves, lds_stages, split_k, group_m, variant)
PyObject* remember(PyObject*, PyObject* args) {
  long long kind, M, N, K;
  mi_tile_cfg c;
  if (!PyArg_ParseTuple(args, "LLLLiiiiiiii", &kind, &M, &N, &K, &c.block_m, &c.block_n, &c.block_k, &c.waves,
                        &c.lds_stages, &c.split_k, &c.group_m, &c.variant))
    return nullptr;
  if (g_configs.size() >= kMaxShapes) g_configs.clear();
  g_configs[Shape{kind, M, N, K}] = c;
  Py_RETURN_NONE;
}

// knows(kind, M, N, K): whether remember() has this shape's config for the
// library in use.  The Python body asks after each call it runs, so that the
// calls it always runs (a mode, a subclass, a view) bind and remember once.
PyObject* knows(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 4) {
    PyErr_SetString(PyExc_TypeError, "knows takes 4 arguments");
    return nullptr;
  }
  long long v[4];
  for (int i = 0; i < 4; ++i) {
    v[i] = PyLong_AsLongLong(args[i]);
    if (v[i] == -1 && PyErr_Occurred()) return nullptr;
  }
  const char* env = std::getenv("MI_KERNELS_LIB");
  return PyBool_FromLong(g_lib.check_rc && g_lib.env == (env ? env : "") && g_configs.count(Shape{v[0], v[1], v[2], v[3]}));
}

// forget(): drop every shape's config (the tuned table changed).
PyObject* forget(PyObject*, PyObject*) {
  g_configs.clear();
  Py_RETURN_NONE;
}

PyMethodDef kMethods[] = {{"call", (PyCFunction)(void (*)(void))call, METH_FASTCALL, nullptr},
                          {"bind", bind, METH_VARARGS, nullptr},
                          {"remember", remember, METH_VARARGS, nullptr},
                          {"knows", (PyCFunction)(void (*)(void))knows, METH_FASTCALL, nullptr},
                          {"forget", forget, METH_NOARGS, nullptr},
                          {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_torch_call", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// Built against one torch's headers, so it loads beside that torch only (the
// Python body then serves the calls).
PyMODINIT_FUNC PyInit__torch_call() {
  PyObject* torch = PyImport_ImportModule("torch");
  if (!torch) return nullptr;
  PyObject* version = PyObject_GetAttrString(torch, "__version__");
  Py_DECREF(torch);
  if (!version) return nullptr;
  const char* now = PyUnicode_AsUTF8(version);
  const size_t n = std::strlen(TORCH_VERSION);
  const bool same = now && std::strncmp(now, TORCH_VERSION, n) == 0 && (now[n] == '\0' || now[n] == '+');
  if (now && !same) PyErr_Format(PyExc_ImportError, "built for torch %s, found %s", TORCH_VERSION, now);
  Py_DECREF(version);
  return same ? PyModule_Create(&kModule) : nullptr;
}
