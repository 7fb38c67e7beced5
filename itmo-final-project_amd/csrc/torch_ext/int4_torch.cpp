// int4_hip._int4_torch: the Python entry points' call path in native code for
// plain operands.
//
// A one-row product of a small linear takes 3.6 us on the GPU; checking five
// tensors, allocating the output and marshalling sixteen ctypes arguments in
// Python took 13 us of host time per call, so eager calls were bound by it.
// These functions do the same checks, allocation and C-ABI call (the addresses
// come from the library that _lib.py has loaded).  They return None, having done
// nothing, for everything else: other types, dtypes, strides or devices,
// invalid arguments, tensor subclasses, tracing, functorch transforms and
// dispatch or function modes.  The Python code then runs as it always did and
// raises the errors it always raised.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>

#include <array>
#include <map>
#include <vector>

#include "int4_hip.h"

namespace {

struct Api {
  decltype(&w4a16_gemm) gemm;
  decltype(&w4a16_workspace_bytes) workspace_bytes;
  decltype(&w4a16_gemm_grouped) gemm_grouped;
  decltype(&w4a16_grouped_workspace_bytes) grouped_workspace_bytes;
  decltype(&w4_quantize_grouped) quantize_grouped;
  decltype(&w4_quantize) quantize;
  decltype(&w4_dequantize) dequantize;
};
Api api{};
PyObject* py_workspace = nullptr;  // (device index, stream, bytes) -> (address, bytes)
PyObject* py_check = nullptr;      // raises for a nonzero status

// Nothing that has to see the individual operations is active on this thread.
bool quiet() {
  return api.gemm != nullptr && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         at::impl::PythonTorchFunctionTLS::stack_len() == 0 && !torch::jit::tracer::isTracing();
}

const c10::DispatchKeySet kWrapped =
    c10::DispatchKeySet({c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                         c10::DispatchKey::Python, c10::DispatchKey::Functionalize});

// The tensor behind a plain GPU tensor or parameter, else null.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != c10::kStrided || t.is_neg() || t.key_set().has_any(kWrapped))
    return nullptr;
  return &t;
}

int act_code(at::ScalarType t) {
  return t == at::kBFloat16 ? W4_DTYPE_BF16 : t == at::kHalf ? W4_DTYPE_FP16 : -1;
}

// Group size of a valid dense weight triple on `dev` for K activations, else 0.
int64_t weight_group(const at::Tensor* q, const at::Tensor* s, const at::Tensor* z, c10::Device dev, int64_t K) {
  if (!q || !s || !z || q->device() != dev || s->device() != dev || z->device() != dev) return 0;
  if (q->scalar_type() != at::kInt || q->dim() != 2 || s->scalar_type() != at::kHalf ||
      z->scalar_type() != at::kHalf || s->dim() != 2 || s->sizes() != z->sizes())
    return 0;
  if (q->size(0) * 8 != K || s->size(1) != q->size(1) || s->size(0) < 1) return 0;
  if (!q->is_contiguous() || !s->is_contiguous() || !z->is_contiguous()) return 0;
  const int64_t G = K / s->size(0);
  return G * s->size(0) == K && G >= 8 && (G & (G - 1)) == 0 ? G : 0;
}

bool current(c10::Device dev) { return c10::hip::current_device() == dev.index(); }

// The stream's workspace (kept and grown by the Python side); false: exception set.
bool workspace(c10::Device dev, void* stream, size_t bytes, void** ptr, size_t* size) {
  *ptr = nullptr;
  *size = 0;
  if (bytes == 0) return true;
  PyObject* r = PyObject_CallFunction(py_workspace, "iKK", (int)dev.index(), (unsigned long long)(uintptr_t)stream,
                                      (unsigned long long)bytes);
  if (!r) return false;
  unsigned long long p = 0, n = 0;
  const bool ok = PyArg_ParseTuple(r, "KK", &p, &n);
  Py_DECREF(r);
  *ptr = reinterpret_cast<void*>(p);
  *size = n;
  return ok;
}

// false: exception set.
bool check(int rc, const char* what) {
  if (rc == W4_OK) return true;
  PyObject* r = PyObject_CallFunction(py_check, "is", rc, what);
  Py_XDECREF(r);
  if (r) PyErr_Format(PyExc_RuntimeError, "%s failed (code %d)", what, rc);
  return false;
}

at::Tensor empty(c10::IntArrayRef sizes, at::ScalarType dtype, c10::Device dev) {
  return at::empty(sizes, at::TensorOptions().dtype(dtype).device(dev));
}

PyObject* matmul(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4 || !quiet()) Py_RETURN_NONE;
  const at::Tensor* x = plain(args[0]);
  if (!x || x->dim() < 1 || !x->is_contiguous()) Py_RETURN_NONE;
  const int dt = act_code(x->scalar_type());
  const int64_t K = x->size(-1);
  const c10::Device dev = x->device();
  if (dt < 0 || K < 8 || x->numel() == 0 || !current(dev)) Py_RETURN_NONE;
  const at::Tensor *q = plain(args[1]), *s = plain(args[2]), *z = plain(args[3]);
  const int64_t G = weight_group(q, s, z, dev, K);
  if (G == 0 || G > INT32_MAX) Py_RETURN_NONE;
  const int64_t M = x->numel() / K, N = q->size(1);
  if (N == 0) Py_RETURN_NONE;
  std::vector<int64_t> sizes(x->sizes().begin(), x->sizes().end());
  sizes.back() = N;
  at::Tensor y = empty(sizes, x->scalar_type(), dev);
  // a pure function of the shape (and the CU count of the one GPU type): memoised
  static std::map<std::array<int64_t, 4>, size_t> memo;
  const std::array<int64_t, 4> key{M, N, K, G};
  auto it = memo.find(key);
  if (it == memo.end()) {
    if (memo.size() > 4096) memo.clear();
    it = memo.emplace(key, api.workspace_bytes(M, N, K, (int)G)).first;
  }
  const size_t need = it->second;  // the callback below may let another thread at the memo
  void* const stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  void* ws;
  size_t ws_bytes;
  if (!workspace(dev, stream, need, &ws, &ws_bytes)) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.gemm(x->const_data_ptr(), dt, M, N, K, K, 1, static_cast<const int32_t*>(q->const_data_ptr()),
                static_cast<const uint16_t*>(s->const_data_ptr()), static_cast<const uint16_t*>(z->const_data_ptr()),
                (int)G, y.mutable_data_ptr(), N, ws, ws_bytes, stream);
  Py_END_ALLOW_THREADS
  if (!check(rc, "w4a16_gemm")) return nullptr;
  return THPVariable_Wrap(std::move(y));
  END_HANDLE_TH_ERRORS
}

// (xs, weights, out or None) -> list of outputs
PyObject* matmul_grouped(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 3 || !quiet()) Py_RETURN_NONE;
  auto seq = [](PyObject* o) { return PyList_CheckExact(o) || PyTuple_CheckExact(o); };
  if (!seq(args[0]) || !seq(args[1]) || (args[2] != Py_None && !seq(args[2]))) Py_RETURN_NONE;
  const Py_ssize_t count = PySequence_Fast_GET_SIZE(args[0]);
  if (count < 1 || count > W4_MAX_GROUPED || PySequence_Fast_GET_SIZE(args[1]) != count ||
      (args[2] != Py_None && PySequence_Fast_GET_SIZE(args[2]) < count))
    Py_RETURN_NONE;
  // Owned: the workspace callback and the launch let other threads run, which may
  // take the operands out of the caller's lists.
  struct Item {
    at::Tensor x, q, s, z, out;
    int64_t K, N, G;
  };
  std::array<Item, W4_MAX_GROUPED> it;
  int64_t M = 0;
  for (Py_ssize_t i = 0; i < count; ++i) {
    Item& a = it[i];
    const at::Tensor* x = plain(PySequence_Fast_GET_ITEM(args[0], i));
    if (!x || x->dim() < 1 || !x->is_contiguous() || x->numel() == 0 || ((uintptr_t)x->const_data_ptr() % 16) != 0)
      Py_RETURN_NONE;
    a.x = *x;
    a.K = x->size(-1);
    const int64_t rows = x->numel() / a.K;
    if (i == 0) M = rows;
    if (rows != M || x->scalar_type() != it[0].x.scalar_type() || x->device() != it[0].x.device()) Py_RETURN_NONE;
    PyObject* w = PySequence_Fast_GET_ITEM(args[1], i);
    if (!seq(w) || PySequence_Fast_GET_SIZE(w) != 3) Py_RETURN_NONE;
    const at::Tensor *q = plain(PySequence_Fast_GET_ITEM(w, 0)), *s = plain(PySequence_Fast_GET_ITEM(w, 1)),
                     *z = plain(PySequence_Fast_GET_ITEM(w, 2));
    a.G = weight_group(q, s, z, x->device(), a.K);
    if (a.G == 0 || a.G > INT32_MAX) Py_RETURN_NONE;
    a.q = *q;
    a.s = *s;
    a.z = *z;
    a.N = q->size(1);
    if (a.N == 0) Py_RETURN_NONE;
    if (args[2] != Py_None) {
      const at::Tensor* out = plain(PySequence_Fast_GET_ITEM(args[2], i));
      if (!out || x->dim() != 2 || out->dim() != 2 || out->size(0) != M || out->size(1) != a.N ||
          !out->is_contiguous() || out->scalar_type() != x->scalar_type() || out->device() != x->device())
        Py_RETURN_NONE;
      a.out = *out;
    }
  }
  const c10::Device dev = it[0].x.device();
  const int dt = act_code(it[0].x.scalar_type());
  if (dt < 0 || !current(dev)) Py_RETURN_NONE;
  w4a16_problem probs[W4_MAX_GROUPED];
  for (Py_ssize_t i = 0; i < count; ++i) {
    Item& a = it[i];
    if (!a.out.defined()) {
      std::vector<int64_t> sizes(a.x.sizes().begin(), a.x.sizes().end());
      sizes.back() = a.N;
      a.out = empty(sizes, a.x.scalar_type(), dev);
    }
    probs[i] = w4a16_problem{a.x.const_data_ptr(),
                             static_cast<const int32_t*>(a.q.const_data_ptr()),
                             static_cast<const uint16_t*>(a.s.const_data_ptr()),
                             static_cast<const uint16_t*>(a.z.const_data_ptr()),
                             a.out.mutable_data_ptr(),
                             a.N,
                             a.K,
                             (int32_t)a.G,
                             0};
  }
  void* const stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  void* ws;
  size_t ws_bytes;
  if (!workspace(dev, stream, api.grouped_workspace_bytes(probs, (int)count, M), &ws, &ws_bytes)) return nullptr;
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.gemm_grouped(probs, (int)count, dt, M, ws, ws_bytes, stream);
  Py_END_ALLOW_THREADS
  if (!check(rc, "w4a16_gemm_grouped")) return nullptr;
  PyObject* list = PyList_New(count);
  if (!list) return nullptr;
  for (Py_ssize_t i = 0; i < count; ++i) PyList_SET_ITEM(list, i, THPVariable_Wrap(std::move(it[i].out)));
  return list;
  END_HANDLE_TH_ERRORS
}

struct Quant {
  const at::Tensor* w;
  int64_t N, K, G;
  at::Tensor q, s, z;
};

// A weight that quantize_int4 accepts, as it is (any strides).
bool quant_item(PyObject* o, int64_t group, Quant* a) {
  a->w = plain(o);
  if (!a->w || a->w->dim() != 2 || a->w->numel() == 0 || act_code(a->w->scalar_type()) < 0) return false;
  a->N = a->w->size(0);
  a->K = a->w->size(1);
  a->G = group == -1 ? a->K : group;
  return a->G > 0 && a->K % a->G == 0 && a->G % 8 == 0 && (a->G & (a->G - 1)) == 0;
}

void quant_outputs(Quant* a) {
  const c10::Device dev = a->w->device();
  a->q = empty({a->K / 8, a->N}, at::kInt, dev);
  a->s = empty({a->K / a->G, a->N}, at::kHalf, dev);
  a->z = empty({a->K / a->G, a->N}, at::kHalf, dev);
}

PyObject* quant_triple(Quant* a) {
  return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(a->q)), THPVariable_Wrap(std::move(a->s)),
                       THPVariable_Wrap(std::move(a->z)));
}

// The group size an int names, or 0 (never valid) if it is no int or does not fit 32 bits.
int64_t group_arg(PyObject* o) {
  if (!PyLong_CheckExact(o)) return 0;
  int overflow = 0;
  const long long g = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow || g < -1 || g > INT32_MAX ? 0 : g;
}

PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !quiet()) Py_RETURN_NONE;
  Quant a;
  if (!quant_item(args[0], group_arg(args[1]), &a) || !current(a.w->device())) Py_RETURN_NONE;
  if (a.G > INT32_MAX) Py_RETURN_NONE;
  quant_outputs(&a);
  void* const stream = c10::hip::getCurrentHIPStream(a.w->device().index()).stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.quantize(a.w->const_data_ptr(), act_code(a.w->scalar_type()), a.N, a.K, a.w->stride(0), a.w->stride(1),
                    (int)a.G, static_cast<int32_t*>(a.q.mutable_data_ptr()),
                    static_cast<uint16_t*>(a.s.mutable_data_ptr()), static_cast<uint16_t*>(a.z.mutable_data_ptr()),
                    stream);
  Py_END_ALLOW_THREADS
  if (!check(rc, "w4_quantize")) return nullptr;
  return quant_triple(&a);
  END_HANDLE_TH_ERRORS
}

PyObject* quantize_grouped(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 2 || !quiet() || !PyList_CheckExact(args[0])) Py_RETURN_NONE;
  const int64_t group = group_arg(args[1]);
  const Py_ssize_t count = PyList_GET_SIZE(args[0]);
  if (count < 1 || count > W4_MAX_GROUPED) Py_RETURN_NONE;
  std::array<Quant, W4_MAX_GROUPED> it;
  for (Py_ssize_t i = 0; i < count; ++i)
    if (!quant_item(PyList_GET_ITEM(args[0], i), group, &it[i]) || it[i].G > INT32_MAX ||
        it[i].w->scalar_type() != it[0].w->scalar_type() || it[i].w->device() != it[0].w->device())
      Py_RETURN_NONE;
  const c10::Device dev = it[0].w->device();
  if (!current(dev)) Py_RETURN_NONE;
  w4_quantize_problem probs[W4_MAX_GROUPED];
  for (Py_ssize_t i = 0; i < count; ++i) {
    Quant& a = it[i];
    quant_outputs(&a);
    probs[i] = w4_quantize_problem{a.w->const_data_ptr(),
                                   static_cast<int32_t*>(a.q.mutable_data_ptr()),
                                   static_cast<uint16_t*>(a.s.mutable_data_ptr()),
                                   static_cast<uint16_t*>(a.z.mutable_data_ptr()),
                                   a.N,
                                   a.K,
                                   a.w->stride(0),
                                   a.w->stride(1),
                                   (int32_t)group,
                                   0};
  }
  void* const stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.quantize_grouped(probs, (int)count, act_code(it[0].w->scalar_type()), stream);
  Py_END_ALLOW_THREADS
  if (!check(rc, "w4_quantize_grouped")) return nullptr;
  PyObject* list = PyList_New(count);
  if (!list) return nullptr;
  for (Py_ssize_t i = 0; i < count; ++i) {
    PyObject* t = quant_triple(&it[i]);
    if (!t) {
      Py_DECREF(list);
      return nullptr;
    }
    PyList_SET_ITEM(list, i, t);
  }
  return list;
  END_HANDLE_TH_ERRORS
}

PyObject* dequantize(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 4 || !quiet() || !THPDtype_Check(args[3])) Py_RETURN_NONE;
  const at::Tensor *q = plain(args[0]), *s = plain(args[1]), *z = plain(args[2]);
  const at::ScalarType dtype = reinterpret_cast<THPDtype*>(args[3])->scalar_type;
  const int dt = dtype == at::kFloat ? W4_DTYPE_FP32 : act_code(dtype);
  if (!q || dt < 0 || q->dim() != 2 || !current(q->device())) Py_RETURN_NONE;
  const int64_t K = q->size(0) * 8, N = q->size(1), G = weight_group(q, s, z, q->device(), K);
  if (G == 0 || G > INT32_MAX || N == 0) Py_RETURN_NONE;
  at::Tensor out = empty({N, K}, dtype, q->device());
  void* const stream = c10::hip::getCurrentHIPStream(q->device().index()).stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = api.dequantize(static_cast<const int32_t*>(q->const_data_ptr()),
                      static_cast<const uint16_t*>(s->const_data_ptr()),
                      static_cast<const uint16_t*>(z->const_data_ptr()), N, K, (int)G, dt, out.mutable_data_ptr(),
                      stream);
  Py_END_ALLOW_THREADS
  if (!check(rc, "w4_dequantize")) return nullptr;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// (addresses of the C-ABI functions in Api's order, workspace, check)
PyObject* init(PyObject*, PyObject* args) {
  unsigned long long p[7];
  PyObject *w, *c;
  if (!PyArg_ParseTuple(args, "(KKKKKKK)OO", &p[0], &p[1], &p[2], &p[3], &p[4], &p[5], &p[6], &w, &c)) return nullptr;
  Py_INCREF(w);
  Py_INCREF(c);
  Py_XDECREF(py_workspace);
  Py_XDECREF(py_check);
  py_workspace = w;
  py_check = c;
  api.workspace_bytes = reinterpret_cast<decltype(api.workspace_bytes)>(p[1]);
  api.gemm_grouped = reinterpret_cast<decltype(api.gemm_grouped)>(p[2]);
  api.grouped_workspace_bytes = reinterpret_cast<decltype(api.grouped_workspace_bytes)>(p[3]);
  api.quantize_grouped = reinterpret_cast<decltype(api.quantize_grouped)>(p[4]);
  api.quantize = reinterpret_cast<decltype(api.quantize)>(p[5]);
  api.dequantize = reinterpret_cast<decltype(api.dequantize)>(p[6]);
  api.gemm = reinterpret_cast<decltype(api.gemm)>(p[0]);
  Py_RETURN_NONE;
}

#define W4_FAST(f) {#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"init", init, METH_VARARGS, nullptr},
                         W4_FAST(matmul),
                         W4_FAST(matmul_grouped),
                         W4_FAST(quantize),
                         W4_FAST(quantize_grouped),
                         W4_FAST(dequantize),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_int4_torch", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__int4_torch() {
  PyObject* m = PyModule_Create(&module);
  // the torch whose headers this was built from: tensors are read through them
  if (m && PyModule_AddStringConstant(m, "torch_version", W4_TORCH_VERSION) != 0) Py_CLEAR(m);
  return m;
}
