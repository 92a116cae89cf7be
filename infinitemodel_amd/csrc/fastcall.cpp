// Native host path of the eager fused calls: one CPython call that checks the operands, allocates the output
// and calls libimq, for the plain case -- exact torch.Tensor operands, one device that is current, dense
// rows, matching shapes and dtypes, no dispatch or function mode, functional transform or tracer active.
// Anything else returns None and the Python path runs as before (with its conversions, its checks and
// its errors), so nothing is accepted or refused here that it would not. Host time per call is what bounds
// a decode step that is not replayed from a graph: a 1 x 4096 -> 4096 linear took 14.4 us through the Python
// checks and ctypes for 4 us of kernel.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include <map>

#include "../../include/imq.h"

namespace {

// libimq's entry points, by address (the library is loaded and checked by _lib.py).
struct Api {
  decltype(&imq_linear_w4) w4 = nullptr, w4t = nullptr, w2 = nullptr, w2t = nullptr;
  decltype(&imq_linear_w8) w8 = nullptr, w8t = nullptr;
  decltype(&imq_linear_w4_workspace_bytes) w4_ws = nullptr;
  decltype(&imq_linear_workspace_bytes) ws = nullptr;
  decltype(&imq_moe_experts_w4_ex) moe = nullptr;
  decltype(&imq_moe_workspace_bytes) moe_ws = nullptr;
} api;
PyObject* scratch_fn = nullptr;   // ops._scratch_ptr(device index, bytes) -> (pointer, bytes, lock)

struct Scratch {
  int64_t ptr = 0, bytes = 0;
  PyObject* lock = nullptr;       // owned; one per (device, stream), ops.py's users hold the same
};
// The workspaces ops.py holds for the life of the process, one per (device, stream); read and written
// with the GIL held.
std::map<std::pair<int, void*>, Scratch> scratches;

// At least `need` bytes of ops.py's workspace for this device and its current stream. false: a Python
// error is set.
bool scratch(int dev, void* stream, int64_t need, Scratch* out) {
  if (need <= 0) return true;
  Scratch& s = scratches[{dev, stream}];
  if (s.bytes < need) {
    PyObject* r = PyObject_CallFunction(scratch_fn, "iL", dev, (long long)need);
    if (r == nullptr) return false;
    long long p = 0, b = 0;
    PyObject* lock = nullptr;
    const bool ok = PyArg_ParseTuple(r, "LLO", &p, &b, &lock) != 0;
    if (ok) {
      if (s.lock == nullptr) s.lock = Py_NewRef(lock);   // the key's lock never changes
      s.ptr = p;
      s.bytes = b;
    }
    Py_DECREF(r);
    if (!ok) return false;
  }
  *out = s;
  return true;
}

// Holds a workspace's lock while a call's launches go out: the GIL is released around them, and the kernel
// that writes the partials and the one that sums them must not be parted by another thread's call on the
// same stream. Taken and released with the GIL held (a waiting acquire lets go of it).
class Held {
 public:
  // false: a Python error is set
  bool take(const Scratch& s) {
    if (s.lock == nullptr) return true;
    PyObject* r = PyObject_CallMethod(s.lock, "acquire", nullptr);
    if (r == nullptr) return false;
    Py_DECREF(r);
    lock_ = s.lock;
    return true;
  }
  ~Held() {
    if (lock_ == nullptr) return;
    PyObject* r = PyObject_CallMethod(lock_, "release", nullptr);
    if (r == nullptr) PyErr_Clear();
    else Py_DECREF(r);
  }

 private:
  PyObject* lock_ = nullptr;
};

int dtype_code(at::ScalarType t) {
  switch (t) {
    case at::kBFloat16: return IMQ_DT_BF16;
    case at::kHalf: return IMQ_DT_FP16;
    case at::kFloat: return IMQ_DT_FP32;
    default: return -1;
  }
}

// No mode or transform that the Python path's torch calls would meet.
bool plain_context() {
  using c10::DispatchKey;
  static const c10::DispatchKeySet odd({DispatchKey::Python, DispatchKey::PythonTLSSnapshot, DispatchKey::Functionalize,
                                        DispatchKey::Tracer, DispatchKey::FuncTorchDynamicLayerFrontMode,
                                        DispatchKey::FuncTorchDynamicLayerBackMode, DispatchKey::FuncTorchVmapMode,
                                        DispatchKey::FuncTorchBatched, DispatchKey::Batched, DispatchKey::VmapMode});
  return !at::impl::torch_function_mode_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
         (c10::impl::tls_local_dispatch_key_set().included_ & odd).empty();
}

// The tensor behind an exact torch.Tensor (or Parameter) on device `dev` (-1: any CUDA device), else null.
const at::Tensor* plain(PyObject* o, int dev) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || t.is_neg() || t.is_conj()) return nullptr;
  if (dev >= 0 && t.get_device() != dev) return nullptr;
  static const c10::DispatchKeySet odd({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                        c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize,
                                        c10::DispatchKey::Batched});
  return (t.key_set() & odd).empty() ? &t : nullptr;
}

bool rows_ok(const at::Tensor& x) {   // _rows2d would pass x through
  return x.scalar_type() == at::kBFloat16 && x.dim() == 2 && x.stride(1) == 1 && x.stride(0) % 8 == 0 &&
         (reinterpret_cast<uintptr_t>(x.data_ptr()) & 15) == 0;
}

// linear(kind, x, q, sz, group, nd): kind = bits, + 16 for line-tiled weights; sz = (scale, zero), or the
// scale for int8; nd: x of any rank, the result of x's leading sizes (a module's forward), else x
// [M, K] -> y [M, N].
PyObject* linear_call(PyObject* const* args, Py_ssize_t n) {
  if (n != 6) Py_RETURN_NONE;
  const long kind = PyLong_AsLong(args[0]), group = PyLong_AsLong(args[4]);
  const bool nd = args[5] == Py_True;
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const int bits = (int)(kind & 15);
  if (bits != 2 && bits != 4 && bits != 8) Py_RETURN_NONE;
  const bool tiled = (kind & 16) != 0;
  const at::Tensor* x = plain(args[1], -1);
  if (x == nullptr || !plain_context()) Py_RETURN_NONE;
  const int dev = x->get_device();
  const at::Tensor* q = plain(args[2], dev);
  const at::Tensor *s = nullptr, *z = nullptr;
  if (bits == 8) {
    s = plain(args[3], dev);
  } else if (PyTuple_CheckExact(args[3]) && PyTuple_GET_SIZE(args[3]) == 2) {
    s = plain(PyTuple_GET_ITEM(args[3], 0), dev);
    z = plain(PyTuple_GET_ITEM(args[3], 1), dev);
    if (z == nullptr) Py_RETURN_NONE;
  }
  if (q == nullptr || s == nullptr || c10::hip::current_device() != dev) Py_RETURN_NONE;
  if (q->dim() != 2 || q->stride(1) != 1 || q->scalar_type() != (bits == 8 ? at::kChar : at::kByte)) Py_RETURN_NONE;
  if (tiled && (!q->is_contiguous() || (bits != 8 && group != (bits == 4 ? 128 : 64)))) Py_RETURN_NONE;
  const int64_t N = q->size(0), K = q->size(1) * (8 / bits);
  if (K < 1) Py_RETURN_NONE;
  int64_t M, sxm;
  if (nd && x->dim() != 2) {
    if (x->dim() < 1 || x->scalar_type() != at::kBFloat16 || !x->is_contiguous() || x->size(-1) != K || K % 8 != 0 ||
        (reinterpret_cast<uintptr_t>(x->data_ptr()) & 15) != 0)
      Py_RETURN_NONE;
    M = x->numel() / K;
    sxm = K;
  } else {
    if (!rows_ok(*x) || x->size(1) != K) Py_RETURN_NONE;
    M = x->size(0);
    sxm = x->stride(0);
  }
  const int sdt = dtype_code(s->scalar_type()), zdt = z ? dtype_code(z->scalar_type()) : 0;
  if (M < 1 || N < 1 || sdt < 0 || zdt < 0) Py_RETURN_NONE;
  if (bits == 8) {
    if (s->dim() < 1) Py_RETURN_NONE;
  } else {
    if (group <= 0 || K % group != 0 || s->dim() != 2 || z->dim() != 2) Py_RETURN_NONE;
    const int64_t ng = K / group;
    if (s->size(0) != N || s->size(1) != ng || z->size(0) != N || z->size(1) != ng) Py_RETURN_NONE;
  }
  void* stream = (void*)c10::hip::getCurrentHIPStream(dev).stream();
  const int64_t need = bits == 4 && !tiled
                           ? api.w4_ws(M, K, N, group, q->stride(0), sxm, s->stride(0), s->stride(1), sdt, z->stride(0),
                                       z->stride(1), zdt)
                           : api.ws(M, N, K);
  Scratch ws;
  if (!scratch(dev, stream, need, &ws)) return nullptr;
  at::Tensor y;
  if (nd && x->dim() != 2) {
    c10::SmallVector<int64_t, 6> shape(x->sizes().begin(), x->sizes().end());
    shape.back() = N;
    y = at::empty(shape, x->options().requires_grad(false));
  } else {
    y = at::empty({M, N}, x->options().requires_grad(false));
  }
  void *xp = x->data_ptr(), *qp = q->data_ptr(), *sp = s->data_ptr(), *zp = z ? z->data_ptr() : nullptr, *yp = y.data_ptr();
  const int64_t sqn = q->stride(0), s0 = s->stride(0);
  const int64_t s1 = bits == 8 ? 0 : s->stride(1), z0 = z ? z->stride(0) : 0, z1 = z ? z->stride(1) : 0;
  int rc;
  Held held;
  if (!held.take(ws)) return nullptr;
  Py_BEGIN_ALLOW_THREADS;
  if (bits == 8)
    rc = (tiled ? api.w8t : api.w8)(xp, sxm, M, K, qp, sqn, sp, s0, sdt, N, yp, N, (void*)ws.ptr, ws.bytes, stream);
  else
    rc = (bits == 4 ? (tiled ? api.w4t : api.w4) : (tiled ? api.w2t : api.w2))(
        xp, sxm, M, K, qp, sqn, sp, s0, s1, sdt, zp, z0, z1, zdt, N, group, yp, N, (void*)ws.ptr, ws.bytes, stream);
  Py_END_ALLOW_THREADS;
  if (rc != IMQ_OK) Py_RETURN_NONE;   // the Python path repeats the call and raises
  return THPVariable_Wrap(std::move(y));
}

// moe(hidden, idx, w, gu, dn, group, act, gu_bias, dn_bias, alpha, limit): moe_experts_w4 without the id
// check and with the cached workspace; gu / dn = (qweight, scale, zero, in_features).
PyObject* moe_call(PyObject* const* args, Py_ssize_t n) {
  if (n != 11) Py_RETURN_NONE;
  const at::Tensor* x = plain(args[0], -1);
  if (x == nullptr || !plain_context()) Py_RETURN_NONE;
  const int dev = x->get_device();
  const at::Tensor *idx = plain(args[1], dev), *w = plain(args[2], dev);
  if (idx == nullptr || w == nullptr || c10::hip::current_device() != dev || !rows_ok(*x)) Py_RETURN_NONE;
  const at::Tensor* t[2][3];
  int64_t feat[2];
  for (int p = 0; p < 2; ++p) {
    PyObject* o = args[3 + p];
    if (!PyTuple_CheckExact(o) || PyTuple_GET_SIZE(o) != 4) Py_RETURN_NONE;
    for (int i = 0; i < 3; ++i) {
      t[p][i] = plain(PyTuple_GET_ITEM(o, i), dev);
      if (t[p][i] == nullptr || t[p][i]->dim() != 3 || t[p][i]->stride(2) != 1) Py_RETURN_NONE;
    }
    PyObject* f = PyTuple_GET_ITEM(o, 3);
    if (!PyLong_CheckExact(f)) Py_RETURN_NONE;
    feat[p] = PyLong_AsLongLong(f);
    if (t[p][0]->scalar_type() != at::kByte || t[p][1]->scalar_type() != t[0][1]->scalar_type() ||
        t[p][2]->scalar_type() != t[0][1]->scalar_type() || t[p][1]->strides() != t[p][2]->strides())
      Py_RETURN_NONE;
  }
  if (!PyLong_CheckExact(args[5]) || !PyLong_CheckExact(args[6]) || !PyFloat_CheckExact(args[9]) || !PyFloat_CheckExact(args[10]))
    Py_RETURN_NONE;
  const int64_t group = PyLong_AsLongLong(args[5]);
  const int act = (int)PyLong_AsLong(args[6]);
  if (PyErr_Occurred()) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const at::Tensor &gq = *t[0][0], &gs = *t[0][1], &dq = *t[1][0], &ds = *t[1][1];
  const int64_t H = feat[0], I = feat[1], E = gq.size(0), T = x->size(0), gK = gq.size(2) * 2, dK = dq.size(2) * 2;
  if (idx->dim() != 2 || !idx->is_contiguous() || (idx->scalar_type() != at::kLong && idx->scalar_type() != at::kInt)) Py_RETURN_NONE;
  const int64_t k = idx->size(1);
  if (w->scalar_type() != at::kBFloat16 || !w->is_contiguous() || T < 1 || k < 1 || idx->size(0) != T) Py_RETURN_NONE;
  if (gq.size(1) != 2 * I || dq.size(1) != H) Py_RETURN_NONE;
  if (x->size(1) != gK && (x->size(1) != H || H % 8 != 0 || (T > 16 && (H % 64 != 0 || gK > 40 * 128)))) Py_RETURN_NONE;
  const int sdt = dtype_code(gs.scalar_type());
  if (sdt < 0) Py_RETURN_NONE;
  const at::Tensor* b[2] = {nullptr, nullptr};
  int bdt = 0;
  for (int p = 0; p < 2; ++p) {
    if (args[7 + p] == Py_None) continue;
    b[p] = plain(args[7 + p], dev);
    if (b[p] == nullptr || b[p]->dim() != 2 || b[p]->size(0) != E || b[p]->size(1) != (p ? H : 2 * I) || b[p]->stride(1) != 1)
      Py_RETURN_NONE;
    const int d = dtype_code(b[p]->scalar_type());
    if (d < 0 || (p && b[0] && d != bdt)) Py_RETURN_NONE;
    bdt = d;
  }
  void* stream = (void*)c10::hip::getCurrentHIPStream(dev).stream();
  const int64_t need = api.moe_ws(T, k, E, H, I, group);
  Scratch ws;
  if (!scratch(dev, stream, need > 1 ? need : 1, &ws)) return nullptr;
  at::Tensor out = at::empty({T, H}, x->options().requires_grad(false));
  void* p[] = {x->data_ptr(), idx->data_ptr(), w->data_ptr(), gq.data_ptr(), gs.data_ptr(), t[0][2]->data_ptr(),
               dq.data_ptr(), ds.data_ptr(), t[1][2]->data_ptr(), b[0] ? b[0]->data_ptr() : nullptr,
               b[1] ? b[1]->data_ptr() : nullptr, out.data_ptr()};
  const int idt = idx->scalar_type() == at::kLong ? IMQ_DT_I64 : IMQ_DT_I32;
  const float alpha = (float)PyFloat_AS_DOUBLE(args[9]), limit = (float)PyFloat_AS_DOUBLE(args[10]);
  const int64_t sx = x->stride(0), gq0 = gq.stride(0), gq1 = gq.stride(1), gs0 = gs.stride(0), gs1 = gs.stride(1);
  const int64_t dq0 = dq.stride(0), dq1 = dq.stride(1), ds0 = ds.stride(0), ds1 = ds.stride(1);
  const int64_t b0 = b[0] ? b[0]->stride(0) : 0, b1 = b[1] ? b[1]->stride(0) : 0;
  int rc;
  Held held;
  if (!held.take(ws)) return nullptr;
  Py_BEGIN_ALLOW_THREADS;
  rc = api.moe(p[0], sx, T, H, k, p[1], idt, p[2], E, p[3], gq0, gq1, gK, p[4], p[5], gs0, gs1, I, p[6], dq0, dq1, dK, p[7],
               p[8], ds0, ds1, sdt, group, p[9], b0, p[10], b1, bdt, act, alpha, limit, p[11], H, (void*)ws.ptr, ws.bytes,
               stream);
  Py_END_ALLOW_THREADS;
  if (rc != IMQ_OK) Py_RETURN_NONE;
  return THPVariable_Wrap(std::move(out));
}

// The two calls at the C boundary: what torch throws anywhere in them (a storage without an address, a device
// error, an allocation that fails) must not leave it. The Python path repeats the call and raises torch's error.
template <PyObject* (*F)(PyObject* const*, Py_ssize_t)>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  try {
    return F(args, n);
  } catch (const std::exception&) {
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
}

// init(addresses by name, scratch function)
PyObject* init(PyObject*, PyObject* args) {
  PyObject *d, *fn;
  if (!PyArg_ParseTuple(args, "O!O", &PyDict_Type, &d, &fn)) return nullptr;
  auto at = [&](const char* name) -> void* {
    PyObject* v = PyDict_GetItemString(d, name);
    if (v == nullptr) {
      PyErr_Format(PyExc_KeyError, "%s", name);
      return nullptr;
    }
    return PyLong_AsVoidPtr(v);
  };
  Api a;
#define IMQ_AT(field, name) \
  if ((a.field = reinterpret_cast<decltype(a.field)>(at(name))) == nullptr) return nullptr
  IMQ_AT(w4, "imq_linear_w4");
  IMQ_AT(w4t, "imq_linear_w4_tiled");
  IMQ_AT(w2, "imq_linear_w2");
  IMQ_AT(w2t, "imq_linear_w2_tiled");
  IMQ_AT(w8, "imq_linear_w8");
  IMQ_AT(w8t, "imq_linear_w8_tiled");
  IMQ_AT(w4_ws, "imq_linear_w4_workspace_bytes");
  IMQ_AT(ws, "imq_linear_workspace_bytes");
  IMQ_AT(moe, "imq_moe_experts_w4_ex");
  IMQ_AT(moe_ws, "imq_moe_workspace_bytes");
#undef IMQ_AT
  Py_INCREF(fn);
  Py_XDECREF(scratch_fn);
  scratch_fn = fn;
  api = a;
  Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"linear", (PyCFunction)(void (*)(void))entry<linear_call>, METH_FASTCALL, "plain fused linear, or None"},
    {"moe", (PyCFunction)(void (*)(void))entry<moe_call>, METH_FASTCALL, "plain fused experts, or None"},
    {"init", init, METH_VARARGS, "entry-point addresses and the workspace function"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "imq_fast", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_imq_fast() { return PyModule_Create(&module); }
