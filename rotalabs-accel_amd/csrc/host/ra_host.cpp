// Native host path of the GPU ops: one CPython call takes the tensors, checks
// that they are the plain case, allocates the outputs and calls the C ABI
// (include/rotaccel.h). The Python layer's own checks, the ctypes call with up
// to 18 arguments and the attribute reads cost more than the short kernels
// take: int8_gemm at M=1 K=N=4096 10.0 -> 4.7 us a call for a 3.4 us
// kernel.
//
// Every function returns None for anything but the plain case (contiguous
// CUDA tensors of the exact shapes, dtypes and device, torch.Tensor itself):
// the caller then takes the Python path, which handles every other form and
// raises every error.
//
// Workspaces stay in the Python layer's dictionary (device, stream) -> tensor,
// which is read here at each call; nothing is kept by address.
#include <Python.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/ScalarType.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <map>
#include <optional>
#include <stdexcept>
#include <tuple>
#include <type_traits>

#include "rotaccel.h"

namespace {

struct Api {
  decltype(&ra_w8a16_gemm_ws) gemm_ws;
  decltype(&ra_w8a16_gemm_auto_workspace) gemm_auto_workspace;
  decltype(&ra_w8a16_gateup_swiglu_ws) gateup_ws;
  decltype(&ra_w8a16_gateup_workspace_size) gateup_workspace;
  decltype(&ra_stream_capture_info) capture_info;
  decltype(&ra_rmsnorm) rmsnorm;
  decltype(&ra_rmsnorm_residual) rmsnorm_residual;
  decltype(&ra_swiglu) swiglu;
  decltype(&ra_swiglu_bias) swiglu_bias;
  decltype(&ra_quantize_per_channel) quantize;
  decltype(&ra_quantize_rows) quantize_rows;
  decltype(&ra_dequantize_rows) dequantize_rows;
  decltype(&ra_quantize_act_rows) quantize_act;
  decltype(&ra_w8a8_gemm) w8a8_gemm;
};
Api api;
bool ready = false;
PyObject *workspaces = nullptr;  // the Python layer's dict (device, stream) -> buffer of the eager calls
PyObject *new_workspace = nullptr;  // its function (device index, bytes) -> (pointer, bytes)

int code(at::ScalarType t) {
  return t == at::kHalf ? RA_F16 : t == at::kBFloat16 ? RA_BF16 : t == at::kFloat ? RA_F32 : -1;
}

// The tensor of `o` if it is a plain contiguous one on the device of the
// call: torch.Tensor or Parameter itself, dense, not wrapped by a transform.
struct Plain {
  const at::Tensor *t = nullptr;
  explicit Plain(PyObject *o) {
    if (!THPVariable_CheckExact(o)) return;
    const at::Tensor &v = THPVariable_Unpack(o);
    const c10::DispatchKeySet ks = v.key_set();
    if (!v.is_cuda() || !v.has_storage() || v.layout() != at::kStrided || !v.is_contiguous() ||
        ks.has(c10::DispatchKey::Python) || ks.has(c10::DispatchKey::FuncTorchBatched) ||
        ks.has(c10::DispatchKey::FuncTorchGradWrapper) || ks.has(c10::DispatchKey::Functionalize) ||
        ks.has(c10::DispatchKey::Conjugate) || ks.has(c10::DispatchKey::Negative) || v.numel() == 0)
      return;
    t = &v;
  }
  explicit operator bool() const { return t != nullptr; }
  const at::Tensor *operator->() const { return t; }
  const at::Tensor &operator*() const { return *t; }
};

// Rows the GEMM kernels read in place: 16-byte aligned wherever their length
// is a whole number of 16 bytes (the Python layer copies the others).
bool rows_ok(const at::Tensor &t, int64_t cols) {
  return (cols * t.element_size()) % 16 != 0 || (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
}

// Device and stream of a call: the tensors' device, which must be current.
struct Ctx {
  int dev = -1;
  hipStream_t stream = nullptr;
  explicit Ctx(const at::Tensor &t) {
    if (t.get_device() != c10::hip::current_device()) return;
    dev = (int)t.get_device();
    stream = c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream();
  }
  bool ok() const { return dev >= 0; }
  bool has(const Plain &p) const { return p && p->get_device() == dev; }
};

// Workspace bytes the automatic choice uses, kept per problem (bounded).
template <typename Fn>
size_t workspace_need(Fn fn, bool gateup, int64_t M, int64_t N, int64_t K, int dt) {
  static std::map<std::tuple<bool, int64_t, int64_t, int64_t, int>, size_t> sizes;
  const auto key = std::make_tuple(gateup, M, N, K, dt);
  const auto it = sizes.find(key);
  if (it != sizes.end()) return it->second;
  if (sizes.size() >= 4096) sizes.clear();
  return sizes[key] = fn(M, N, K, dt);
}

// A buffer of at least `need` bytes (0: none) for the next call on the
// stream: the stream's own, read from the dict, or what the Python layer
// hands out (nothing there yet, one too small, a graph being captured).
void workspace(const Ctx &c, size_t need, void *&ws, size_t &bytes) {
  ws = nullptr;
  bytes = 0;
  if (need == 0) return;
  int capturing = 0;
  unsigned long long id = 0;
  if (api.capture_info(c.stream, &capturing, &id) == RA_OK && !capturing) {
    THPObjectPtr key(Py_BuildValue("(iK)", c.dev, (unsigned long long)(uintptr_t)c.stream));
    if (!key) throw python_error();
    PyObject *v = PyDict_GetItemWithError(workspaces, key.get());  // borrowed
    if (v && THPVariable_CheckExact(v) && (size_t)THPVariable_Unpack(v).numel() >= need) {
      const at::Tensor &t = THPVariable_Unpack(v);
      ws = t.data_ptr();
      bytes = (size_t)t.numel();
      return;
    }
    if (!v && PyErr_Occurred()) throw python_error();
  }
  THPObjectPtr got(PyObject_CallFunction(new_workspace, "in", c.dev, (Py_ssize_t)need));
  if (!got) throw python_error();
  if (!PyTuple_Check(got.get()) || PyTuple_GET_SIZE(got.get()) != 2) throw std::runtime_error("workspace: bad reply");
  ws = PyLong_AsVoidPtr(PyTuple_GET_ITEM(got.get(), 0));
  bytes = PyLong_AsSize_t(PyTuple_GET_ITEM(got.get(), 1));
  if (PyErr_Occurred()) throw python_error();
}

// A C ABI call without the interpreter lock (a launch waits when the device's
// queue is full; other threads go on, as with ctypes).
template <typename... P, typename... A>
int enqueue(int (*fn)(P...), A... args) {
  PyThreadState *const st = PyEval_SaveThread();
  const int r = fn(args...);
  PyEval_RestoreThread(st);
  return r;
}

at::Tensor make(at::IntArrayRef sizes, const at::Tensor &like, at::ScalarType dt) {
  return at::empty(sizes, at::TensorOptions().dtype(dt).device(like.device()));
}

c10::SmallVector<int64_t, 5> with_last(const at::Tensor &x, int64_t n) {
  c10::SmallVector<int64_t, 5> s(x.sizes().begin(), x.sizes().end());
  s.back() = n;
  return s;
}

// ---- the ops, on checked tensors; an undefined result: the Python path ----

at::Tensor gemm(const Ctx &c, const at::Tensor &x, const Plain &w, const Plain &s, const Plain *b) {
  const int dt = code(x.scalar_type());
  if (dt < 0 || x.dim() < 1 || !c.has(w) || !c.has(s) || w->scalar_type() != at::kChar || w->dim() != 2 ||
      s->scalar_type() != at::kFloat || s->dim() != 1)
    return {};
  const int64_t K = x.size(-1), N = w->size(0), M = x.numel() / K;
  if (w->size(1) != K || s->size(0) != N || !rows_ok(x, K) || !rows_ok(*w, K)) return {};
  if (b && (!c.has(*b) || (*b)->dim() != 1 || (*b)->size(0) != N || code((*b)->scalar_type()) < 0)) return {};
  void *ws;
  size_t bytes;
  workspace(c, workspace_need(api.gemm_auto_workspace, false, M, N, K, dt), ws, bytes);
  at::Tensor y = make(with_last(x, N), x, x.scalar_type());
  const int st = enqueue(api.gemm_ws, x.data_ptr(), K, dt, static_cast<const int8_t *>(w->data_ptr()), K,
                             static_cast<const float *>(s->data_ptr()), b ? (*b)->data_ptr() : nullptr,
                             b ? code((*b)->scalar_type()) : RA_F32, y.data_ptr(), N, M, N, K, ws, bytes, c.stream);
  return st == RA_OK ? y : at::Tensor();
}

at::Tensor gateup(const Ctx &c, const at::Tensor &x, const Plain &w, const Plain &s) {
  const int dt = code(x.scalar_type());
  if (dt < 0 || x.dim() < 1 || !c.has(w) || !c.has(s) || w->scalar_type() != at::kChar || w->dim() != 2 ||
      s->scalar_type() != at::kFloat || s->dim() != 1)
    return {};
  const int64_t K = x.size(-1), N2 = w->size(0), inter = N2 / 2, M = x.numel() / K;
  if (N2 % 2 || w->size(1) != K || s->size(0) != N2 || !rows_ok(x, K) || !rows_ok(*w, K)) return {};
  void *ws;
  size_t bytes;
  workspace(c, workspace_need(api.gateup_workspace, true, M, inter, K, dt), ws, bytes);
  at::Tensor h = make(with_last(x, inter), x, x.scalar_type());
  const int st = enqueue(api.gateup_ws, x.data_ptr(), K, dt, static_cast<const int8_t *>(w->data_ptr()), K,
                               static_cast<const float *>(s->data_ptr()), h.data_ptr(), inter, M, inter, K, ws, bytes,
                               c.stream);
  return st == RA_OK ? h : at::Tensor();
}

at::Tensor rmsnorm(const Ctx &c, const Plain &x, const Plain *r, const Plain &w, double eps) {
  if (!c.has(x) || !c.has(w) || x->dim() < 1 || w->dim() != 1) return {};
  const int64_t H = x->size(-1), rows = x->numel() / H;
  const int xd = code(x->scalar_type()), wd = code(w->scalar_type());
  if (xd < 0 || wd < 0 || w->size(0) != H) return {};
  if (r && (!c.has(*r) || (*r)->sizes() != x->sizes() || code((*r)->scalar_type()) < 0)) return {};
  const at::ScalarType od = xd == wd ? x->scalar_type() : at::kFloat;
  at::Tensor y = make(x->sizes(), *x, od);
  const int st =
      r ? enqueue(api.rmsnorm_residual, x->data_ptr(), H, xd, (*r)->data_ptr(), H, code((*r)->scalar_type()), w->data_ptr(), wd,
                               y.data_ptr(), H, code(od), rows, H, (float)eps, c.stream)
        : enqueue(api.rmsnorm, x->data_ptr(), H, xd, w->data_ptr(), wd, y.data_ptr(), H, code(od), rows, H, (float)eps, c.stream);
  return st == RA_OK ? y : at::Tensor();
}

PyObject *give(const at::Tensor &t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}

PyObject *give2(const at::Tensor &a, const at::Tensor &b) {
  PyObject *pa = THPVariable_Wrap(a), *pb = pa ? THPVariable_Wrap(b) : nullptr;
  if (!pb) {
    Py_XDECREF(pa);
    return nullptr;
  }
  PyObject *t = PyTuple_Pack(2, pa, pb);
  Py_DECREF(pa);
  Py_DECREF(pb);
  return t;
}

// Argument count and readiness common to all; x: the first tensor.
#define RA_HOST_BEGIN(n_)                        \
  HANDLE_TH_ERRORS                               \
  if (!ready || nargs != (n_)) Py_RETURN_NONE;   \
  const Plain x(args[0]);                        \
  if (!x) Py_RETURN_NONE;                        \
  const Ctx c(*x);                               \
  if (!c.ok()) Py_RETURN_NONE;
#define RA_HOST_END END_HANDLE_TH_ERRORS

// gemm(x, weight, scale, bias | None)
PyObject *py_gemm(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  RA_HOST_BEGIN(4)
  std::optional<Plain> b;
  if (args[3] != Py_None) b.emplace(args[3]);
  return give(gemm(c, *x, Plain(args[1]), Plain(args[2]), b ? &*b : nullptr));
  RA_HOST_END
}

// gateup(x, weight, scale)
PyObject *py_gateup(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  RA_HOST_BEGIN(3)
  return give(gateup(c, *x, Plain(args[1]), Plain(args[2])));
  RA_HOST_END
}

// rmsnorm(x, residual | None, weight, eps)
PyObject *py_rmsnorm(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  RA_HOST_BEGIN(4)
  if (!PyFloat_CheckExact(args[3])) Py_RETURN_NONE;
  std::optional<Plain> r;
  if (args[1] != Py_None) r.emplace(args[1]);
  return give(rmsnorm(c, x, r ? &*r : nullptr, Plain(args[2]), PyFloat_AS_DOUBLE(args[3])));
  RA_HOST_END
}

// swiglu(gate, up)
PyObject *py_swiglu(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  RA_HOST_BEGIN(2)
  const Plain u(args[1]);
  const int dt = code(x->scalar_type());
  if (!c.has(u) || dt < 0 || u->scalar_type() != x->scalar_type() || u->sizes() != x->sizes()) Py_RETURN_NONE;
  at::Tensor y = make(x->sizes(), *x, x->scalar_type());
  if (enqueue(api.swiglu, x->data_ptr(), u->data_ptr(), y.data_ptr(), x->numel(), dt, c.stream) != RA_OK) Py_RETURN_NONE;
  return give(y);
  RA_HOST_END
}

// swiglu_bias(gate, up, bias_gate, bias_up)
PyObject *py_swiglu_bias(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  RA_HOST_BEGIN(4)
  const Plain u(args[1]), bg(args[2]), bu(args[3]);
  const int dt = code(x->scalar_type());
  if (!c.has(u) || !c.has(bg) || !c.has(bu) || dt < 0 || x->dim() < 1 || u->scalar_type() != x->scalar_type() ||
      u->sizes() != x->sizes())
    Py_RETURN_NONE;
  const int64_t H = x->size(-1);
  const int bd = code(bg->scalar_type());
  if (bd < 0 || bu->scalar_type() != bg->scalar_type() || bg->dim() != 1 || bu->dim() != 1 || bg->size(0) != H ||
      bu->size(0) != H)
    Py_RETURN_NONE;
  at::Tensor y = make(x->sizes(), *x, x->scalar_type());
  if (enqueue(api.swiglu_bias, x->data_ptr(), u->data_ptr(), bg->data_ptr(), bu->data_ptr(), bd, y.data_ptr(), x->numel(), H, dt,
                      c.stream) != RA_OK)
    Py_RETURN_NONE;
  return give(y);
  RA_HOST_END
}

// quantize(weight) -> (codes, scale)
PyObject *py_quantize(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  RA_HOST_BEGIN(1)
  const int dt = code(x->scalar_type());
  if (dt < 0 || x->dim() != 2) Py_RETURN_NONE;
  const int64_t N = x->size(0), K = x->size(1);
  at::Tensor q = make({N, K}, *x, at::kChar), s = make({N}, *x, at::kFloat);
  if (enqueue(api.quantize, x->data_ptr(), K, dt, N, K, static_cast<int8_t *>(q.data_ptr()), K,
                   static_cast<float *>(s.data_ptr()), c.stream) != RA_OK)
    Py_RETURN_NONE;
  return give2(q, s);
  RA_HOST_END
}

// kv_quantize(tensor, bits) -> (codes, scale)
PyObject *py_kv_quantize(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  RA_HOST_BEGIN(2)
  const int dt = code(x->scalar_type());
  const long bits = PyLong_Check(args[1]) ? PyLong_AsLong(args[1]) : 0;
  if (dt < 0 || x->dim() < 1 || (bits != 8 && bits != 4)) {
    PyErr_Clear();
    Py_RETURN_NONE;
  }
  const int64_t cols = x->size(-1), rows = x->numel() / cols;
  at::Tensor q = make(x->sizes(), *x, at::kChar), s = make(with_last(*x, 1), *x, x->scalar_type());
  if (enqueue(api.quantize_rows, x->data_ptr(), cols, dt, rows, cols, (int)bits, static_cast<int8_t *>(q.data_ptr()), cols,
                        s.data_ptr(), c.stream) != RA_OK)
    Py_RETURN_NONE;
  return give2(q, s);
  RA_HOST_END
}

// kv_dequantize(codes, scale): values in the scale's dtype
PyObject *py_kv_dequantize(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  RA_HOST_BEGIN(2)
  const Plain s(args[1]);
  if (!c.has(s) || x->scalar_type() != at::kChar || x->dim() < 1 || s->dim() != x->dim() || s->size(-1) != 1 ||
      s->requires_grad())
    Py_RETURN_NONE;
  const int dt = code(s->scalar_type());
  const int64_t cols = x->size(-1), rows = x->numel() / cols;
  if (dt < 0 || s->sizes().slice(0, s->dim() - 1) != x->sizes().slice(0, x->dim() - 1)) Py_RETURN_NONE;
  at::Tensor y = make(x->sizes(), *x, s->scalar_type());
  if (enqueue(api.dequantize_rows, static_cast<const int8_t *>(x->data_ptr()), s->data_ptr(), dt, rows, cols, y.data_ptr(),
                          c.stream) != RA_OK)
    Py_RETURN_NONE;
  return give(y);
  RA_HOST_END
}

// w8a8(x, weight, scale, bias | None, act_scale)
PyObject *py_w8a8(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  RA_HOST_BEGIN(5)
  const Plain w(args[1]), s(args[2]);
  std::optional<Plain> b;
  if (args[3] != Py_None) b.emplace(args[3]);
  const int dt = code(x->scalar_type());
  if (!PyFloat_CheckExact(args[4]) || (dt != RA_F16 && dt != RA_BF16) || x->dim() < 1 || !c.has(w) || !c.has(s) ||
      w->scalar_type() != at::kChar || w->dim() != 2 || s->scalar_type() != at::kFloat || s->dim() != 1)
    Py_RETURN_NONE;
  const int64_t K = x->size(-1), N = w->size(0), M = x->numel() / K;
  if (w->size(1) != K || s->size(0) != N || !rows_ok(*x, K) || !rows_ok(*w, K)) Py_RETURN_NONE;
  if (b && (!c.has(*b) || (*b)->dim() != 1 || (*b)->size(0) != N || code((*b)->scalar_type()) < 0)) Py_RETURN_NONE;
  at::Tensor q = make({M, K}, *x, at::kChar), xs = make({M}, *x, x->scalar_type());
  at::Tensor y = make(with_last(*x, N), *x, x->scalar_type());
  if (enqueue(api.quantize_act, x->data_ptr(), K, dt, M, K, static_cast<int8_t *>(q.data_ptr()), K, xs.data_ptr(),
                       (float)PyFloat_AS_DOUBLE(args[4]), c.stream) != RA_OK)
    Py_RETURN_NONE;
  if (enqueue(api.w8a8_gemm, static_cast<const int8_t *>(q.data_ptr()), K, xs.data_ptr(),
                    static_cast<const int8_t *>(w->data_ptr()), K, static_cast<const float *>(s->data_ptr()),
                    b ? (*b)->data_ptr() : nullptr, b ? code((*b)->scalar_type()) : RA_F32, y.data_ptr(), N, dt, M, N, K,
                    c.stream) != RA_OK)
    Py_RETURN_NONE;
  return give(y);
  RA_HOST_END
}

// mlp(x, residual | None, norm_weight, eps, weight_gate_up, scale_gate_up, weight_down, scale_down).
// (The later stages' tensors are checked before the first launch; where one
// still declines, the Python path does the whole product again.)
PyObject *py_mlp(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  RA_HOST_BEGIN(8)
  if (!PyFloat_CheckExact(args[3])) Py_RETURN_NONE;
  std::optional<Plain> r;
  if (args[1] != Py_None) r.emplace(args[1]);
  const Plain nw(args[2]), wgu(args[4]), sgu(args[5]), wd(args[6]), sd(args[7]);
  auto pair_ok = [&](const Plain &w, const Plain &s, int64_t k) {
    return c.has(w) && c.has(s) && w->scalar_type() == at::kChar && w->dim() == 2 && w->size(1) == k &&
           s->scalar_type() == at::kFloat && s->dim() == 1 && s->size(0) == w->size(0) && rows_ok(*w, k);
  };
  if (!c.has(nw) || x->dim() < 1 || !pair_ok(wgu, sgu, x->size(-1)) || wgu->size(0) % 2 ||
      !pair_ok(wd, sd, wgu->size(0) / 2))
    Py_RETURN_NONE;
  const at::Tensor h = rmsnorm(c, x, r ? &*r : nullptr, nw, PyFloat_AS_DOUBLE(args[3]));
  if (!h.defined()) Py_RETURN_NONE;
  const at::Tensor a = gateup(c, h, wgu, sgu);
  if (!a.defined()) Py_RETURN_NONE;
  return give(gemm(c, a, wd, sd, nullptr));
  RA_HOST_END
}

// init(library path, workspace dict, workspace function) -> bool
PyObject *py_init(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
  const char *path = nargs == 3 ? PyUnicode_AsUTF8(args[0]) : nullptr;
  if (!path || !PyDict_CheckExact(args[1]) || !PyCallable_Check(args[2])) {
    PyErr_Clear();
    Py_RETURN_FALSE;
  }
  void *h = dlopen(path, RTLD_NOW | RTLD_LOCAL);
  if (!h) Py_RETURN_FALSE;
  bool all = true;
  auto get = [&](auto &fn, const char *name) {
    fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(dlsym(h, name));
    all = all && fn != nullptr;
  };
  get(api.gemm_ws, "ra_w8a16_gemm_ws");
  get(api.gemm_auto_workspace, "ra_w8a16_gemm_auto_workspace");
  get(api.gateup_ws, "ra_w8a16_gateup_swiglu_ws");
  get(api.gateup_workspace, "ra_w8a16_gateup_workspace_size");
  get(api.capture_info, "ra_stream_capture_info");
  get(api.rmsnorm, "ra_rmsnorm");
  get(api.rmsnorm_residual, "ra_rmsnorm_residual");
  get(api.swiglu, "ra_swiglu");
  get(api.swiglu_bias, "ra_swiglu_bias");
  get(api.quantize, "ra_quantize_per_channel");
  get(api.quantize_rows, "ra_quantize_rows");
  get(api.dequantize_rows, "ra_dequantize_rows");
  get(api.quantize_act, "ra_quantize_act_rows");
  get(api.w8a8_gemm, "ra_w8a8_gemm");
  if (!all) Py_RETURN_FALSE;
  Py_INCREF(args[1]);
  Py_INCREF(args[2]);
  Py_XDECREF(workspaces);
  Py_XDECREF(new_workspace);
  workspaces = args[1];
  new_workspace = args[2];
  ready = true;
  Py_RETURN_TRUE;
}

#define RA_METHOD(name_, fn_) {name_, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn_)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {RA_METHOD("init", py_init),
                         RA_METHOD("gemm", py_gemm),
                         RA_METHOD("gateup", py_gateup),
                         RA_METHOD("rmsnorm", py_rmsnorm),
                         RA_METHOD("swiglu", py_swiglu),
                         RA_METHOD("swiglu_bias", py_swiglu_bias),
                         RA_METHOD("quantize", py_quantize),
                         RA_METHOD("kv_quantize", py_kv_quantize),
                         RA_METHOD("kv_dequantize", py_kv_dequantize),
                         RA_METHOD("w8a8", py_w8a8),
                         RA_METHOD("mlp", py_mlp),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_ra_host", "native host path of the GPU ops", -1, methods,
                      nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__ra_host(void) { return PyModule_Create(&module); }
