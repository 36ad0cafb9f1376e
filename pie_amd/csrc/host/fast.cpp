// Native call path of the ops a decode step issues one by one: argument checks, output allocation
// and the C-ABI call without the interpreter between them.
//
// An op of a single decode token runs 2.5-4 us on the GPU, and the Python wrappers spent 13 us on a
// call (kwargs checks, torch.Size and device objects, ctypes conversion of up to 30 arguments), so a
// small step ran at the host's rate: a one-token decode layer (5 calls, 6 kernels) 67 us. Here a call
// costs little more than its output allocations and launches.
//
// Every function handles the plain case and returns None for anything else (another type or tensor
// subclass, a transform's or mode's tensor, a dtype, shape, stride or device it does not serve, a
// call the library refuses before any launch): the Python wrapper then takes its general path, which
// accepts, converts or refuses the call as it always has. An error of the launch itself is raised
// here: it is found after the kernel was handed to the runtime, so the op must not be issued again.
// Nothing is kept between calls.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>

#include <cmath>

#include "../../../include/pie_hip.h"

namespace {

// The C ABI of the kernel library the Python binding loaded (bind()).
#define PIE_ENTRY_POINTS(X)                                                                       \
  X(pie_hip_abi_version) X(pie_hip_rmsnorm) X(pie_hip_gemma_rmsnorm)                              \
  X(pie_hip_fused_add_rmsnorm) X(pie_hip_gemma_fused_add_rmsnorm) X(pie_hip_silu_and_mul)         \
  X(pie_hip_gelu_tanh_and_mul) X(pie_hip_embedding) X(pie_hip_qk_rmsnorm_rope_append)             \
  X(pie_hip_attention_decode) X(pie_hip_attention_prefill_split)
struct Lib {
#define X(name) decltype(&::name) name = nullptr;
  PIE_ENTRY_POINTS(X)
#undef X
} lib;

const c10::DispatchKeySet kTransforms({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched,
                                       c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Batched,
                                       c10::DispatchKey::Functionalize});

// The tensor behind a plain GPU tensor object of `dtype`, or nullptr.
const at::Tensor* tensor(PyObject* o, at::ScalarType dtype) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || t.scalar_type() != dtype || !t.is_cuda() || t.layout() != at::kStrided ||
      !t.unsafeGetTensorImpl()->has_storage() || t.key_set().has_any(kTransforms))
    return nullptr;
  return &t;
}
const at::Tensor* bf16(PyObject* o) { return tensor(o, at::kBFloat16); }
const at::Tensor* i32(PyObject* o) { return tensor(o, at::kInt); }

bool modes_active() {
  return at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set();
}

// A tensor as rows of `cols` elements with unit inner stride, without a copy.
struct Rows {
  uint16_t* p = nullptr;
  int64_t n = 0, stride = 0;
  bool ok = false;
};
Rows rows(const at::Tensor& t, int64_t cols) {
  Rows r;
  const int64_t d = t.dim();
  if (d < 1 || cols <= 0 || t.size(d - 1) != cols || t.numel() == 0) return r;
  if (d == 2 && t.stride(1) == 1) {
    r.n = t.size(0);
    r.stride = t.stride(0);
  } else if (t.is_contiguous()) {
    r.n = t.numel() / cols;
    r.stride = cols;
  } else {
    return r;
  }
  r.p = static_cast<uint16_t*>(t.data_ptr());
  r.ok = true;
  return r;
}
bool vec1(const at::Tensor& t, int64_t n) { return t.dim() == 1 && t.size(0) == n && (n == 1 || t.stride(0) == 1); }

// The output: the caller's tensor where given (no_out otherwise), else a new one.
bool output(PyObject* o, const at::Tensor& like, at::IntArrayRef sizes, at::Tensor& out) {
  if (o == Py_None) {
    out = at::empty(sizes, at::TensorOptions().dtype(at::kBFloat16).device(like.device()));
    return out.unsafeGetTensorImpl()->has_storage() && !out.key_set().has_any(kTransforms);
  }
  const at::Tensor* t = bf16(o);
  if (!t || t->device() != like.device() || t->sizes() != sizes) return false;
  out = *t;
  return true;
}
// The object to hand back for an output: the caller's own where it gave one.
PyObject* give(PyObject* o, const at::Tensor& t) {
  if (o != Py_None) {
    Py_INCREF(o);
    return o;
  }
  return THPVariable_Wrap(t);
}

void* stream_of(const at::Tensor& t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
template <typename T>
T* ptr(const at::Tensor& t) { return static_cast<T*>(t.data_ptr()); }

bool f64(PyObject* o, double& v) {
  if (!PyFloat_CheckExact(o) && !PyLong_CheckExact(o)) return false;
  v = PyFloat_AsDouble(o);
  return !(v == -1.0 && PyErr_Occurred());
}

#define NOT_SERVED                     \
  do {                                 \
    PyErr_Clear();                     \
    Py_RETURN_NONE;                    \
  } while (0)
#define SERVE(cond) \
  if (!(cond)) NOT_SERVED

template <typename F>
int launch(F&& f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = f();
  Py_END_ALLOW_THREADS
  return rc;
}

// The binding's check(entry point name, return code), which raises the library's error (bind()).
PyObject* on_error = nullptr;

// Makes the call; hands it to the general path where the library refused it before any launch, and
// raises any other error.
#define LAUNCH(name, ...)                                                    \
  do {                                                                       \
    const int rc = launch([&] { return __VA_ARGS__; });                      \
    if (rc == PIE_HIP_EINVAL || rc == PIE_HIP_EBUSY) NOT_SERVED;             \
    if (rc != PIE_HIP_OK) {                                                  \
      Py_XDECREF(PyObject_CallFunction(on_error, "si", name, rc));           \
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, name);      \
      return nullptr;                                                        \
    }                                                                        \
  } while (0)

// rmsnorm(input, weight, eps, out, gemma)
PyObject* rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  double eps;
  SERVE(n == 5 && !modes_active());
  const at::Tensor *x = bf16(a[0]), *w = bf16(a[1]);
  SERVE(x && w && x->dim() != 3 && x->dim() >= 1 && x->device() == w->device() && f64(a[2], eps));
  const int64_t H = x->size(-1);
  const Rows xr = rows(*x, H);
  SERVE(xr.ok && vec1(*w, H));
  at::Tensor out;
  SERVE(output(a[3], *x, x->sizes(), out));
  const Rows yr = rows(out, H);
  SERVE(yr.ok);
  const bool gemma = a[4] == Py_True;
  const auto fn = gemma ? lib.pie_hip_gemma_rmsnorm : lib.pie_hip_rmsnorm;
  void* st = stream_of(*x);
  const uint16_t* wp = ptr<uint16_t>(*w);
  LAUNCH(gemma ? "pie_hip_gemma_rmsnorm" : "pie_hip_rmsnorm",
         fn(xr.p, xr.stride, wp, yr.p, yr.stride, xr.n, H, (float)eps, st));
  return give(a[3], out);
  END_HANDLE_TH_ERRORS
}

// add_rms_norm(input, residual, weight, eps, out, residual_out, gemma)
PyObject* add_rms_norm(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  double eps;
  SERVE(n == 7 && !modes_active());
  const at::Tensor *x = bf16(a[0]), *r = bf16(a[1]), *w = bf16(a[2]);
  SERVE(x && r && w && x->dim() >= 1 && x->device() == r->device() && x->device() == w->device() &&
        x->sizes() == r->sizes() && f64(a[3], eps));
  const int64_t H = x->size(-1);
  const Rows xr = rows(*x, H), rr = rows(*r, H);
  SERVE(xr.ok && rr.ok && vec1(*w, H));
  at::Tensor out, sum;
  SERVE(output(a[4], *x, x->sizes(), out) && output(a[5], *x, x->sizes(), sum));
  const Rows yr = rows(out, H), sr = rows(sum, H);
  SERVE(yr.ok && sr.ok);
  const bool gemma = a[6] == Py_True;
  const auto fn = gemma ? lib.pie_hip_gemma_fused_add_rmsnorm : lib.pie_hip_fused_add_rmsnorm;
  void* st = stream_of(*x);
  const uint16_t* wp = ptr<uint16_t>(*w);
  LAUNCH(gemma ? "pie_hip_gemma_fused_add_rmsnorm" : "pie_hip_fused_add_rmsnorm",
         fn(xr.p, xr.stride, rr.p, rr.stride, sr.p, sr.stride, yr.p, yr.stride, wp, xr.n, H, (float)eps, st));
  PyObject* pair = PyTuple_New(2);
  if (!pair) return nullptr;
  PyTuple_SET_ITEM(pair, 0, give(a[4], out));
  PyTuple_SET_ITEM(pair, 1, give(a[5], sum));
  return pair;
  END_HANDLE_TH_ERRORS
}

// act_and_mul(input, out, gelu)
PyObject* act_and_mul(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  SERVE(n == 3 && !modes_active());
  const at::Tensor* x = bf16(a[0]);
  SERVE(x && x->dim() >= 1 && x->size(-1) % 2 == 0);
  const int64_t I = x->size(-1) / 2;
  const Rows xr = rows(*x, 2 * I);
  SERVE(xr.ok);
  at::DimVector sizes(x->sizes().begin(), x->sizes().end());
  sizes.back() = I;
  at::Tensor out;
  SERVE(output(a[1], *x, sizes, out));
  const Rows yr = rows(out, I);
  SERVE(yr.ok);
  const bool gelu = a[2] == Py_True;
  const auto fn = gelu ? lib.pie_hip_gelu_tanh_and_mul : lib.pie_hip_silu_and_mul;
  void* st = stream_of(*x);
  LAUNCH(gelu ? "pie_hip_gelu_tanh_and_mul" : "pie_hip_silu_and_mul", fn(xr.p, xr.stride, yr.p, yr.stride, xr.n, I, st));
  return give(a[1], out);
  END_HANDLE_TH_ERRORS
}

// embedding(ids, weight, out)
PyObject* embedding(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  SERVE(n == 3 && !modes_active());
  const at::Tensor *ids = i32(a[0]), *w = bf16(a[1]);
  SERVE(ids && w && ids->device() == w->device() && ids->is_contiguous() && ids->numel() > 0 && w->dim() == 2 &&
        w->stride(1) == 1 && w->numel() > 0);
  const int64_t H = w->size(1), T = ids->numel();
  at::DimVector sizes(ids->sizes().begin(), ids->sizes().end());
  sizes.push_back(H);
  at::Tensor out;
  SERVE(output(a[2], *w, sizes, out));
  const Rows yr = rows(out, H);
  SERVE(yr.ok && yr.n == T);
  void* st = stream_of(*w);
  const int32_t* ip = ptr<int32_t>(*ids);
  const uint16_t* wp = ptr<uint16_t>(*w);
  LAUNCH("pie_hip_embedding", lib.pie_hip_embedding(ip, T, wp, w->size(0), H, w->stride(0), yr.p, yr.stride, st));
  return give(a[2], out);
  END_HANDLE_TH_ERRORS
}

// The paged cache as one [pages, 2, ...] tensor of unit inner stride.
struct Cache {
  uint16_t *k = nullptr, *v = nullptr;
  int64_t pages = 0, page = 0, slot = 0, head = 0, page_size = 0;
  bool ok = false;
};
Cache cache(PyObject* o, bool nhd, int64_t Hkv, int64_t D, const at::Device& dev) {
  Cache c;
  const at::Tensor* t = bf16(o);
  if (!t || t->device() != dev || t->dim() != 5 || t->size(1) != 2) return c;
  const int sl = nhd ? 2 : 3, hd = nhd ? 3 : 2;
  if (t->size(hd) != Hkv || t->size(4) != D || t->stride(4) != 1) return c;
  c.k = ptr<uint16_t>(*t);
  c.v = c.k + t->stride(1);
  c.pages = t->size(0);
  c.page = t->stride(0);
  c.slot = t->stride(sl);
  c.head = t->stride(hd);
  c.page_size = t->size(sl);
  c.ok = true;
  return c;
}
// 1 for "NHD", 0 for "HND", -1 otherwise
int layout(PyObject* o) {
  if (!PyUnicode_CheckExact(o)) return -1;
  if (PyUnicode_CompareWithASCIIString(o, "NHD") == 0) return 1;
  return PyUnicode_CompareWithASCIIString(o, "HND") == 0 ? 0 : -1;
}

// qk_rms_norm_rope_append(q, k, v, q_weight, k_weight, eps, pos_ids, batch_indices, positions, cache,
//   kv_indices, kv_indptr, kv_last_page_len, kv_layout, inv_freq address, q_out, k_out)
PyObject* qk_rms_norm_rope_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  double eps;
  SERVE(n == 17 && !modes_active());
  const at::Tensor *q = bf16(a[0]), *k = bf16(a[1]), *v = bf16(a[2]), *qw = bf16(a[3]), *kw = bf16(a[4]);
  SERVE(q && k && v && qw && kw && f64(a[5], eps));
  const at::Tensor *pos = i32(a[6]), *bi = i32(a[7]), *ps = i32(a[8]), *ki = i32(a[10]), *kp = i32(a[11]),
                   *ll = i32(a[12]);
  SERVE(pos && bi && ps && ki && kp && ll);
  const auto dev = q->device();
  for (const at::Tensor* t : {k, v, qw, kw, pos, bi, ps, ki, kp, ll}) SERVE(t->device() == dev);
  SERVE(q->dim() == 3 && k->dim() == 3 && k->sizes() == v->sizes());
  const int64_t T = q->size(0), Hq = q->size(1), D = q->size(2), Hkv = k->size(1);
  SERVE(T > 0 && Hq > 0 && Hkv > 0 && D > 0 && D % 2 == 0 && D <= 512 && k->size(0) == T && k->size(2) == D &&
        q->stride(2) == 1 && k->stride(2) == 1 && v->stride(2) == 1 && vec1(*qw, D) && vec1(*kw, D));
  for (const at::Tensor* t : {pos, bi, ps}) SERVE(t->dim() == 1 && t->size(0) == T && t->is_contiguous());
  SERVE(kp->dim() == 1 && kp->numel() >= 1 && kp->is_contiguous() && ki->is_contiguous());
  const int nhd = layout(a[13]);
  SERVE(nhd >= 0);
  const Cache c = cache(a[9], nhd == 1, Hkv, D, dev);
  SERVE(c.ok);
  const float* inv = static_cast<const float*>(PyLong_AsVoidPtr(a[14]));
  SERVE(inv);
  at::Tensor qo, ko;
  SERVE(output(a[15], *q, q->sizes(), qo) && output(a[16], *k, k->sizes(), ko));
  SERVE(qo.stride(2) == 1 && ko.stride(2) == 1);
  void* st = stream_of(*q);
  uint16_t *qp = ptr<uint16_t>(*q), *kpp = ptr<uint16_t>(*k), *vp = ptr<uint16_t>(*v), *qop = ptr<uint16_t>(qo),
           *kop = ptr<uint16_t>(ko), *qwp = ptr<uint16_t>(*qw), *kwp = ptr<uint16_t>(*kw);
  const int32_t *pp = ptr<int32_t>(*pos), *bp = ptr<int32_t>(*bi), *sp = ptr<int32_t>(*ps), *kip = ptr<int32_t>(*ki),
                *kpi = ptr<int32_t>(*kp);
  LAUNCH("pie_hip_qk_rmsnorm_rope_append",
         lib.pie_hip_qk_rmsnorm_rope_append(
             qp, q->stride(0), q->stride(1), kpp, k->stride(0), k->stride(1), vp, v->stride(0), v->stride(1), qop,
             qo.stride(0), qo.stride(1), kop, ko.stride(0), ko.stride(1), qwp, kwp, (float)eps, pp, T, Hq, Hkv, D,
             inv, bp, sp, kip, kpi, kp->numel() - 1, c.k, c.v, c.pages, c.page, c.slot, c.head, c.page_size, st));
  PyObject* pair = PyTuple_New(2);
  if (!pair) return nullptr;
  PyTuple_SET_ITEM(pair, 0, give(a[15], qo));
  PyTuple_SET_ITEM(pair, 1, give(a[16], ko));
  return pair;
  END_HANDLE_TH_ERRORS
}

// Fields of a wrapper's plan dict.
PyObject* field(PyObject* plan, const char* name) { return PyDict_GetItemString(plan, name); }
bool whole(PyObject* plan, const char* name, int64_t& v) {
  PyObject* o = field(plan, name);
  if (!o || !PyLong_CheckExact(o)) return false;
  v = PyLong_AsLongLong(o);
  return !(v == -1 && PyErr_Occurred());
}
const at::Tensor* table(PyObject* plan, const char* name, const at::Device& dev) {
  PyObject* o = field(plan, name);
  const at::Tensor* t = o ? i32(o) : nullptr;
  return t && t->device() == dev ? t : nullptr;
}
// The float32 sinks the wrapper prepared (None: none).
bool sinks_of(PyObject* o, const at::Device& dev, const float*& p) {
  p = nullptr;
  if (o == Py_None) return true;
  const at::Tensor* t = tensor(o, at::kFloat);
  if (!t || t->device() != dev || !t->is_contiguous()) return false;
  p = ptr<float>(*t);
  return true;
}

// attention_decode(plan, q, cache, kv_layout, workspace, out, sinks)
PyObject* attention_decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  SERVE(n == 7 && PyDict_CheckExact(a[0]) && !modes_active());
  const at::Tensor* q = bf16(a[1]);
  int64_t B, Hq, Hkv, D, P, splits, window;
  SERVE(q && whole(a[0], "batch", B) && whole(a[0], "Hq", Hq) && whole(a[0], "Hkv", Hkv) && whole(a[0], "D", D) &&
        whole(a[0], "P", P) && whole(a[0], "splits", splits) && whole(a[0], "window_left", window));
  const auto dev = q->device();
  const at::Tensor *ip = table(a[0], "indptr", dev), *ix = table(a[0], "indices", dev),
                   *ll = table(a[0], "last_page_len", dev);
  PyObject* so = field(a[0], "sm_scale");
  double scale;
  SERVE(ip && ix && ll && so && f64(so, scale));
  SERVE(q->dim() == 3 && q->size(0) == B && q->size(1) == Hq && q->size(2) == D && q->stride(2) == 1);
  const int nhd = layout(a[3]);
  SERVE(nhd >= 0);
  const Cache c = cache(a[2], nhd == 1, Hkv, D, dev);
  SERVE(c.ok && c.page_size == P);
  SERVE(THPVariable_CheckExact(a[4]));
  const at::Tensor& ws = THPVariable_Unpack(a[4]);
  SERVE(ws.is_cuda() && ws.unsafeGetTensorImpl()->has_storage() && !ws.key_set().has_any(kTransforms));
  const float* sinks;
  SERVE(sinks_of(a[6], dev, sinks));
  at::Tensor out;
  SERVE(output(a[5], *q, q->sizes(), out) && out.stride(2) == 1);
  void *st = stream_of(*q), *wp = ws.data_ptr();
  const int64_t wn = ws.numel() * (int64_t)ws.element_size();
  uint16_t *qp = ptr<uint16_t>(*q), *op = ptr<uint16_t>(out);
  const int32_t *ipp = ptr<int32_t>(*ip), *ixp = ptr<int32_t>(*ix), *llp = ptr<int32_t>(*ll);
  LAUNCH("pie_hip_attention_decode",
         lib.pie_hip_attention_decode(qp, q->stride(0), q->stride(1), c.k, c.v, c.page, c.slot, c.head, c.pages, ipp,
                                      ixp, llp, B, Hq, Hkv, D, P, (float)scale, window, sinks, splits, wp, wn, op,
                                      out.stride(0), out.stride(1), st));
  return give(a[5], out);
  END_HANDLE_TH_ERRORS
}

// attention_prefill(plan, q, cache, kv_layout, split address, out, sinks)
PyObject* attention_prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  SERVE(n == 7 && PyDict_CheckExact(a[0]) && !modes_active());
  const at::Tensor* q = bf16(a[1]);
  int64_t T, Hq, Hkv, D, P, mode, window, items, woff;
  SERVE(q && whole(a[0], "T", T) && whole(a[0], "Hq", Hq) && whole(a[0], "Hkv", Hkv) && whole(a[0], "D", D) &&
        whole(a[0], "P", P) && whole(a[0], "mode", mode) && whole(a[0], "window_left", window) &&
        whole(a[0], "items", items) && whole(a[0], "woff_word", woff));
  const auto dev = q->device();
  const at::Tensor *qi = table(a[0], "qo_indptr", dev), *ip = table(a[0], "indptr", dev),
                   *ix = table(a[0], "indices", dev), *ll = table(a[0], "last_page_len", dev),
                   *plan = table(a[0], "plan", dev);
  PyObject *so = field(a[0], "sm_scale"), *pk = field(a[0], "packed"), *ex = field(a[0], "extent"),
           *sc = field(a[0], "scratch");
  double scale;
  SERVE(qi && ip && ix && ll && plan && so && pk && ex && sc && f64(so, scale));
  const at::Tensor *packed = nullptr, *extent = nullptr, *scratch = tensor(sc, at::kByte);
  SERVE(scratch && scratch->device() == dev);
  if (mode == 2) {
    packed = table(a[0], "packed", dev);
    extent = table(a[0], "extent", dev);
    SERVE(packed && extent);
  }
  SERVE(q->dim() == 3 && q->size(0) == T && q->size(1) == Hq && q->size(2) == D && q->stride(2) == 1);
  const int nhd = layout(a[3]);
  SERVE(nhd >= 0);
  const Cache c = cache(a[2], nhd == 1, Hkv, D, dev);
  SERVE(c.ok && c.page_size == P);
  const int64_t* split = static_cast<const int64_t*>(PyLong_AsVoidPtr(a[4]));
  SERVE(split);
  const float* sinks;
  SERVE(sinks_of(a[6], dev, sinks));
  at::Tensor out;
  SERVE(output(a[5], *q, q->sizes(), out) && out.stride(2) == 1);
  void *st = stream_of(*q), *scp = scratch->data_ptr();
  uint16_t *qp = ptr<uint16_t>(*q), *op = ptr<uint16_t>(out);
  const int32_t *qip = ptr<int32_t>(*qi), *ipp = ptr<int32_t>(*ip), *ixp = ptr<int32_t>(*ix), *llp = ptr<int32_t>(*ll),
                *plp = ptr<int32_t>(*plan), *exp = extent ? ptr<int32_t>(*extent) : nullptr;
  const uint32_t* pkp = packed ? ptr<uint32_t>(*packed) : nullptr;
  const int64_t scn = scratch->numel();
  LAUNCH("pie_hip_attention_prefill_split",
         lib.pie_hip_attention_prefill_split(qp, q->stride(0), q->stride(1), c.k, c.v, c.page, c.slot, c.head, c.pages,
                                             qip, ipp, ixp, llp, Hq, Hkv, D, P, (float)scale, (int32_t)mode, window,
                                             sinks, pkp, exp, plp, items, woff, split, scp, scn, op, out.stride(0),
                                             out.stride(1), st));
  return give(a[5], out);
  END_HANDLE_TH_ERRORS
}

// bind({entry point name: address}, check): the loaded library's functions, and check(name, code)
// raising the library's error of a call that returned code. The calls below are compiled against one
// version of the C ABI, so a library of another is refused (ImportError).
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  if (n != 2 || !PyDict_CheckExact(a[0]) || !PyCallable_Check(a[1])) {
    PyErr_SetString(PyExc_TypeError, "bind: a dict of entry point addresses and the error check");
    return nullptr;
  }
  PyObject* d = a[0];
  Lib next;
#define X(name)                                                              \
  {                                                                          \
    PyObject* o = PyDict_GetItemString(d, #name);                            \
    void* p = o ? PyLong_AsVoidPtr(o) : nullptr;                             \
    if (!p) {                                                                \
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_KeyError, #name);         \
      return nullptr;                                                        \
    }                                                                        \
    next.name = reinterpret_cast<decltype(&::name)>(p);                      \
  }
  PIE_ENTRY_POINTS(X)
#undef X
  const int version = next.pie_hip_abi_version();
  if (version != PIE_HIP_ABI_VERSION) {
    PyErr_Format(PyExc_ImportError, "pie_amd: the native call path is built for ABI %d, the library has %d; rebuild it",
                 PIE_HIP_ABI_VERSION, version);
    return nullptr;
  }
  lib = next;
  Py_INCREF(a[1]);
  Py_XSETREF(on_error, a[1]);
  Py_RETURN_NONE;
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST(bind),
                         FAST(rmsnorm),
                         FAST(add_rms_norm),
                         FAST(act_and_mul),
                         FAST(embedding),
                         FAST(qk_rms_norm_rope_append),
                         FAST(attention_decode),
                         FAST(attention_prefill),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__fast() { return PyModule_Create(&module_def); }
