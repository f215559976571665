// Native call path of the Python ops: from torch tensors to the C ABI of libkq without the interpreter in between.
//
// What bounds it: the host.  A decode step's kernels run 5 - 15 us each, and a call through Python checks, two ctypes
// calls, a device guard and the stream lookup took 16.5 us; the same work here takes about a third.  Each function takes
// the ordinary call only -- contiguous CUDA tensors of the op's own types on the current device, no gradient wanted, no
// stream argument -- and returns None for anything else, also for anything invalid: the Python function behind it then
// converts, or raises the error it has always raised.  Outputs and workspace come from torch's caching allocator on the
// current stream, as before; nothing is kept between calls.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include "kq.h"

namespace {

// ---- the C ABI, resolved from the library the Python side has loaded
struct Abi {
#define KQ_FN(name) decltype(&::name) name
  KQ_FN(kq_last_error);
  KQ_FN(kq_codec_get);
  KQ_FN(kq_dequantize);
  KQ_FN(kq_qmm_workspace_size);
  KQ_FN(kq_qmm);
  KQ_FN(kq_gather_qmm_workspace_used);
  KQ_FN(kq_gather_qmm);
  KQ_FN(kq_moe_workspace_size);
  KQ_FN(kq_moe_glu_gather);
  KQ_FN(kq_gather_qmv);
  KQ_FN(kq_moe_glu_gather_shexp_workspace_size);
  KQ_FN(kq_moe_glu_gather_shexp);
  KQ_FN(kq_gather_qmv_mix_workspace_size);
  KQ_FN(kq_gather_qmv_mix);
  KQ_FN(kq_moe_router_topk);
  KQ_FN(kq_quantize_dev_supported);
  KQ_FN(kq_quantize_dev);
#undef KQ_FN
} abi;

kq_codec_info g_codec[KQ_NUM_CODECS];
PyObject* g_codec_ids = nullptr;    // name -> id
PyObject* g_raw_stream = nullptr;   // torch._C._cuda_getCurrentRawStream

struct Decline {};  // not an ordinary call: the Python function takes it

const at::Tensor& tensor(PyObject* o) {
  if (!THPVariable_Check(o)) throw Decline();
  return THPVariable_Unpack(o);
}
const at::Tensor* maybe_tensor(PyObject* o) { return o == Py_None ? nullptr : &tensor(o); }

int codec_id(PyObject* name) {
  PyObject* v = PyUnicode_CheckExact(name) ? PyDict_GetItem(g_codec_ids, name) : nullptr;
  if (!v) throw Decline();
  return (int)PyLong_AsLong(v);
}
int dtype_code(at::ScalarType t) {
  return t == at::kBFloat16 ? KQ_BF16 : t == at::kHalf ? KQ_F16 : t == at::kFloat ? KQ_F32 : -1;
}
// f16 or bf16 activations
int half_code(const at::Tensor& t) {
  const int c = dtype_code(t.scalar_type());
  if (c != KQ_F16 && c != KQ_BF16) throw Decline();
  return c;
}

// The device of a call: that of its first tensor, and current.
struct Call {
  c10::Device dev;
  explicit Call(const at::Tensor& t) : dev(t.device()) {
    if (!dev.is_cuda() || dev.index() != c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getDevice().index()) throw Decline();
    if (at::GradMode::is_enabled() && t.requires_grad()) throw Decline();
  }
  const at::Tensor& plain(const at::Tensor& t, int64_t dim) const {
    if (t.device() != dev || !t.is_contiguous() || (dim >= 0 && t.dim() != dim)) throw Decline();
    return t;
  }
  const at::Tensor& wire(const at::Tensor& t, int64_t dim) const {
    if (t.scalar_type() != at::kByte) throw Decline();
    return plain(t, dim);
  }
  const uint32_t* ids(const at::Tensor& t, int64_t dim) const {
    if (t.scalar_type() != at::kInt) throw Decline();
    return static_cast<const uint32_t*>(plain(t, dim).data_ptr());
  }
  const float* floats(const at::Tensor& t, int64_t dim) const {
    if (t.scalar_type() != at::kFloat) throw Decline();
    return static_cast<const float*>(plain(t, dim).data_ptr());
  }
  at::Tensor empty(at::IntArrayRef size, at::ScalarType type) const {
    return at::empty(size, at::TensorOptions().dtype(type).device(dev));
  }
  void* stream() const {
    PyObject* i = PyLong_FromLong(dev.index());
    PyObject* s = PyObject_CallOneArg(g_raw_stream, i);
    Py_DECREF(i);
    if (!s) throw python_error();
    void* p = PyLong_AsVoidPtr(s);
    Py_DECREF(s);
    return p;
  }
};

struct Workspace {
  at::Tensor t;
  void* p = nullptr;
  size_t n;
  Workspace(const Call& c, size_t bytes) : n(bytes) {
    if (bytes) {
      t = c.empty({(int64_t)bytes}, at::kByte);
      p = t.data_ptr();
    }
  }
};

// weights in a row of `bytes` wire bytes
int64_t row_weights(int codec, int64_t bytes) {
  const kq_codec_info& g = g_codec[codec];
  if (bytes % g.bytes_per_block) throw Decline();
  return bytes / g.bytes_per_block * g.weights_per_block;
}

int dim(int64_t v) {
  if (v < 0 || v > 0x7fffffff) throw Decline();
  return (int)v;
}

struct NoGil {
  PyThreadState* s = PyEval_SaveThread();
  ~NoGil() { PyEval_RestoreThread(s); }
};

PyObject* finish(int rc, at::Tensor out) {
  if (rc == KQ_OK) return THPVariable_Wrap(std::move(out));
  if (rc == KQ_ERR_INVALID) throw Decline();  // the Python function words it
  PyErr_Format(PyExc_RuntimeError, "[kq] %s", abi.kq_last_error());
  return nullptr;
}

// expert stack uint8 [E, N, bytes of K weights]
const at::Tensor& stack(const Call& c, const at::Tensor& w, int codec, int64_t K, int64_t E = -1, int64_t N = -1) {
  c.wire(w, 3);
  if (row_weights(codec, w.size(2)) != K || w.size(1) % 8 || (E >= 0 && (w.size(0) != E || w.size(1) != N))) throw Decline();
  return w;
}

// ------------------------------------------------------------------ ops
PyObject* op_qmm(PyObject* const* a) {  // x, w, codec, transpose
  const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]);
  const Call c(x);
  const int codec = codec_id(a[2]), dt = half_code(x);
  const int tr = PyObject_IsTrue(a[3]);
  if (x.dim() < 1) throw Decline();
  c.plain(x, -1);
  c.wire(w, 2);
  const int64_t wpr = row_weights(codec, w.size(1)), rows = w.size(0);
  const int K = dim(tr ? wpr : rows), N = dim(tr ? rows : wpr);
  if (K == 0 || x.size(-1) != K) throw Decline();
  const int M = dim(x.numel() / K);
  c10::SmallVector<int64_t, 5> size(x.sizes().begin(), x.sizes().end());
  size.back() = N;
  at::Tensor out = c.empty(size, x.scalar_type());
  const Workspace ws(c, abi.kq_qmm_workspace_size(M, N, K, tr, codec, dt));
  void* s = c.stream();
  int rc;
  {
    NoGil g;
    rc = abi.kq_qmm(x.data_ptr(), w.data_ptr(), out.data_ptr(), M, N, K, tr, codec, dt, ws.p, ws.n, s);
  }
  return finish(rc, std::move(out));
}

PyObject* op_dequantize(PyObject* const* a) {  // w, codec, dtype code
  const at::Tensor& w = tensor(a[0]);
  const Call c(w);
  const int codec = codec_id(a[1]), dt = (int)PyLong_AsLong(a[2]);
  c.wire(w, -1);
  if (w.dim() < 1) throw Decline();
  c10::SmallVector<int64_t, 5> size(w.sizes().begin(), w.sizes().end());
  size.back() = row_weights(codec, size.back());
  at::Tensor out = c.empty(size, dt == KQ_F32 ? at::kFloat : dt == KQ_F16 ? at::kHalf : at::kBFloat16);
  void* s = c.stream();
  int rc;
  {
    NoGil g;
    rc = abi.kq_dequantize(w.data_ptr(), out.data_ptr(), (uint64_t)out.numel(), codec, dt, s);
  }
  return finish(rc, std::move(out));
}

PyObject* op_gather_qmm(PyObject* const* a) {  // x, w, codec, lhs, rhs, transpose
  const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]), &lhs = tensor(a[3]), &rhs = tensor(a[4]);
  const Call c(x);
  const int codec = codec_id(a[2]), dt = half_code(x);
  const int tr = PyObject_IsTrue(a[5]);
  if (x.dim() < 2) throw Decline();
  c.plain(x, -1);
  c.wire(w, 3);
  const uint32_t *li = c.ids(lhs, -1), *ri = c.ids(rhs, -1);
  if (!lhs.sizes().equals(rhs.sizes())) throw Decline();
  const int64_t wpr = row_weights(codec, w.size(2));
  const int K = dim(tr ? wpr : w.size(1)), N = dim(tr ? w.size(1) : wpr), E = dim(w.size(0)), M = dim(x.size(-2));
  if (K == 0 || x.size(-1) != K) throw Decline();
  const int B = dim(lhs.numel());
  c10::SmallVector<int64_t, 5> size(lhs.sizes().begin(), lhs.sizes().end());
  size.push_back(M);
  size.push_back(N);
  at::Tensor out = c.empty(size, x.scalar_type());
  const Workspace ws(c, abi.kq_gather_qmm_workspace_used(x.data_ptr(), w.data_ptr(), B, M, E, N, K, (int64_t)M * K,
                                                           w.size(1) * w.size(2), tr, codec, dt));
  void* s = c.stream();
  int rc;
  {
    NoGil g;
    rc = abi.kq_gather_qmm(x.data_ptr(), w.data_ptr(), li, ri, out.data_ptr(), B, M, E, N, K, (int64_t)M * K,
                           w.size(1) * w.size(2), tr, 0, codec, dt, ws.p, ws.n, s);
  }
  return finish(rc, std::move(out));
}

PyObject* op_moe_glu(PyObject* const* a) {  // x, gate, up, codec, idx, act code, limit, gate bias, up bias, alpha
  const at::Tensor &x = tensor(a[0]), &gate = tensor(a[1]), &up = tensor(a[2]), &idx = tensor(a[4]);
  const at::Tensor *gb = maybe_tensor(a[7]), *ub = maybe_tensor(a[8]);
  const Call c(x);
  const int codec = codec_id(a[3]), dt = half_code(x), act = (int)PyLong_AsLong(a[5]);
  const double limit = PyFloat_AsDouble(a[6]), alpha = PyFloat_AsDouble(a[9]);
  if (PyErr_Occurred()) throw python_error();
  c.plain(x, 2);
  const int64_t K = x.size(1);
  stack(c, gate, codec, K);
  const int E = dim(gate.size(0)), N = dim(gate.size(1));
  stack(c, up, codec, K, E, N);
  const uint32_t* ids = c.ids(idx, 2);
  const int T = dim(idx.size(0)), R = dim(idx.size(1));
  if (T != x.size(0) || T == 0) throw Decline();
  const bool biased = gb || ub;
  if (act == KQ_ACT_SILU_LIMIT && !(limit > 0)) throw Decline();
  if (act == KQ_ACT_SWIGLU_CLAMP) {
    if (!gb || !ub || !(limit > 0) || !(alpha > 0) || gb->dim() != 2 || gb->size(0) != E || gb->size(1) != N ||
        !ub->sizes().equals(gb->sizes()))
      throw Decline();
  } else if (biased) {
    throw Decline();
  }
  const float *gbp = biased ? c.floats(*gb, 2) : nullptr, *ubp = biased ? c.floats(*ub, 2) : nullptr;
  at::Tensor out = c.empty({T, R, N}, x.scalar_type());
  const Workspace ws(c, abi.kq_moe_workspace_size(T, R, E, N, (int)K, 1, codec, dt));
  void* s = c.stream();
  int rc;
  {
    NoGil g;
    rc = abi.kq_moe_glu_gather(x.data_ptr(), gate.data_ptr(), up.data_ptr(), ids, gbp, ubp, out.data_ptr(), T, R, E, N,
                               (int)K, act, (float)limit, (float)alpha, codec, dt, ws.p, ws.n, s);
  }
  return finish(rc, std::move(out));
}

PyObject* op_gather_qmv(PyObject* const* a) {  // x, w, codec, idx, bias
  const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]), &idx = tensor(a[3]);
  const at::Tensor* bias = maybe_tensor(a[4]);
  const Call c(x);
  const int codec = codec_id(a[2]), dt = half_code(x);
  c.plain(x, 3);
  const int64_t K = x.size(2);
  stack(c, w, codec, K);
  const int E = dim(w.size(0)), N = dim(w.size(1));
  const uint32_t* ids = c.ids(idx, 2);
  const int T = dim(idx.size(0)), R = dim(idx.size(1));
  if (T != x.size(0) || R != x.size(1) || T == 0 || R == 0) throw Decline();
  if (bias && (bias->dim() != 2 || bias->size(0) != E || bias->size(1) != N)) throw Decline();
  const float* bp = bias ? c.floats(*bias, 2) : nullptr;
  at::Tensor out = c.empty({T, R, N}, x.scalar_type());
  const Workspace ws(c, abi.kq_moe_workspace_size(T, R, E, N, (int)K, 0, codec, dt));
  void* s = c.stream();
  int rc;
  {
    NoGil g;
    rc = abi.kq_gather_qmv(x.data_ptr(), w.data_ptr(), ids, bp, out.data_ptr(), T, R, E, N, (int)K, codec, dt, ws.p, ws.n, s);
  }
  return finish(rc, std::move(out));
}

// shared-expert matrix uint8 [N, bytes of K weights]; its codec: the stack's, or q6_k / q8_0
void shexp_row(const Call& c, const at::Tensor& w, int codec, int64_t K, int64_t N) {
  c.wire(w, 2);
  if (row_weights(codec, w.size(1)) != K || w.size(0) != N) throw Decline();
}
int shexp_codec(PyObject* name, int codec) {
  if (PyUnicode_CheckExact(name) && PyUnicode_GET_LENGTH(name) == 0) return codec;
  const int s = codec_id(name);
  const char* n = g_codec[s].name;
  if (s != codec && strcmp(n, "q6_k") && strcmp(n, "q8_0")) throw Decline();
  return s;
}

PyObject* op_moe_glu_shexp(PyObject* const* a) {  // x, gate, up, shared gate, shared up, codec, idx, act code, shared codec
  const at::Tensor &x = tensor(a[0]), &gate = tensor(a[1]), &up = tensor(a[2]), &sg = tensor(a[3]), &su = tensor(a[4]),
                   &idx = tensor(a[6]);
  const Call c(x);
  const int codec = codec_id(a[5]), dt = half_code(x), act = (int)PyLong_AsLong(a[7]), sc = shexp_codec(a[8], codec);
  if (act != KQ_ACT_SILU && act != KQ_ACT_GELU) throw Decline();
  c.plain(x, 2);
  const int64_t K = x.size(1);
  stack(c, gate, codec, K);
  const int E = dim(gate.size(0)), N = dim(gate.size(1));
  stack(c, up, codec, K, E, N);
  shexp_row(c, sg, sc, K, N);
  shexp_row(c, su, sc, K, N);
  const uint32_t* ids = c.ids(idx, 2);
  const int T = dim(idx.size(0)), R = dim(idx.size(1));
  if (T != x.size(0) || T == 0) throw Decline();
  at::Tensor out = c.empty({T, R + 1, N}, x.scalar_type());
  const size_t need = abi.kq_moe_glu_gather_shexp_workspace_size(T, R, E, N, (int)K, codec, sc, dt);
  const Workspace ws(c, need > 256 ? need : 256);
  void* s = c.stream();
  int rc;
  {
    NoGil g;
    rc = abi.kq_moe_glu_gather_shexp(x.data_ptr(), gate.data_ptr(), up.data_ptr(), sg.data_ptr(), su.data_ptr(), ids,
                                     out.data_ptr(), T, R, E, N, (int)K, act, codec, sc, dt, ws.p, need, s);
  }
  return finish(rc, std::move(out));
}

PyObject* op_mix(PyObject* const* a) {  // x, w, shared w, codec, shared codec, idx, scores
  const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]), &idx = tensor(a[5]), &scores = tensor(a[6]);
  const at::Tensor* sh = maybe_tensor(a[2]);
  const Call c(x);
  const int codec = codec_id(a[3]), dt = half_code(x), sc = sh ? shexp_codec(a[4], codec) : -1;
  c.plain(x, 3);
  const int64_t K = x.size(2);
  const int T = dim(x.size(0)), S = dim(x.size(1));
  stack(c, w, codec, K);
  const int E = dim(w.size(0)), N = dim(w.size(1));
  if (sh) shexp_row(c, *sh, sc, K, N);
  const uint32_t* ids = c.ids(idx, 2);
  const float* sp = c.floats(scores, 2);
  if (idx.size(0) != T || idx.size(1) != S - (sh ? 1 : 0) || scores.size(0) != T || scores.size(1) != S || T == 0) throw Decline();
  at::Tensor out = c.empty({T, N}, x.scalar_type());
  const size_t need = abi.kq_gather_qmv_mix_workspace_size(T, S, E, N, (int)K, codec, sc, dt);
  const Workspace ws(c, need > 256 ? need : 256);
  void* s = c.stream();
  int rc;
  {
    NoGil g;
    rc = abi.kq_gather_qmv_mix(x.data_ptr(), w.data_ptr(), sh ? sh->data_ptr() : nullptr, ids, sp, out.data_ptr(), T, S, E, N,
                               (int)K, codec, sc, dt, ws.p, need, s);
  }
  return finish(rc, std::move(out));
}

PyObject* op_router(PyObject* const* a) {  // logits, top_k, norm, shared, per-expert scale, bias, scoring code, scale
  const at::Tensor& l = tensor(a[0]);
  const at::Tensor *pes = maybe_tensor(a[4]), *bias = maybe_tensor(a[5]);
  const Call c(l);
  const int dt = dtype_code(l.scalar_type());
  const int64_t k = PyLong_AsLong(a[1]);
  const int norm = PyObject_IsTrue(a[2]), shared = PyObject_IsTrue(a[3]), scoring = (int)PyLong_AsLong(a[6]);
  const double scale = PyFloat_AsDouble(a[7]);
  if (PyErr_Occurred()) throw python_error();
  c.plain(l, 2);
  const int64_t T = l.size(0), E = l.size(1) - shared;
  if (dt < 0 || k < 1 || k > 16 || k > E || E > 1024 || (scoring == 1 && !norm) || T == 0) throw Decline();
  for (const at::Tensor* v : {pes, bias})
    if (v && (v->dim() != 1 || v->size(0) != E)) throw Decline();
  const float *pp = pes ? c.floats(*pes, 1) : nullptr, *bp = bias ? c.floats(*bias, 1) : nullptr;
  at::Tensor idx = c.empty({T, k}, at::kInt), scores = c.empty({T, k + shared}, at::kFloat);
  void* s = c.stream();
  int rc;
  {
    NoGil g;
    rc = abi.kq_moe_router_topk(l.data_ptr(), dt, dim(T), (int)E, (int)k, norm, shared, pp, bp, scoring, (float)scale,
                                static_cast<uint32_t*>(idx.data_ptr()), static_cast<float*>(scores.data_ptr()), s);
  }
  PyObject* first = finish(rc, std::move(idx));
  if (!first) return nullptr;
  PyObject* second = THPVariable_Wrap(std::move(scores));
  if (!second) {
    Py_DECREF(first);
    return nullptr;
  }
  PyObject* r = PyTuple_New(2);
  PyTuple_SET_ITEM(r, 0, first);
  PyTuple_SET_ITEM(r, 1, second);
  return r;
}

PyObject* op_quantize(PyObject* const* a) {  // w, codec, imatrix
  const at::Tensor& w = tensor(a[0]);
  const at::Tensor* im = maybe_tensor(a[2]);
  const int codec = codec_id(a[1]), dt = dtype_code(w.scalar_type());
  const c10::Device dev = w.device();
  if (w.requires_grad() || dt < 0) throw Decline();
  const Call c(w);
  const kq_codec_info& g = g_codec[codec];
  c.plain(w, -1);
  if (w.dim() < 1 || w.size(-1) == 0 || w.size(-1) % g.weights_per_block || !abi.kq_quantize_dev_supported(codec)) throw Decline();
  const int64_t K = w.size(-1);
  if (im && (im->dim() != 1 || im->size(0) != K || im->device() != dev)) throw Decline();
  const float* ip = im ? c.floats(*im, 1) : nullptr;
  c10::SmallVector<int64_t, 5> size(w.sizes().begin(), w.sizes().end());
  size.back() = K / g.weights_per_block * g.bytes_per_block;
  at::Tensor out = c.empty(size, at::kByte);
  void* s = c.stream();
  int rc;
  {
    NoGil n;
    rc = abi.kq_quantize_dev(w.data_ptr(), dt, ip, out.data_ptr(), w.numel() / K, K, codec, s);
  }
  return finish(rc, std::move(out));
}

template <PyObject* (*F)(PyObject* const*), int N>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != N) {
    PyErr_Format(PyExc_TypeError, "expected %d arguments, got %zd", N, n);
    return nullptr;
  }
  try {
    return F(args);
  } catch (const Decline&) {
    Py_RETURN_NONE;
  }
  END_HANDLE_TH_ERRORS
}

// init(handle of the loaded libkq, torch._C._cuda_getCurrentRawStream)
PyObject* init(PyObject*, PyObject* const* args, Py_ssize_t n) {
  if (n != 2) {
    PyErr_SetString(PyExc_TypeError, "init(handle, raw_stream)");
    return nullptr;
  }
  void* h = PyLong_AsVoidPtr(args[0]);
  if (PyErr_Occurred()) return nullptr;
#define KQ_FN(name)                                                          \
  abi.name = reinterpret_cast<decltype(abi.name)>(dlsym(h, #name));          \
  if (!abi.name) {                                                           \
    PyErr_SetString(PyExc_RuntimeError, "[kq] libkq has no symbol " #name);  \
    return nullptr;                                                          \
  }
  KQ_FN(kq_last_error) KQ_FN(kq_codec_get) KQ_FN(kq_dequantize) KQ_FN(kq_qmm_workspace_size) KQ_FN(kq_qmm)
  KQ_FN(kq_gather_qmm_workspace_used) KQ_FN(kq_gather_qmm) KQ_FN(kq_moe_workspace_size) KQ_FN(kq_moe_glu_gather)
  KQ_FN(kq_gather_qmv) KQ_FN(kq_moe_glu_gather_shexp_workspace_size) KQ_FN(kq_moe_glu_gather_shexp)
  KQ_FN(kq_gather_qmv_mix_workspace_size) KQ_FN(kq_gather_qmv_mix) KQ_FN(kq_moe_router_topk)
  KQ_FN(kq_quantize_dev_supported) KQ_FN(kq_quantize_dev)
#undef KQ_FN
  PyObject* ids = PyDict_New();
  if (!ids) return nullptr;
  for (int i = 0; i < KQ_NUM_CODECS; i++) {
    abi.kq_codec_get(i, &g_codec[i]);
    PyObject* v = PyLong_FromLong(i);
    PyDict_SetItemString(ids, g_codec[i].name, v);
    Py_XDECREF(v);
  }
  Py_INCREF(args[1]);
  Py_XDECREF(g_raw_stream);
  g_raw_stream = args[1];
  Py_XDECREF(g_codec_ids);
  g_codec_ids = ids;
  Py_RETURN_NONE;
}

#define KQ_METHOD(name, f, n) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&entry<f, n>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    {"init", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(&init)), METH_FASTCALL, nullptr},
    KQ_METHOD("qmm", op_qmm, 4),
    KQ_METHOD("dequantize", op_dequantize, 3),
    KQ_METHOD("gather_qmm", op_gather_qmm, 6),
    KQ_METHOD("moe_glu", op_moe_glu, 10),
    KQ_METHOD("gather_qmv", op_gather_qmv, 5),
    KQ_METHOD("moe_glu_shexp", op_moe_glu_shexp, 9),
    KQ_METHOD("mix", op_mix, 7),
    KQ_METHOD("router", op_router, 8),
    KQ_METHOD("quantize", op_quantize, 3),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_kqhost", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__kqhost() { return PyModule_Create(&module); }
