// CPython module of the calls that a decoder layer makes per step: Attention.forward
// (nanovllm/layers/attention.py:58-79) and qk_norm_rope (qwen3.py:91-105) from their
// Python arguments to the C ABI's launches.
//
// A small call is bound by the host: with the checks, tensor creations and ctypes
// conversions in Python, a decode of one sequence took 30 us for 10 us of kernels; here
// the whole call costs 10.2 us, little more than its two launches.
//
// Every function takes the ordinary form of its arguments -- plain dense GPU tensors of the
// documented types, shapes and strides on one device, no dispatch or function mode -- and
// returns None, having launched nothing it should not have, for everything else and for
// every status but success.  The caller then runs the general Python path, which raises
// the documented error or handles the form; a store done before that is done again.
#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <cstring>

#include "nva_attention.h"

namespace {

// The C ABI of the library that the Python side loaded.
struct Abi {
  decltype(&nva_store_kvcache) store_kvcache;
  decltype(&nva_prefill) prefill;
  decltype(&nva_prefill_fp8) prefill_fp8;
  decltype(&nva_store_prefill) store_prefill;
  decltype(&nva_decode_workspace_bytes) decode_workspace_bytes;
  decltype(&nva_decode) decode;
  decltype(&nva_store_decode) store_decode;
  decltype(&nva_store_then_decode) store_then_decode;
  decltype(&nva_qk_norm_rope) qk_norm_rope;
} abi{};
bool bound = false;

// Tensors that are not what their memory holds: wrappers, views with a pending operation,
// batches of a transform, functional and fake tensors.
bool plain(const at::Tensor& t) {
  static const c10::DispatchKeySet wrapped({
      c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
      c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::FuncTorchVmapMode, c10::DispatchKey::BatchedNestedTensor,
      c10::DispatchKey::Batched, c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate,
      c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
  return t.defined() && t.is_cuda() && t.layout() == at::kStrided && !t.is_nested() && !t.key_set().has_any(wrapped);
}

// A tensor argument, or null where it is not a plain tensor.
const at::Tensor* tensor(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  return plain(t) ? &t : nullptr;
}

bool modes_active() {
  return c10::impl::TorchDispatchModeTLS::any_modes_set() || at::impl::torch_function_mode_enabled() ||
         at::tracer::impl::is_dispatch_enabled();
}

bool to_int(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool to_float(PyObject* o, double& v) {
  if (!PyFloat_CheckExact(o)) return false;
  v = PyFloat_AS_DOUBLE(o);
  return true;
}

// bf16 rows of `heads` heads of `d`: (T, heads * d) or (T, heads, d), contiguous inside a row.
bool head_rows(const at::Tensor& t, int64_t heads, int64_t d) {
  if (t.scalar_type() != at::kBFloat16) return false;
  if (t.dim() == 2) return t.size(1) == heads * d && t.stride(1) == 1;
  return t.dim() == 3 && t.size(1) == heads && t.size(2) == d && t.stride(2) == 1 && t.stride(1) == d;
}

bool index_vector(const at::Tensor& t, int64_t n) {
  return t.scalar_type() == at::kInt && t.numel() == n && t.is_contiguous();
}

template <class T>
const T* data(const at::Tensor* t) {
  return t ? static_cast<const T*>(t->const_data_ptr()) : nullptr;
}

constexpr int64_t kMax32 = 0x7fffffff;

PyObject* none() { Py_RETURN_NONE; }

// bind(addresses): the entry points in Abi's order.
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
  constexpr Py_ssize_t kEntries = sizeof(Abi) / sizeof(void*);
  void* at[kEntries];
  if (n != kEntries) {
    PyErr_SetString(PyExc_TypeError, "bind takes the addresses of the library's entry points");
    return nullptr;
  }
  for (Py_ssize_t i = 0; i < n; ++i) {
    at[i] = PyLong_AsVoidPtr(args[i]);
    if (!at[i]) {
      if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null entry point");
      return nullptr;
    }
  }
  memcpy(&abi, at, sizeof(abi));
  bound = true;
  return none();
}

// attention(q, k, v, k_cache, v_cache, k_scale, v_scale, num_heads, num_kv_heads, head_dim, scale, fuse_store,
//           is_prefill, cu_seqlens_q, cu_seqlens_k, max_seqlen_q, max_seqlen_k, slot_mapping, context_lens,
//           block_tables, prefill_workspaces, fp8_in_place_tokens) -> (T, num_heads * head_dim) or None
// prefill_workspaces: {(device, stream): uint8 tensor}.
PyObject* attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 22 || !bound || modes_active()) return none();
  const at::Tensor *q = tensor(a[0]), *k = tensor(a[1]), *v = tensor(a[2]), *kc = tensor(a[3]), *vc = tensor(a[4]);
  if (!q || !k || !v || !kc || !vc) return none();
  const at::Tensor *ks = nullptr, *vs = nullptr;
  if (a[5] != Py_None && !(ks = tensor(a[5]))) return none();
  if (a[6] != Py_None && !(vs = tensor(a[6]))) return none();
  int64_t nh, nkv, d;
  double scale;
  if (!to_int(a[7], nh) || !to_int(a[8], nkv) || !to_int(a[9], d) || !to_float(a[10], scale)) return none();
  if (nh <= 0 || nkv <= 0 || d <= 0 || nh > kMax32 || nkv > kMax32 || d > kMax32) return none();
  if (!PyBool_Check(a[11]) || !PyBool_Check(a[12])) return none();
  const bool fuse = a[11] == Py_True, is_prefill = a[12] == Py_True;
  const at::Tensor *slots = tensor(a[17]), *bt = nullptr;
  if (!slots) return none();
  if (a[19] != Py_None && !(bt = tensor(a[19]))) return none();

  if (!head_rows(*q, nh, d) || !head_rows(*k, nkv, d) || !head_rows(*v, nkv, d)) return none();
  const int64_t T = q->size(0), N = k->size(0);
  if (v->size(0) != N || T == 0 || N == 0 || T > kMax32 || N > kMax32 || !index_vector(*slots, N)) return none();
  if (kc->dim() != 4 || kc->sizes() != vc->sizes() || kc->size(2) != nkv || kc->size(3) != d || kc->numel() == 0 ||
      !kc->is_contiguous() || !vc->is_contiguous() || kc->stride(1) != nkv * d || vc->stride(1) != nkv * d)
    return none();
  const int64_t num_blocks = kc->size(0), block_size = kc->size(1);
  if (block_size > kMax32) return none();
  auto dtype_code = [](const at::Tensor& c) {
    if (c.scalar_type() == at::kBFloat16) return NVA_DTYPE_BF16;
    return c.scalar_type() == at::kFloat8_e4m3fn || c.scalar_type() == at::kByte ? NVA_DTYPE_FP8_E4M3 : -1;
  };
  const int code = dtype_code(*kc);
  if (code < 0 || dtype_code(*vc) != code) return none();
  const bool fp8 = code == NVA_DTYPE_FP8_E4M3;
  for (const at::Tensor* s : {ks, vs})
    if (fp8 && (!s || s->scalar_type() != at::kFloat || s->numel() != nkv || !s->is_contiguous())) return none();
  const c10::Device dev = q->device();
  for (const at::Tensor* t : {k, v, kc, vc, ks, vs, slots, bt})
    if (t && t->device() != dev) return none();
  if (bt && (bt->scalar_type() != at::kInt || bt->dim() != 2 || bt->stride(1) != 1 || bt->size(1) > kMax32)) return none();
  void* const stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  const float sc = static_cast<float>(scale);
  const auto opt = q->options();
  int rc;

  if (!is_prefill) {
    const at::Tensor* lens = tensor(a[18]);
    if (!lens || !bt || lens->device() != dev || !index_vector(*lens, T) || bt->size(0) != T) return none();
    if (fuse && N != T) return none();
    const int64_t ws_bytes =
        abi.decode_workspace_bytes(static_cast<int32_t>(T), static_cast<int32_t>(nh), static_cast<int32_t>(nkv),
                                   static_cast<int32_t>(d), static_cast<int32_t>(bt->size(1)),
                                   static_cast<int32_t>(block_size), code, 0);
    at::Tensor out = at::empty({T, nh * d}, opt), ws;
    if (ws_bytes > 0) ws = at::empty({ws_bytes}, opt.dtype(at::kByte));
    void* const wsp = ws_bytes > 0 ? ws.mutable_data_ptr() : nullptr;
    void *op = out.mutable_data_ptr(), *kp = kc->mutable_data_ptr(), *vp = vc->mutable_data_ptr();
    Py_BEGIN_ALLOW_THREADS
    if (N == T) {
      rc = (fuse ? abi.store_decode : abi.store_then_decode)(
          data<void>(k), k->stride(0), data<void>(v), v->stride(0), data<int32_t>(slots), data<void>(q), q->stride(0),
          kp, vp, code, data<float>(ks), data<float>(vs), num_blocks, data<int32_t>(lens), data<int32_t>(bt),
          bt->stride(0), static_cast<int32_t>(bt->size(1)), static_cast<int32_t>(block_size), static_cast<int32_t>(T),
          static_cast<int32_t>(nh), static_cast<int32_t>(nkv), static_cast<int32_t>(d), sc, 0, op, nh * d, wsp, ws_bytes,
          stream);
    } else {
      rc = abi.store_kvcache(data<void>(k), k->stride(0), data<void>(v), v->stride(0), kp, vp, num_blocks * block_size,
                             data<int32_t>(slots), N, static_cast<int32_t>(nkv), static_cast<int32_t>(d), code,
                             data<float>(ks), data<float>(vs), stream);
      if (rc == NVA_OK)
        rc = abi.decode(data<void>(q), q->stride(0), kp, vp, code, data<float>(ks), data<float>(vs), num_blocks,
                        data<int32_t>(lens), data<int32_t>(bt), bt->stride(0), static_cast<int32_t>(bt->size(1)),
                        static_cast<int32_t>(block_size), static_cast<int32_t>(T), static_cast<int32_t>(nh),
                        static_cast<int32_t>(nkv), static_cast<int32_t>(d), sc, 0, op, nh * d, wsp, ws_bytes, stream);
    }
    Py_END_ALLOW_THREADS
    if (rc != NVA_OK) return none();
    return THPVariable_Wrap(std::move(out));
  }

  const at::Tensor *cq = tensor(a[13]), *ck = tensor(a[14]);
  int64_t mq, mk, in_place;
  if (!cq || !ck || !to_int(a[15], mq) || !to_int(a[16], mk) || !to_int(a[21], in_place)) return none();
  const int64_t S = cq->numel() - 1;
  if (S < 1 || S > kMax32 || mq < 0 || mq > kMax32 || mk < 0 || mk > kMax32 || cq->device() != dev || ck->device() != dev ||
      !index_vector(*cq, S + 1) || !index_vector(*ck, S + 1))
    return none();
  if (bt && (bt->size(0) != S || (fp8 && !(d == 128 && block_size % 64 == 0 && mq <= in_place)))) return none();
  if (!PyDict_CheckExact(a[20])) return none();
  PyObject* key = Py_BuildValue("(iL)", static_cast<int>(dev.index()),
                                static_cast<long long>(reinterpret_cast<intptr_t>(stream)));
  if (!key) return nullptr;
  PyObject* held = PyDict_GetItemWithError(a[20], key);  // borrowed
  Py_DECREF(key);
  if (!held) {
    if (PyErr_Occurred()) return nullptr;
    return none();  // the general path makes the workspace
  }
  const at::Tensor* ws = tensor(held);
  if (!ws || ws->device() != dev) return none();
  at::Tensor keep = *ws;  // another thread may drop the dict's reference while this one launches
  at::Tensor out = at::empty({T, nh * d}, opt);
  void *op = out.mutable_data_ptr(), *kp = kc->mutable_data_ptr(), *vp = vc->mutable_data_ptr(),
       *wsp = keep.mutable_data_ptr();
  const int64_t ws_bytes = keep.numel();
  Py_BEGIN_ALLOW_THREADS
  if (!bt) {
    rc = abi.store_prefill(kp, vp, num_blocks * block_size, data<int32_t>(slots), N, code, data<float>(ks),
                           data<float>(vs), data<void>(q), q->stride(0), T, data<void>(k), k->stride(0), data<void>(v),
                           v->stride(0), data<int32_t>(cq), data<int32_t>(ck), static_cast<int32_t>(S),
                           static_cast<int32_t>(mq), static_cast<int32_t>(mk), static_cast<int32_t>(nh),
                           static_cast<int32_t>(nkv), static_cast<int32_t>(d), sc, op, nh * d, wsp, ws_bytes, stream);
  } else {
    rc = abi.store_kvcache(data<void>(k), k->stride(0), data<void>(v), v->stride(0), kp, vp, num_blocks * block_size,
                           data<int32_t>(slots), N, static_cast<int32_t>(nkv), static_cast<int32_t>(d), code,
                           data<float>(ks), data<float>(vs), stream);
    if (rc == NVA_OK && fp8)
      rc = abi.prefill_fp8(data<void>(q), q->stride(0), kp, vp, data<float>(ks), data<float>(vs), data<int32_t>(bt),
                           bt->stride(0), static_cast<int32_t>(bt->size(1)), static_cast<int32_t>(block_size), num_blocks,
                           data<int32_t>(cq), data<int32_t>(ck), static_cast<int32_t>(S), static_cast<int32_t>(mq),
                           static_cast<int32_t>(mk), static_cast<int32_t>(nh), static_cast<int32_t>(nkv),
                           static_cast<int32_t>(d), sc, op, nh * d, wsp, ws_bytes, stream);
    else if (rc == NVA_OK)
      rc = abi.prefill(data<void>(q), q->stride(0), kp, nkv * d, vp, nkv * d, data<int32_t>(bt), bt->stride(0),
                       static_cast<int32_t>(bt->size(1)), static_cast<int32_t>(block_size), num_blocks,
                       data<int32_t>(cq), data<int32_t>(ck), static_cast<int32_t>(S), static_cast<int32_t>(mq),
                       static_cast<int32_t>(mk), static_cast<int32_t>(nh), static_cast<int32_t>(nkv),
                       static_cast<int32_t>(d), sc, op, nh * d, wsp, ws_bytes, stream);
  }
  Py_END_ALLOW_THREADS
  if (rc != NVA_OK) return none();
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// qk_norm_rope(positions, q, k, cos_sin_cache, num_heads, num_kv_heads, head_dim, q_norm_weight, k_norm_weight, eps)
//   -> (q, k) in new tensors of the arguments' shapes, or None
PyObject* qk_norm_rope(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  if (n != 10 || !bound || modes_active()) return none();
  const at::Tensor *pos = tensor(a[0]), *q = tensor(a[1]), *k = tensor(a[2]), *cs = tensor(a[3]);
  if (!pos || !q || !k || !cs) return none();
  int64_t nh, nkv, d;
  double eps;
  if (!to_int(a[4], nh) || !to_int(a[5], nkv) || !to_int(a[6], d) || !to_float(a[9], eps)) return none();
  if (nh <= 0 || nkv <= 0 || d <= 0 || nh > kMax32 || nkv > kMax32 || d > kMax32) return none();
  if (!head_rows(*q, nh, d) || !head_rows(*k, nkv, d)) return none();
  const int64_t T = q->size(0);
  const c10::Device dev = q->device();
  if (T == 0 || k->size(0) != T || pos->scalar_type() != at::kLong || pos->dim() != 1 || pos->size(0) != T ||
      !pos->is_contiguous() || cs->scalar_type() != at::kFloat || cs->dim() != 2 || cs->size(1) != d ||
      !cs->is_contiguous())
    return none();
  const at::Tensor* w[2] = {nullptr, nullptr};
  if ((a[7] == Py_None) != (a[8] == Py_None)) return none();
  if (a[7] != Py_None)
    for (int i = 0; i < 2; ++i) {
      w[i] = tensor(a[7 + i]);
      if (!w[i] || w[i]->scalar_type() != at::kBFloat16 || w[i]->dim() != 1 || w[i]->size(0) != d || !w[i]->is_contiguous())
        return none();
    }
  for (const at::Tensor* t : {pos, k, cs, w[0], w[1]})
    if (t && t->device() != dev) return none();
  at::Tensor qo = at::empty(q->sizes(), q->options()), ko = at::empty(k->sizes(), k->options());
  void *qp = qo.mutable_data_ptr(), *kp = ko.mutable_data_ptr();
  void* const stream = c10::hip::getCurrentHIPStream(dev.index()).stream();
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = abi.qk_norm_rope(data<void>(q), q->stride(0), data<void>(k), k->stride(0), qp, nh * d, kp, nkv * d,
                        data<void>(w[0]), data<void>(w[1]), static_cast<float>(eps), data<float>(cs), cs->size(0),
                        data<int64_t>(pos), T, static_cast<int32_t>(nh), static_cast<int32_t>(nkv),
                        static_cast<int32_t>(d), stream);
  Py_END_ALLOW_THREADS
  if (rc != NVA_OK) return none();
  PyObject* pair = PyTuple_New(2);
  if (!pair) return nullptr;
  PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(std::move(qo)));
  PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(std::move(ko)));
  return pair;
  END_HANDLE_TH_ERRORS
}

#define NVA_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f))
PyMethodDef methods[] = {
    {"bind", NVA_FAST(bind), METH_FASTCALL, "Entry points of the loaded library."},
    {"attention", NVA_FAST(attention), METH_FASTCALL, "Attention.forward's ordinary form, or None."},
    {"qk_norm_rope", NVA_FAST(qk_norm_rope), METH_FASTCALL, "qk_norm_rope's ordinary form, or None."},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_nva_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__nva_host() {
  PyObject* m = PyModule_Create(&module);
  // the torch whose C++ ABI this was compiled against; the loader compares it
  if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) Py_CLEAR(m);
  return m;
}
