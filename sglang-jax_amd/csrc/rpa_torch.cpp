// Host path of the Python operators in native code: one attention call = read the arguments, allocate the output,
// fill the C struct, launch.  Python spends 25 us on that for a call whose kernels take 8; here it is 2 us plus the
// launches, which is what a decode step of a small model is made of (28 layers, 8 rows of a few hundred tokens:
// 1000 us of host time per step before).
//
// Only calls in their common form are taken (device tensors of the right types and shapes, contiguous, options in
// range).  Anything else -- other query types, narrow cache rows, host metadata, a wrong argument -- makes these
// functions return None, and the general code in Python converts, or words the error.  Nothing is kept between calls
// but the split-KV workspace, one grow-only buffer per (device, stream).

#include <ATen/ATen.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <map>
#include <utility>
#include <vector>

#include "../../include/rpa.h"

namespace {

// ---- the workspace, shared with the Python side (`workspace()` below); the map is touched under the GIL only.  A call holds
// on to the buffer it was given: without the GIL, while it launches, another thread's call on the same stream may grow it.
at::Tensor workspace(const at::Device& dev, void* stream, size_t bytes) {
  static auto* pool = new std::map<std::pair<int, void*>, at::Tensor>;  // never destroyed: tensors outlive no device
  at::Tensor& t = (*pool)[{dev.index(), stream}];
  if (!t.defined() || (size_t)t.numel() < bytes)
    t = at::empty({(int64_t)std::max<size_t>(bytes, 1 << 20)}, at::TensorOptions().dtype(at::kByte).device(dev));
  return t;
}

// ---- readers of one argument: false = not in the common form
bool none(PyObject* o) { return o == nullptr || o == Py_None; }

const at::Tensor* tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

const at::Tensor* on_device(PyObject* o, const at::Device& dev, at::ScalarType type) {
  const at::Tensor* t = tensor(o);
  return t && t->device() == dev && t->scalar_type() == type && t->is_contiguous() ? t : nullptr;
}

bool real(PyObject* o, double& v) {
  v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

bool whole(PyObject* o, int64_t& v) {
  if (PyLong_Check(o)) {
    v = PyLong_AsLongLong(o);
  } else {
    PyObject* n = PyNumber_Index(o);
    v = n ? PyLong_AsLongLong(n) : -1;
    Py_XDECREF(n);
  }
  if (v == -1 && PyErr_Occurred()) PyErr_Clear();
  else return v >= INT32_MIN && v <= INT32_MAX;
  return false;
}

// None -> `off`, else a number that has to be positive
bool positive(PyObject* o, float& v, float off = 0.f) {
  double d;
  if (none(o)) {
    v = off;
    return true;
  }
  if (!real(o, d) || !(d > 0)) return false;
  v = (float)d;
  return true;
}

bool bound(PyObject* o, int32_t& v) {  // None -> 0
  int64_t n = 0;
  if (!none(o) && !whole(o, n)) return false;
  v = (int32_t)n;
  return true;
}

// A host array of 32- or 64-bit integers (numpy, through the buffer protocol)
struct HostInts {
  Py_buffer b{};
  bool held = false;
  bool open(PyObject* o) {
    if (PyObject_GetBuffer(o, &b, PyBUF_FORMAT | PyBUF_C_CONTIGUOUS) != 0) {
      PyErr_Clear();
      return false;
    }
    held = true;
    const char f = b.format ? b.format[0] : 0;
    return b.ndim == 1 && b.format && b.format[1] == 0 && (b.itemsize == 4 || b.itemsize == 8) &&
           (f == 'i' || f == 'l' || f == 'q');
  }
  int64_t size() const { return b.len / b.itemsize; }
  int64_t at(int64_t i) const {
    return b.itemsize == 4 ? static_cast<const int32_t*>(b.buf)[i] : static_cast<const int64_t*>(b.buf)[i];
  }
  ~HostInts() {
    if (held) PyBuffer_Release(&b);
  }
};

// distribution: a device tensor (composition read by the kernels) or three host numbers
struct Distribution {
  const int32_t* device = nullptr;
  int64_t i = 0, j = 0, k = 0;
  bool read(PyObject* o, const at::Device& dev) {
    if (const at::Tensor* t = tensor(o)) {
      if (t->dim() != 1 || t->size(0) != 3 || t->scalar_type() != at::kInt || !t->is_contiguous()) return false;
      if (t->device() == dev) {
        device = t->const_data_ptr<int32_t>();
        return true;
      }
      if (!t->is_cpu()) return false;
      const int32_t* v = t->const_data_ptr<int32_t>();
      i = v[0], j = v[1], k = v[2];
    } else if (PyTuple_CheckExact(o) || PyList_CheckExact(o)) {
      if (PySequence_Fast_GET_SIZE(o) != 3) return false;
      PyObject** v = PySequence_Fast_ITEMS(o);
      if (!whole(v[0], i) || !whole(v[1], j) || !whole(v[2], k)) return false;
    } else {
      HostInts h;
      if (!h.open(o) || h.size() != 3 || h.b.itemsize != 4) return false;
      i = h.at(0), j = h.at(1), k = h.at(2);
    }
    return 0 <= i && i <= j && j <= k;
  }
};

// The softmax types as Python holds them: 0 f32, 1 bf16, 2 f16, -1 another
int softmax_code(PyObject* o) {
  if (none(o)) return RPA_SOFTMAX_F32;
  if (!THPDtype_Check(o)) return -1;
  switch (reinterpret_cast<THPDtype*>(o)->scalar_type) {
    case at::kFloat: return RPA_SOFTMAX_F32;
    case at::kBFloat16: return RPA_SOFTMAX_BF16;
    case at::kHalf: return RPA_SOFTMAX_F16;
    default: return -1;
  }
}

void* stream_of(const at::Device& dev) { return c10::hip::getCurrentHIPStream(dev.index()).stream(); }

template <typename F>
int without_gil(F f) {
  PyThreadState* s = PyEval_SaveThread();
  const int rc = f();
  PyEval_RestoreThread(s);
  return rc;
}

#define COMMON(cond) \
  if (!(cond)) Py_RETURN_NONE

// attention(q, k, v, cache, kv_lens, page_indices, cu_q_lens, cu_kv_lens, distribution, attention_sink, causal, sm_scale,
//           sliding_window, soft_cap, mask_value, q_scale, k_scale, v_scale, xai_temperature_len, softmax_dtype,
//           chunk_prefill_size, max_kv_len, max_q_len, num_splits, host_kv_lens, head_dim, custom_mask, mask_aligned,
//           prompts_only)
// -> output, a status below 0, or None.  head_dim 0: q, k, v are [T, heads, D]; else they may be [T, heads * D], and
// so is the output.  custom_mask is read where causal is false.
PyObject* attention(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 29) {
    PyErr_SetString(PyExc_TypeError, "attention takes 29 arguments");
    return nullptr;
  }
  const at::Tensor* q = tensor(a[0]);
  const at::Tensor* cache = tensor(a[3]);
  COMMON(q && cache && q->is_cuda() && q->scalar_type() == at::kBFloat16 && q->is_contiguous());
  const at::Device dev = q->device();
  const at::ScalarType kv_type = cache->scalar_type();
  COMMON(cache->device() == dev && cache->dim() == 4 && cache->is_contiguous() &&
         (kv_type == at::kBFloat16 || kv_type == at::kFloat8_e4m3fn));
  int64_t head_dim;
  COMMON(whole(a[25], head_dim));
  const int64_t D = cache->size(3), T = q->size(0), Hkv = cache->size(2) / 2;
  COMMON((D == 128 || D == 256) && (q->dim() == 2 || q->dim() == 3));
  // rows narrower than the cache's (which end in zeros)
  const int64_t row = q->dim() == 3 ? q->size(2) : head_dim;
  COMMON(row > 0 && row <= D && D - row < 128 && row % (kv_type == at::kBFloat16 ? 8 : 16) == 0);
  int64_t Hq;
  if (q->dim() == 3) {
    COMMON(head_dim == 0 || head_dim == row);
    Hq = q->size(1);
  } else {
    COMMON(q->size(1) % row == 0);
    Hq = q->size(1) / row;
  }
  COMMON(Hkv > 0 && cache->size(2) % 2 == 0 && Hq > 0 && Hq % Hkv == 0);

  at::Tensor keys, values;  // hold contiguous copies where the caller's are none
  if (!none(a[1])) {
    const at::Tensor *k = tensor(a[1]), *v = tensor(a[2]);
    COMMON(k && v && k->device() == dev && v->device() == dev && k->scalar_type() == kv_type &&
           v->scalar_type() == kv_type && k->sizes() == v->sizes() && k->dim() == q->dim() && k->size(0) == T);
    COMMON(k->dim() == 3 ? (k->size(1) == Hkv && k->size(2) == row) : k->size(1) == Hkv * row);
    keys = k->contiguous();
    values = v->contiguous();
  } else {
    COMMON(none(a[2]));
  }

  const at::Tensor* kv_lens = on_device(a[4], dev, at::kInt);
  const at::Tensor* pages = on_device(a[5], dev, at::kInt);
  const at::Tensor* cu_q = on_device(a[6], dev, at::kInt);
  const at::Tensor* cu_kv = on_device(a[7], dev, at::kInt);
  COMMON(kv_lens && pages && cu_q && cu_kv && kv_lens->dim() == 1 && pages->dim() == 1 && cu_q->dim() == 1 &&
         cu_kv->dim() == 1);
  const int64_t S = kv_lens->size(0);
  COMMON(cu_q->size(0) == S + 1 && cu_kv->size(0) == S + 1);
  Distribution dist;
  COMMON(dist.read(a[8], dev) && dist.k <= S);

  RpaParams p = {};
  if (!none(a[9])) {
    const at::Tensor* sink = on_device(a[9], dev, at::kFloat);
    COMMON(sink && sink->numel() == Hq);
    p.attention_sink = sink->const_data_ptr<float>();
  }
  const int causal = PyObject_IsTrue(a[10]);
  COMMON(causal >= 0);
  p.mask_mode = causal ? RPA_MASK_CAUSAL : RPA_MASK_NONE;
  if (!causal && !none(a[26])) {
    const at::Tensor* mask = on_device(a[26], dev, at::kInt);
    const int aligned = PyObject_IsTrue(a[27]);
    COMMON(mask && aligned >= 0);
    p.mask_mode = RPA_MASK_CUSTOM;
    p.custom_mask = mask->const_data_ptr<int32_t>();
    p.mask_rows_page_aligned = aligned;
  }
  double d;
  COMMON(real(a[11], d));
  p.sm_scale = (float)d;
  int64_t n;
  if (!none(a[12])) {
    COMMON(whole(a[12], n) && n > 0);
    p.sliding_window = (int32_t)n;
  }
  if (!none(a[13])) {
    COMMON(real(a[13], d) && d != 0.0);
    p.soft_cap = (float)d;
  }
  if (!none(a[14])) {
    COMMON(real(a[14], d));
    p.mask_value = (float)d;
  }
  COMMON(positive(a[15], p.q_scale));
  for (int s = 0; s < 2; ++s) {
    if (none(a[16 + s])) continue;
    const at::Tensor* t = on_device(a[16 + s], dev, at::kFloat);
    COMMON(t && t->numel() == Hkv);
    (s ? p.v_scale : p.k_scale) = t->const_data_ptr<float>();
  }
  COMMON(positive(a[18], p.xai_temperature_len));
  p.softmax_dtype = softmax_code(a[19]);
  COMMON(p.softmax_dtype >= 0);
  int32_t chunk;
  COMMON(bound(a[20], chunk) && (none(a[20]) || chunk > 0));

  // host-side bounds: from the caller, or from the host copy of the lengths
  p.decode_end = (int32_t)dist.i;
  p.num_seqs = dist.device ? (int32_t)S : (int32_t)dist.k;
  if (!none(a[24])) {
    HostInts lens;
    COMMON(lens.open(a[24]));
    const int64_t count = lens.size(), rows = std::min(count, dist.device ? 0 : dist.i);
    int64_t sum = 0, most = 0;
    for (int64_t s = 0; s < count; ++s) {
      const int64_t x = lens.at(s);
      if (s < rows) sum += x;
      most = std::max(most, x);
    }
    p.sum_decode_kv_len = sum;
    p.max_kv_len = (int32_t)std::min<int64_t>(most, INT32_MAX);
  }
  if (!none(a[21])) COMMON(bound(a[21], p.max_kv_len));
  if (!none(a[22])) {
    COMMON(bound(a[22], p.max_q_len));
  } else if (!dist.device && chunk > 0 && dist.j == dist.k) {
    p.max_q_len = chunk;  // sequences of the MIXED partition [j, k) may be of any length
  }
  COMMON(bound(a[23], p.num_splits));

  at::Tensor out = at::empty_like(*q);
  void* stream = stream_of(dev);
  p.q = q->const_data_ptr();
  p.out = out.data_ptr();
  p.kv_cache = cache->const_data_ptr();
  p.kv_lens = kv_lens->const_data_ptr<int32_t>();
  p.page_indices = pages->const_data_ptr<int32_t>();
  p.cu_q_lens = cu_q->const_data_ptr<int32_t>();
  p.cu_kv_lens = cu_kv->const_data_ptr<int32_t>();
  p.distribution = dist.device;
  p.num_tokens = (int32_t)T;
  p.num_q_heads = (int32_t)Hq;
  p.num_kv_heads = (int32_t)Hkv;
  p.head_dim = (int32_t)D;
  p.q_head_dim = (int32_t)row;
  p.page_size = (int32_t)cache->size(1);
  p.total_pages = (int32_t)cache->size(0);
  p.layout = RPA_LAYOUT_FUSED | RPA_PARAMS_TAIL;
  p.kv_dtype = kv_type == at::kBFloat16 ? RPA_KV_BF16 : RPA_KV_FP8_E4M3;
  COMMON(!rpa_mask_needs_starts(&p));
  p.prompts_only = keys.defined() && PyObject_IsTrue(a[28]) == 1;
  at::Tensor ws;
  if (const size_t need = rpa_workspace_bytes(&p)) {
    ws = workspace(dev, stream, need);
    p.workspace = ws.data_ptr();
    p.workspace_bytes = (size_t)ws.numel();
  }
  const void* kp = keys.defined() ? keys.const_data_ptr() : nullptr;
  const void* vp = values.defined() ? values.const_data_ptr() : nullptr;
  const int rc = without_gil([&] { return rpa_attention_update(&p, kp, vp, stream); });
  if (rc != RPA_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// The tensors of an absorbed-MLA call: queries, latent cache, new rows.
struct MlaTensors {
  const at::Tensor *q, *q_pe, *cache;
  at::Tensor new_c, new_r;
  // false: not in the common form
  bool read(PyObject* const* a, RpaMlaParams& p) {
    q = tensor(a[0]), q_pe = tensor(a[1]), cache = tensor(a[4]);
    if (!(q && q_pe && cache && q->is_cuda())) return false;
    const at::Device dev = q->device();
    const at::ScalarType kv_type = cache->scalar_type();
    if (!(q->scalar_type() == at::kBFloat16 && q_pe->scalar_type() == at::kBFloat16 && q->dim() == 3 && q_pe->dim() == 3 &&
          q->is_contiguous() && q_pe->is_contiguous() && q_pe->device() == dev && q->size(0) == q_pe->size(0) &&
          q->size(1) == q_pe->size(1)))
      return false;
    if (!(cache->device() == dev && cache->is_contiguous() && (cache->dim() == 3 || cache->dim() == 4) &&
          (kv_type == at::kBFloat16 || kv_type == at::kFloat8_e4m3fn)))
      return false;
    const int64_t T = q->size(0), lkv = q->size(2), rope = q_pe->size(2), width = cache->size(-1);
    if (width == lkv + rope) p.rope_offset = (int32_t)lkv;
    else if (width == (lkv + 127) / 128 * 128 + (rope + 127) / 128 * 128) p.rope_offset = (int32_t)((lkv + 127) / 128 * 128);
    else return false;
    if (!none(a[2])) {
      const at::Tensor *c = tensor(a[2]), *r = tensor(a[3]);
      if (!(c && r && c->device() == dev && r->device() == dev && c->scalar_type() == kv_type && r->scalar_type() == kv_type &&
            c->dim() == 2 && r->dim() == 2 && c->size(0) == T && r->size(0) == T && c->size(1) == lkv && r->size(1) == rope))
        return false;
      new_c = c->contiguous();
      new_r = r->contiguous();
    } else if (!none(a[3])) {
      return false;
    }
    p.ql_nope = q->const_data_ptr();
    p.q_pe = q_pe->const_data_ptr();
    p.cache_kv = cache->const_data_ptr();
    p.num_tokens = (int32_t)T;
    p.num_q_heads = (int32_t)q->size(1);
    p.lkv_dim = (int32_t)lkv;
    p.rope_dim = (int32_t)rope;
    p.row_stride = (int32_t)width;
    p.page_size = (int32_t)(cache->dim() == 3 ? cache->size(1) : cache->size(1) * cache->size(2));
    p.total_pages = (int32_t)cache->size(0);
    p.cache_dtype = kv_type == at::kBFloat16 ? RPA_KV_BF16 : RPA_KV_FP8_E4M3;
    return true;
  }
  const void* new_c_ptr() const { return new_c.defined() ? new_c.const_data_ptr() : nullptr; }
  const void* new_r_ptr() const { return new_r.defined() ? new_r.const_data_ptr() : nullptr; }
};

// mla(ql_nope, q_pe, new_kv_c, new_k_pe, cache, kv_lens, page_indices, cu_q_lens, cu_kv_lens, distribution, sm_scale,
//     sliding_window, soft_cap, mask_value, q_scale, k_scale, v_scale, max_kv_len, num_splits, sum_kv_len)
// -> output, a status below 0, or None.
PyObject* mla(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 20) {
    PyErr_SetString(PyExc_TypeError, "mla takes 20 arguments");
    return nullptr;
  }
  RpaMlaParams p = {};
  MlaTensors x;
  COMMON(x.read(a, p));
  const at::Device dev = x.q->device();
  const at::Tensor* kv_lens = on_device(a[5], dev, at::kInt);
  const at::Tensor* pages = on_device(a[6], dev, at::kInt);
  const at::Tensor* cu_q = on_device(a[7], dev, at::kInt);
  COMMON(kv_lens && pages && cu_q && kv_lens->dim() == 1);
  if (!none(a[8])) {
    const at::Tensor* cu_kv = on_device(a[8], dev, at::kInt);
    COMMON(cu_kv);
    p.cu_kv_lens = cu_kv->const_data_ptr<int32_t>();
  } else {
    p.pages_per_seq = (int32_t)(pages->numel() / std::max<int64_t>(kv_lens->size(0), 1));
  }
  Distribution dist;
  COMMON(dist.read(a[9], dev));
  const bool decode_only = !dist.device && dist.i == dist.j && dist.j == dist.k;
  double d;
  int64_t n;
  COMMON(real(a[10], d));
  p.sm_scale = (float)d;
  if (!none(a[11])) {
    COMMON(whole(a[11], n) && n > 0);
    p.sliding_window = (int32_t)n;
  }
  if (!none(a[12])) {
    COMMON(real(a[12], d) && d != 0.0);
    p.soft_cap = (float)d;
  }
  if (!none(a[13])) {
    COMMON(real(a[13], d));
    p.mask_value = (float)d;
  }
  COMMON(positive(a[14], p.q_scale) && positive(a[15], p.k_scale) && positive(a[16], p.v_scale));
  COMMON(bound(a[17], p.max_kv_len) && bound(a[18], p.num_splits));
  if (!none(a[19])) {
    const long long v = PyLong_AsLongLong(a[19]);
    if (v == -1 && PyErr_Occurred()) {
      PyErr_Clear();
      Py_RETURN_NONE;
    }
    p.sum_kv_len = v;
  }

  at::Tensor out = at::empty_like(*x.q);
  void* stream = stream_of(dev);
  p.out = out.data_ptr();
  p.kv_lens = kv_lens->const_data_ptr<int32_t>();
  p.page_indices = pages->const_data_ptr<int32_t>();
  p.cu_q_lens = cu_q->const_data_ptr<int32_t>();
  p.distribution = dist.device;
  p.num_seqs = dist.device ? (int32_t)kv_lens->size(0) : (int32_t)dist.k;
  at::Tensor ws;
  if (const size_t need = decode_only ? rpa_mla_workspace_bytes(&p) : rpa_mla_attention_workspace_bytes(&p)) {
    ws = workspace(dev, stream, need);
    p.workspace = ws.data_ptr();
    p.workspace_bytes = (size_t)ws.numel();
  }
  const int rc = without_gil([&] { return rpa_mla_attention_update(&p, x.new_c_ptr(), x.new_r_ptr(), decode_only ? 0 : 1, stream); });
  if (rc != RPA_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// sparse_mla(ql_nope, q_pe, new_kv_c, new_k_pe, cache, kv_lens, topk, topk_is_pages, page_indices, cu_q_lens, cu_kv_lens,
//            sm_scale, page_size, pages_per_seq, k_pages_max)
// -> output, a status below 0, or None.  k_pages_max 0: single tokens, else whole pages.
PyObject* sparse_mla(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 15) {
    PyErr_SetString(PyExc_TypeError, "sparse_mla takes 15 arguments");
    return nullptr;
  }
  RpaMlaParams p = {};
  MlaTensors x;
  COMMON(x.read(a, p));
  const at::Device dev = x.q->device();
  const at::Tensor* kv_lens = on_device(a[5], dev, at::kInt);
  const at::Tensor* topk = on_device(a[6], dev, at::kInt);
  const at::Tensor* pages = on_device(a[8], dev, at::kInt);
  const at::Tensor* cu_q = on_device(a[9], dev, at::kInt);
  const at::Tensor* cu_kv = on_device(a[10], dev, at::kInt);
  COMMON(kv_lens && topk && pages && cu_q && cu_kv && kv_lens->dim() == 1 && topk->dim() == 2 &&
         topk->size(0) == x.q->size(0) && cu_q->numel() == kv_lens->size(0) + 1 && cu_kv->numel() == kv_lens->size(0) + 1);
  RpaMlaSparse s = {};
  int64_t page, per_seq, most;
  double scale;
  COMMON(real(a[11], scale) && whole(a[12], page) && whole(a[13], per_seq) && whole(a[14], most));
  COMMON(page == p.page_size && most >= 0 && topk->size(1) <= INT32_MAX && pages->numel() <= INT32_MAX);
  s.topk = topk->const_data_ptr<int32_t>();
  s.topk_is_pages = PyObject_IsTrue(a[7]) == 1;
  s.topk_stride = (int32_t)topk->size(1);
  // precomputed pages: the last of a row's k_pages_max entries is the new token's
  s.topk_count = s.topk_is_pages ? (int32_t)std::min<int64_t>(s.topk_stride, most - 1) : s.topk_stride;
  s.pages_per_seq = (int32_t)per_seq;
  s.k_pages_max = (int32_t)most;
  s.num_page_indices = (int32_t)pages->numel();
  p.sm_scale = (float)scale;
  p.kv_lens = kv_lens->const_data_ptr<int32_t>();
  p.page_indices = pages->const_data_ptr<int32_t>();
  p.cu_q_lens = cu_q->const_data_ptr<int32_t>();
  p.cu_kv_lens = cu_kv->const_data_ptr<int32_t>();
  p.num_seqs = (int32_t)kv_lens->size(0);
  at::Tensor out = at::empty_like(*x.q);
  void* stream = stream_of(dev);
  p.out = out.data_ptr();
  const size_t need = rpa_mla_sparse_workspace_bytes(&p, &s);
  const at::Tensor ws = workspace(dev, stream, need);
  p.workspace = ws.data_ptr();
  p.workspace_bytes = (size_t)ws.numel();
  const int rc = without_gil([&] { return rpa_mla_sparse_attention(&p, &s, x.new_c_ptr(), x.new_r_ptr(), stream); });
  if (rc != RPA_OK) return PyLong_FromLong(rc);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// metadata(decode, seq_lens, cache_loc, extend_seq_lens, page_size, extend_is_mixed, device index)
// -> (cu_q_lens, cu_kv_lens, page_indices, seq_lens, distribution on the device, distribution as a tuple, max_kv_len,
// max_q_len, sum of visible lengths, whether no sequence has a prefix), or None: what build_forward_metadata works out for one data-parallel rank, in one
// pass over the host arrays and one upload.
PyObject* metadata(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  if (nargs != 7) {
    PyErr_SetString(PyExc_TypeError, "metadata takes 7 arguments");
    return nullptr;
  }
  const bool decode = PyObject_IsTrue(a[0]) == 1, mixed = PyObject_IsTrue(a[5]) == 1;
  HostInts lens, loc, ext;
  int64_t P, index;
  COMMON(lens.open(a[1]) && loc.open(a[2]) && (decode || (!none(a[3]) && ext.open(a[3]))) && whole(a[4], P) && P > 0 && whole(a[6], index));
  const int64_t S = lens.size(), np = (loc.size() + P - 1) / P;
  COMMON(S > 0 && (decode || ext.size() == S) && np <= INT32_MAX / 2);
  // (16-byte aligned pieces of one buffer)
  auto up4 = [](int64_t n) { return (n + 3) & ~(int64_t)3; };
  const int64_t at_q = 0, at_kv = up4(S + 1), at_len = at_kv + up4(S + 1), at_dist = at_len + up4(S), at_page = at_dist + 4;
  const int64_t total = at_page + np;
  std::vector<int32_t> w((size_t)total);
  bool no_prefix = !decode;
  int64_t cu_q = 0, cu_kv = 0, n = 0, max_kv = INT64_MIN, max_q = INT64_MIN;
  for (int64_t s = 0; s < S; ++s) {
    const int64_t kv = lens.at(s), q = decode ? 1 : ext.at(s);
    COMMON(kv >= 0 && kv <= INT32_MAX - P && q >= 0);
    cu_q += q;
    cu_kv += (kv + P - 1) / P * P;
    COMMON(cu_q <= INT32_MAX && cu_kv <= INT32_MAX);
    w[at_q + s + 1] = (int32_t)cu_q;
    w[at_kv + s + 1] = (int32_t)cu_kv;
    w[at_len + s] = (int32_t)kv;
    n += kv > 0;
    no_prefix = no_prefix && q == kv;
    max_kv = std::max(max_kv, kv);
    max_q = std::max(max_q, q);
  }
  int64_t visible = 0;
  for (int64_t s = 0; s < n; ++s) {
    const int64_t q = decode ? 1 : ext.at(s);
    visible += q * lens.at(s) - q * (q - 1) / 2;
  }
  const int32_t first = decode ? (int32_t)n : 0, mid = !decode && mixed ? 0 : (int32_t)n;
  w[at_dist] = first, w[at_dist + 1] = mid, w[at_dist + 2] = (int32_t)n;
  for (int64_t i = 0; i < np; ++i) {
    const int64_t slot = loc.at(i * P);
    COMMON(slot >= 0 && slot <= INT32_MAX);
    w[at_page + i] = (int32_t)(slot / P);
  }
  const at::Device dev(at::kCUDA, (c10::DeviceIndex)index);
  const c10::DeviceGuard guard(dev);
  at::Tensor base = at::empty({total}, at::TensorOptions().dtype(at::kInt).device(dev));
  const int rc = rpa_upload_words(base.data_ptr<int32_t>(), w.data(), (int32_t)total, stream_of(dev));
  COMMON(rc == RPA_OK);
  const int64_t from[5] = {at_q, at_kv, at_page, at_len, at_dist}, size[5] = {S + 1, S + 1, np, S, 3};
  PyObject* out = PyTuple_New(10);
  if (!out) return nullptr;
  for (int i = 0; i < 5; ++i) PyTuple_SET_ITEM(out, i, THPVariable_Wrap(base.narrow(0, from[i], size[i])));
  PyTuple_SET_ITEM(out, 5, Py_BuildValue("(iii)", first, mid, (int)n));
  PyTuple_SET_ITEM(out, 6, PyLong_FromLongLong(max_kv));
  PyTuple_SET_ITEM(out, 7, PyLong_FromLongLong(max_q));
  PyTuple_SET_ITEM(out, 8, PyLong_FromLongLong(visible));
  PyTuple_SET_ITEM(out, 9, PyBool_FromLong(no_prefix));
  return out;
  END_HANDLE_TH_ERRORS
}

// workspace(tensor on the device, bytes) -> the buffer of its device's current stream, at least that long
PyObject* py_workspace(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
  HANDLE_TH_ERRORS
  const at::Tensor* t = nargs == 2 ? tensor(a[0]) : nullptr;
  const long long bytes = nargs == 2 ? PyLong_AsLongLong(a[1]) : -1;
  if (!t || bytes < 0) {
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "workspace(tensor, bytes)");
    return nullptr;
  }
  return THPVariable_Wrap(workspace(t->device(), stream_of(t->device()), (size_t)bytes));
  END_HANDLE_TH_ERRORS
}

PyMethodDef kMethods[] = {
    {"attention", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(attention)), METH_FASTCALL, nullptr},
    {"mla", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(mla)), METH_FASTCALL, nullptr},
    {"sparse_mla", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(sparse_mla)), METH_FASTCALL, nullptr},
    {"metadata", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(metadata)), METH_FASTCALL, nullptr},
    {"workspace", reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(py_workspace)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "rpa_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit_rpa_torch() { return PyModule_Create(&kModule); }
