// CPython binding of the calls a serving step makes: tensors in, one library call out, without a trip through Python per
// argument.  (Some forty arguments, each a method call and a ctypes conversion, were 20 of the 30 us a decode step of a short
// context took the host, and its four kernels end before that.)
//
// Only well-formed calls are taken: plain device tensors of one device with the types, strides and sizes the kernels read.
// For anything else -- other types, layouts that need a copy, wrappers, active dispatch or function modes, a workspace that is
// too small -- a function returns None and the caller goes the long way in Python, which converts, allocates or raises.  An
// integer is a status of the library.  Nothing is kept from one call for the next but the addresses of the library's functions.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include "../../include/aitherkv.h"

namespace {

struct Library {
  decltype(&akv_paged_attn_workspace_bytes) attn_bytes;
  decltype(&akv_paged_attn) attn;
  decltype(&akv_encode_paged_kv) encode;
  decltype(&akv_hybrid_paged_attn_workspace_bytes) hybrid_bytes;
  decltype(&akv_hybrid_paged_attn) hybrid_attn[2];                  // tq35, tq25
  decltype(&akv_hybrid_encode_paged_kv) hybrid_encode[2];
  decltype(&akv_decode_blocks_kv) decode_blocks;
  decltype(&akv_tri_encode_paged_kv) tri_encode;
  decltype(&akv_tri_decode_workspace_bytes) tri_bytes;
  decltype(&akv_tri_decode_paged) tri_decode;
} g_lib;
static_assert(std::is_same_v<decltype(&akv_hybrid_paged_attn), decltype(&akv_hybrid25_paged_attn)> && std::is_same_v<decltype(&akv_hybrid_encode_paged_kv), decltype(&akv_hybrid25_encode_paged_kv)>);
constexpr int kFunctions = 12;
PyObject* g_raw_stream = nullptr;      // torch's function: handle of the current stream of a device

// the tensors of a call; ok() once all of them are plain device tensors of one device
class Tensors {
 public:
  Tensors() { ok_ = !c10::impl::dispatch_mode_enabled() && !at::impl::torch_function_mode_enabled(); }
  const at::Tensor& take(PyObject* o) {
    static const at::Tensor none;
    if (!ok_ || !THPVariable_CheckExact(o)) {
      ok_ = false;
      return none;
    }
    const at::Tensor& t = THPVariable_Unpack(o);
    const auto keys = t.key_set() - c10::autograd_dispatch_keyset_with_ADInplaceOrView - c10::autocast_dispatch_keyset;
    if (keys != c10::DispatchKeySet(c10::DispatchKey::CUDA)) {
      ok_ = false;
      return none;
    }
    const int dev = t.get_device();
    if (dev_ < 0) dev_ = dev;
    if (dev != dev_) ok_ = false;
    return t;
  }
  bool ok() const { return ok_; }
  int device() const { return dev_; }

 private:
  bool ok_;
  int dev_ = -1;
};

int float_code(const at::Tensor& t) {
  switch (t.scalar_type()) {
    case at::kHalf: return AKV_F16;
    case at::kBFloat16: return AKV_BF16;
    case at::kFloat: return AKV_F32;
    default: return -1;
  }
}
int index_code(const at::Tensor& t) { return t.scalar_type() == at::kInt ? AKV_I32 : t.scalar_type() == at::kLong ? AKV_I64 : -1; }

// an int, or `none` for None
bool integer(PyObject* o, int64_t& v, int64_t none = -1, bool may_be_none = false) {
  if (may_be_none && o == Py_None) {
    v = none;
    return true;
  }
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  v = PyLong_AsLongLongAndOverflow(o, &overflow);
  return overflow == 0;
}
// 0 when there is an exception
bool stream_of(int device, void*& stream) {
  PyObject* index = PyLong_FromLong(device);
  if (!index) return false;
  PyObject* handle = PyObject_CallFunctionObjArgs(g_raw_stream, index, nullptr);
  Py_DECREF(index);
  if (!handle) return false;
  stream = PyLong_AsVoidPtr(handle);
  Py_DECREF(handle);
  return !PyErr_Occurred();
}
// f(args...) with the interpreter's lock given up.  What is read of tensors is in `args`, read while it is held: another thread may
// give a tensor other storage or sizes once it is not.
template <class F, class... Args>
int without_gil(F f, Args... args) noexcept {
  int rc;
  Py_BEGIN_ALLOW_THREADS;
  rc = f(args...);
  Py_END_ALLOW_THREADS;
  return rc;
}
PyObject* status(int rc) { return PyLong_FromLong(rc); }

// rows of a cache: [blocks, positions, heads, bytes], and their norms; a call addresses `block` positions and `heads` heads
bool packed_rows(const at::Tensor& t, int64_t bytes, int64_t block, int64_t heads) {
  return t.dim() == 4 && t.scalar_type() == at::kByte && t.stride(3) == 1 && t.size(3) >= bytes && t.size(1) >= block && t.size(2) >= heads;
}
bool norm_rows(const at::Tensor& t, int64_t block, int64_t heads) {
  return t.dim() == 3 && t.scalar_type() == at::kFloat && t.size(1) >= block && t.size(2) >= heads;
}
// a table of at least n floats
bool floats(const at::Tensor& t, int64_t n) { return t.scalar_type() == at::kFloat && t.is_contiguous() && t.numel() >= n; }
// the blocks a write may go to: those the caller names (0: all), as far as they exist
int64_t blocks_of(int64_t named, int64_t held) { return named != 0 ? std::min(named, held) : held; }

// what every attention call checks of its queries, tables and lengths
bool attn_inputs(const at::Tensor& q, const at::Tensor& tables, const at::Tensor& lens, int64_t heads, int64_t d) {
  return q.dim() == 3 && q.size(0) > 0 && q.size(1) == heads && q.size(2) == d && q.stride(2) == 1 && float_code(q) >= 0 && tables.dim() == 2 &&
         tables.size(0) >= q.size(0) && lens.numel() >= q.size(0) && tables.stride(1) == 1 && index_code(tables) >= 0 && lens.dim() == 1 && lens.is_contiguous() && index_code(lens) >= 0;
}

// (query, k_packed, k_norms, v_packed, v_norms, block_tables, context_lens, centroids, workspace or None, prepared rotation,
//  kv heads or None, query heads, head size, bytes of a row, bits, block size, scale)
PyObject* uniform_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t v[7];
  if (n != 17 || a[8] == Py_None || !PyFloat_CheckExact(a[16])) Py_RETURN_NONE;
  for (int i = 0; i < 7; ++i)
    if (!integer(a[9 + i], v[i], 0, i == 1)) Py_RETURN_NONE;
  Tensors ts;
  const at::Tensor &q = ts.take(a[0]), &kp = ts.take(a[1]), &kn = ts.take(a[2]), &vp = ts.take(a[3]), &vn = ts.take(a[4]);
  const at::Tensor &bt = ts.take(a[5]), &cl = ts.take(a[6]), &cen = ts.take(a[7]), &ws = ts.take(a[8]);
  const int64_t heads = v[2], d = v[3], row = v[4], bits = v[5], block = v[6];
  if (!ts.ok() || !attn_inputs(q, bt, cl, heads, d) || kp.dim() != 4 || bits < 2 || bits > 4 || !floats(cen, 1 << bits)) Py_RETURN_NONE;
  const int64_t seqs = q.size(0), kv_heads = a[10] == Py_None ? kp.size(2) : v[1];
  if (!packed_rows(kp, row, block, kv_heads) || !packed_rows(vp, row, block, kv_heads) || !norm_rows(kn, block, kv_heads) || !norm_rows(vn, block, kv_heads)) Py_RETURN_NONE;
  if (ws.numel() < (int64_t)g_lib.attn_bytes((int)seqs, (int)heads, (int)d)) Py_RETURN_NONE;
  const int64_t blocks = std::min(std::min(kp.size(0), kn.size(0)), std::min(vp.size(0), vn.size(0)));
  void* stream;
  if (!stream_of(ts.device(), stream)) return nullptr;
  at::Tensor out = at::empty({seqs, heads, d}, q.options());
  const int rc = without_gil(g_lib.attn, q.const_data_ptr(), float_code(q), q.stride(0), q.stride(1), (const uint8_t*)kp.const_data_ptr(), kp.stride(0), kp.stride(1), kp.stride(2),
                             (const float*)kn.const_data_ptr(), kn.stride(0), kn.stride(1), kn.stride(2), (const uint8_t*)vp.const_data_ptr(), vp.stride(0), vp.stride(1),
                             vp.stride(2), (const float*)vn.const_data_ptr(), vn.stride(0), vn.stride(1), vn.stride(2), bt.const_data_ptr(), index_code(bt), bt.stride(0),
                             cl.const_data_ptr(), index_code(cl), (const void*)(uintptr_t)v[0], (const float*)cen.const_data_ptr(), (int)bits, out.mutable_data_ptr(),
                             float_code(out), out.stride(0), out.stride(1), (int)seqs, (int)heads, (int)kv_heads, (int)d, (int)block, blocks, bt.size(1),
                             (float)PyFloat_AS_DOUBLE(a[16]), ws.mutable_data_ptr(), (size_t)ws.numel(), stream);
  return rc ? status(rc) : THPVariable_Wrap(std::move(out));
}

// (query, k_cache, v_cache, block_tables, context_lens, table, workspace or None, format (0: tq35, 1: tq25), kv heads or None,
//  query heads, head size, bytes of a row, block size, scale)
PyObject* hybrid_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t v[6];
  if (n != 14 || a[6] == Py_None || !PyFloat_CheckExact(a[13])) Py_RETURN_NONE;
  for (int i = 0; i < 6; ++i)
    if (!integer(a[7 + i], v[i], 0, i == 1)) Py_RETURN_NONE;
  Tensors ts;
  const at::Tensor &q = ts.take(a[0]), &kc = ts.take(a[1]), &vc = ts.take(a[2]), &bt = ts.take(a[3]), &cl = ts.take(a[4]);
  const at::Tensor &table = ts.take(a[5]), &ws = ts.take(a[6]);
  const int64_t heads = v[2], d = v[3], row = v[4], block = v[5];
  if (!ts.ok() || v[0] < 0 || v[0] > 1 || !attn_inputs(q, bt, cl, heads, d) || kc.dim() != 4 || !floats(table, AKV_HYB_TABLE_FLOATS)) Py_RETURN_NONE;
  const int64_t seqs = q.size(0), kv_heads = a[8] == Py_None ? kc.size(2) : v[1];
  if (!packed_rows(kc, row, block, kv_heads) || !packed_rows(vc, row, block, kv_heads)) Py_RETURN_NONE;
  if (ws.numel() < (int64_t)g_lib.hybrid_bytes((int)seqs, (int)heads)) Py_RETURN_NONE;
  void* stream;
  if (!stream_of(ts.device(), stream)) return nullptr;
  at::Tensor out = at::empty({seqs, heads, d}, q.options());
  const int rc = without_gil(g_lib.hybrid_attn[v[0]], q.const_data_ptr(), float_code(q), q.stride(0), q.stride(1), (const uint8_t*)kc.const_data_ptr(), kc.stride(0), kc.stride(1),
                             kc.stride(2), (const uint8_t*)vc.const_data_ptr(), vc.stride(0), vc.stride(1), vc.stride(2), bt.const_data_ptr(), index_code(bt),
                             bt.stride(0), cl.const_data_ptr(), index_code(cl), (const float*)table.const_data_ptr(), out.mutable_data_ptr(), float_code(out),
                             out.stride(0), out.stride(1), (int)seqs, (int)heads, (int)kv_heads, (int)block, std::min(kc.size(0), vc.size(0)), bt.size(1),
                             (float)PyFloat_AS_DOUBLE(a[13]), ws.mutable_data_ptr(), (size_t)ws.numel(), stream);
  return rc ? status(rc) : THPVariable_Wrap(std::move(out));
}

// key and value of a call: [tokens, heads, d], alike, and so are their caches
bool pair_inputs(const at::Tensor& k, const at::Tensor& v, const at::Tensor& slots) {
  return k.dim() == 3 && v.dim() == 3 && k.size(0) > 0 && k.sizes() == v.sizes() && k.strides() == v.strides() && k.stride(2) == 1 &&
         k.scalar_type() == v.scalar_type() && float_code(k) >= 0 && slots.is_contiguous() && slots.numel() >= k.size(0) && index_code(slots) >= 0;
}

// (key, value, slot_mapping, k_packed, k_norms, v_packed, v_norms, rotation, boundaries, prepared rotation, bits, block size, blocks
//  (0: those of the cache)) -> status
PyObject* uniform_encode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t v[4];
  if (n != 13) Py_RETURN_NONE;
  for (int i = 0; i < 4; ++i)
    if (!integer(a[9 + i], v[i])) Py_RETURN_NONE;
  Tensors ts;
  const at::Tensor &key = ts.take(a[0]), &value = ts.take(a[1]), &slots = ts.take(a[2]), &kp = ts.take(a[3]), &kn = ts.take(a[4]);
  const at::Tensor &vp = ts.take(a[5]), &vn = ts.take(a[6]), &rot = ts.take(a[7]), &bnd = ts.take(a[8]);
  if (!ts.ok() || !pair_inputs(key, value, slots) || v[1] < 2 || v[1] > 4 || key.size(2) % 8 != 0) Py_RETURN_NONE;
  const int64_t heads = key.size(1), d = key.size(2), row = d * v[1] / 8, block = v[2];
  if (!packed_rows(kp, row, block, heads) || !norm_rows(kn, block, heads) || vp.scalar_type() != at::kByte || vn.scalar_type() != at::kFloat ||
      kp.sizes() != vp.sizes() || kp.strides() != vp.strides() || kn.sizes() != vn.sizes() || kn.strides() != vn.strides() || rot.dim() != 2 ||
      rot.size(0) != d || rot.size(1) != d || !floats(bnd, (1 << v[1]) - 1) || (d & (d - 1)) != 0)
    Py_RETURN_NONE;
  void* stream;
  if (!stream_of(ts.device(), stream)) return nullptr;
  const int rc = without_gil(g_lib.encode, key.const_data_ptr(), value.const_data_ptr(), float_code(key), key.size(0), (int)key.size(1), (int)key.size(2), key.stride(0), key.stride(1),
                             slots.const_data_ptr(), index_code(slots), (const void*)(uintptr_t)v[0], (const float*)bnd.const_data_ptr(), (int)v[1],
                             (uint8_t*)kp.mutable_data_ptr(), (uint8_t*)vp.mutable_data_ptr(), kp.stride(0), kp.stride(1), kp.stride(2),
                             (float*)kn.mutable_data_ptr(), (float*)vn.mutable_data_ptr(), kn.stride(0), kn.stride(1), kn.stride(2), (int)v[2],
                             blocks_of(v[3], std::min(kp.size(0), kn.size(0))), stream);
  return status(rc);
}

// (key, value, slot_mapping, k_cache, v_cache, table, format (0: tq35, 1: tq25), head size, bytes of a row, block size, blocks (0:
//  those of the cache)) -> status
PyObject* hybrid_encode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t v[5];
  if (n != 11) Py_RETURN_NONE;
  for (int i = 0; i < 5; ++i)
    if (!integer(a[6 + i], v[i])) Py_RETURN_NONE;
  Tensors ts;
  const at::Tensor &key = ts.take(a[0]), &value = ts.take(a[1]), &slots = ts.take(a[2]), &kc = ts.take(a[3]), &vc = ts.take(a[4]), &table = ts.take(a[5]);
  if (!ts.ok() || v[0] < 0 || v[0] > 1 || !floats(table, AKV_HYB_TABLE_FLOATS) || !pair_inputs(key, value, slots) || key.size(2) != v[1] || !packed_rows(kc, v[2], v[3], key.size(1)) ||
      vc.scalar_type() != at::kByte || kc.sizes() != vc.sizes() || kc.strides() != vc.strides())
    Py_RETURN_NONE;
  void* stream;
  if (!stream_of(ts.device(), stream)) return nullptr;
  const int rc = without_gil(g_lib.hybrid_encode[v[0]], key.const_data_ptr(), value.const_data_ptr(), float_code(key), key.size(0), (int)key.size(1), key.stride(0), key.stride(1),
                             slots.const_data_ptr(), index_code(slots), (const float*)table.const_data_ptr(), (uint8_t*)kc.mutable_data_ptr(),
                             (uint8_t*)vc.mutable_data_ptr(), kc.stride(0), kc.stride(1), kc.stride(2), (int)v[3], blocks_of(v[4], kc.size(0)), stream);
  return status(rc);
}

// first and last byte a tensor reaches
std::pair<uintptr_t, uintptr_t> span(const at::Tensor& t) {
  int64_t last = 0;
  for (int64_t i = 0; i < t.dim(); ++i) last += (t.size(i) - 1) * t.stride(i);
  const uintptr_t at = (uintptr_t)t.const_data_ptr();
  return {at, at + (uintptr_t)(last + 1) * t.element_size()};
}

// (key_cache, value_cache, k_buf, v_buf, block ids, k_norms, v_norms, centroids, prepared rotation, blocks, head size, bytes of a row,
//  bits) -> status
PyObject* decode_blocks(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t v[5];
  if (n != 13) Py_RETURN_NONE;
  for (int i = 0; i < 5; ++i)
    if (!integer(a[8 + i], v[i])) Py_RETURN_NONE;
  Tensors ts;
  const at::Tensor &kc = ts.take(a[0]), &vc = ts.take(a[1]), &kb = ts.take(a[2]), &vb = ts.take(a[3]), &ids = ts.take(a[4]);
  const at::Tensor &kn = ts.take(a[5]), &vn = ts.take(a[6]), &cen = ts.take(a[7]);
  const int64_t blocks = v[1], d = v[2];
  if (!ts.ok() || !packed_rows(kc, v[3], 0, 0) || !packed_rows(vc, v[3], 0, 0) || !norm_rows(kn, 0, 0) || !norm_rows(vn, 0, 0) || kb.dim() != 4 || kb.stride(3) != 1 ||
      float_code(kb) < 0 || kb.size(3) != d || kb.numel() == 0 || vb.scalar_type() != kb.scalar_type() || kb.sizes() != vb.sizes() ||
      kb.strides() != vb.strides() || kc.sizes() != vc.sizes() || kc.strides() != vc.strides() || kn.sizes() != vn.sizes() || kn.strides() != vn.strides() ||
      kc.sizes().slice(0, 3) != kn.sizes() || kc.sizes().slice(0, 3) != kb.sizes().slice(0, 3) || blocks <= 0 || blocks > kc.size(0) ||
      v[4] < 2 || v[4] > 4 || !floats(cen, 1 << v[4]) || index_code(ids) < 0 || !ids.is_contiguous() || ids.numel() == 0)
    Py_RETURN_NONE;
  const auto k = span(kb), w = span(vb);
  if (!(k.second <= w.first || w.second <= k.first)) Py_RETURN_NONE;
  void* stream;
  if (!stream_of(ts.device(), stream)) return nullptr;
  const int rc = without_gil(g_lib.decode_blocks, (const uint8_t*)kc.const_data_ptr(), (const uint8_t*)vc.const_data_ptr(), kc.stride(0), kc.stride(1), kc.stride(2),
                             (const float*)kn.const_data_ptr(), (const float*)vn.const_data_ptr(), kn.stride(0), kn.stride(1), kn.stride(2), ids.const_data_ptr(),
                             index_code(ids), ids.numel(), blocks, (int)kc.size(1), (int)kc.size(2), (int)d, (const void*)(uintptr_t)v[0],
                             (const float*)cen.const_data_ptr(), (int)v[4], kb.mutable_data_ptr(), vb.mutable_data_ptr(), float_code(kb), kb.stride(0), kb.stride(1),
                             kb.stride(2), stream);
  return status(rc);
}

// (keys, values, slot_mapping, k indices, k coefficients, k scales, v indices, v coefficients, v scales, kv heads, head size, pairs,
//  slots of the cache) -> status
PyObject* spectral_encode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t v[4];
  if (n != 13) Py_RETURN_NONE;
  for (int i = 0; i < 4; ++i)
    if (!integer(a[9 + i], v[i])) Py_RETURN_NONE;
  Tensors ts;
  const at::Tensor &keys = ts.take(a[0]), &values = ts.take(a[1]), &slots = ts.take(a[2]);
  const at::Tensor* c[6];
  for (int i = 0; i < 6; ++i) c[i] = &ts.take(a[3 + i]);
  if (!ts.ok() || keys.dim() != 3 || keys.size(0) == 0 || keys.size(1) != v[0] || keys.size(2) != v[1] || values.sizes() != keys.sizes() ||
      values.strides() != keys.strides() || keys.stride(2) != 1 || float_code(keys) < 0 || values.scalar_type() != keys.scalar_type() || index_code(slots) < 0 || !slots.is_contiguous() ||
      slots.numel() != keys.size(0))
    Py_RETURN_NONE;
  void* stream;
  if (!stream_of(ts.device(), stream)) return nullptr;
  const int rc = without_gil(g_lib.tri_encode, keys.const_data_ptr(), values.const_data_ptr(), float_code(keys), keys.size(0), (int)v[0], (int)v[1], keys.stride(0), keys.stride(1),
                             (int)v[2], slots.const_data_ptr(), index_code(slots), v[3], (uint8_t*)c[0]->mutable_data_ptr(), (uint8_t*)c[1]->mutable_data_ptr(),
                             c[2]->mutable_data_ptr(), (uint8_t*)c[3]->mutable_data_ptr(), (uint8_t*)c[4]->mutable_data_ptr(), c[5]->mutable_data_ptr(), stream);
  return status(rc);
}

// (query, k indices, k coefficients, k scales, v indices, v coefficients, v scales, theta, block_tables, context_lens, workspace or
//  None, head size, keys before RoPE (0 or 1)).  A shape the paged kernel does not take: None.
PyObject* spectral_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
  int64_t v[2];
  if (n != 13 || a[10] == Py_None || !integer(a[11], v[0]) || !integer(a[12], v[1])) Py_RETURN_NONE;
  Tensors ts;
  const at::Tensor& q = ts.take(a[0]);
  const at::Tensor* c[6];
  for (int i = 0; i < 6; ++i) c[i] = &ts.take(a[1 + i]);
  const at::Tensor &theta = ts.take(a[7]), &bt = ts.take(a[8]), &cl = ts.take(a[9]), &ws = ts.take(a[10]);
  if (!ts.ok() || q.dim() != 3 || c[0]->dim() != 4 || q.size(0) == 0 || q.size(2) != v[0] || !q.is_contiguous() || float_code(q) < 0) Py_RETURN_NONE;
  const int64_t b = q.size(0), qh = q.size(1), d = q.size(2), kvh = c[0]->size(2);
  for (int i = 0; i < 6; ++i)
    if (!c[i]->is_contiguous()) Py_RETURN_NONE;
  if (kvh == 0 || qh % kvh != 0 || bt.dim() != 2 || bt.size(0) != b || bt.stride(1) != 1 || index_code(bt) < 0 || cl.numel() != b || !cl.is_contiguous() ||
      index_code(cl) < 0 || ws.numel() < (int64_t)g_lib.tri_bytes((int)b, (int)qh, (int)d))
    Py_RETURN_NONE;
  void* stream;
  if (!stream_of(ts.device(), stream)) return nullptr;
  at::Tensor out = at::empty({b, qh, d}, q.options().dtype(at::kFloat));
  const int rc = without_gil(g_lib.tri_decode, q.const_data_ptr(), float_code(q), (const uint8_t*)c[0]->const_data_ptr(), (const uint8_t*)c[1]->const_data_ptr(),
                             c[2]->const_data_ptr(), (const uint8_t*)c[3]->const_data_ptr(), (const uint8_t*)c[4]->const_data_ptr(), c[5]->const_data_ptr(),
                             (const float*)theta.const_data_ptr(), nullptr, 0, bt.const_data_ptr(), index_code(bt), bt.stride(0), cl.const_data_ptr(), index_code(cl),
                             (float*)out.mutable_data_ptr(), (int)b, c[0]->size(0), (int)c[0]->size(1), bt.size(1), (int)qh, (int)kvh, (int)d, (int)c[0]->size(3),
                             (int)v[1], ws.mutable_data_ptr(), (size_t)ws.numel(), stream);
  if (rc == AKV_ERR_UNSUPPORTED) Py_RETURN_NONE;
  return rc ? status(rc) : THPVariable_Wrap(std::move(out));
}

// (raw stream function, addresses in the order of Library)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
  static_assert(sizeof(Library) == kFunctions * sizeof(void*), "one address a member");
  if (n != 1 + kFunctions) {
    PyErr_SetString(PyExc_TypeError, "bind: a function and the addresses");
    return nullptr;
  }
  void* at[kFunctions];
  for (int i = 0; i < kFunctions; ++i) {
    at[i] = PyLong_AsVoidPtr(a[1 + i]);
    if (PyErr_Occurred()) return nullptr;
  }
  memcpy((void*)&g_lib, at, sizeof(g_lib));
  Py_INCREF(a[0]);
  Py_XSETREF(g_raw_stream, a[0]);
  Py_RETURN_NONE;
}

// an exception of torch (no memory for an output, a tensor without storage): the long way tries again and raises torch's own error
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* guarded(PyObject* self, PyObject* const* a, Py_ssize_t n) noexcept {
  try {
    return F(self, a, n);
  } catch (const std::exception&) {
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
  }
}

PyMethodDef kMethods[] = {
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
    {"uniform_attention", (PyCFunction)(void (*)(void))guarded<uniform_attention>, METH_FASTCALL, nullptr},
    {"hybrid_attention", (PyCFunction)(void (*)(void))guarded<hybrid_attention>, METH_FASTCALL, nullptr},
    {"uniform_encode", (PyCFunction)(void (*)(void))guarded<uniform_encode>, METH_FASTCALL, nullptr},
    {"hybrid_encode", (PyCFunction)(void (*)(void))guarded<hybrid_encode>, METH_FASTCALL, nullptr},
    {"decode_blocks", (PyCFunction)(void (*)(void))guarded<decode_blocks>, METH_FASTCALL, nullptr},
    {"spectral_encode", (PyCFunction)(void (*)(void))guarded<spectral_encode>, METH_FASTCALL, nullptr},
    {"spectral_attention", (PyCFunction)(void (*)(void))guarded<spectral_attention>, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding(void) {
  PyObject* m = PyModule_Create(&kModule);
  // (what it was compiled against: _lib.py loads no other)
  PyObject* built = Py_BuildValue("(ss)", TORCH_VERSION, Py_STRINGIFY(PY_MAJOR_VERSION) "." Py_STRINGIFY(PY_MINOR_VERSION));
  if (!m || !built || PyModule_AddObject(m, "BUILT_FOR", built) < 0) {
    Py_XDECREF(built);
    Py_XDECREF(m);
    return nullptr;
  }
  return m;
}
