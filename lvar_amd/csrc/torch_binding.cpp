// Compiled host path for torch callers: argument checks, output allocation and launches happen in C++, which takes the
// host cost of a call from 15 .. 70 us (Python + ctypes) to 4 .. 12 us -- small scales and small batches are bound by
// exactly that.  Two forms:
//   fast_*                            the operators of lvar_amd.sparse_attn_ops and the two steps of SparseDiffAttn for
//                                     well-formed inputs on the current device; every other input returns None and takes
//                                     the Python path, which raises the errors
//   register_dense_attn(ns)           defines and implements the torch-library op
//                                     `<ns>::dense_attn(Tensor q, Tensor k, Tensor v) -> Tensor[]`
//                                     natively, as the reference registers torch.ops.chipmunk.dense_attn
//                                     (kernels/chipmunk/csrc/chipmunk.cu:50-89, dense_attn at :57):
//                                     returns [o, 1/(2^M L)], softmax scale fixed to 1 (dense_attn.cu:161-163)
//
// The fast_* functions take their arguments as a C array (METH_FASTCALL) and allocate with torch's caching allocator
// directly: parsing through a signature and dispatching an `empty` would cost as much as the launch.
//
// The module does not link the C-ABI library: bind() receives the entry points' addresses from the Python
// side (which has loaded the library with ctypes), so both paths always call the same library.
#include <cmath>
#include <memory>
#include <optional>
#include <string>
#include <vector>
#include <torch/extension.h>
#include <torch/library.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/core/DeviceGuard.h>
#include <c10/hip/HIPStream.h>
#include "../../include/lvar_sparse_attn.h"

namespace {

// entry points of the C-ABI library, by name
#define LVAR_ENTRIES(X)                                                                                                   \
  X(lvar_dense_attn_fwd) X(lvar_dense_attn_rcp_fwd) X(lvar_row_lse_scratch_bytes) X(lvar_row_lse_fwd)                     \
  X(lvar_lse2_from_stats) X(lvar_colsum_fwd) X(lvar_csp_attn_fwd) X(lvar_csp_attn_upsample_fwd)                           \
  X(lvar_csp_attn_remap_fwd)                                                                                              \
  X(lvar_block_sparse_attn_fwd) X(lvar_block_topk_lists) X(lvar_topk_token_lists) X(lvar_topk_union_lists)                \
  X(lvar_remap_concat_lists) X(lvar_mask_to_lists) X(lvar_window_key_scores)
struct Api {
#define LVAR_FIELD(name) decltype(&::name) name = nullptr;
  LVAR_ENTRIES(LVAR_FIELD)
#undef LVAR_FIELD
} api;
bool bound = false;

std::vector<std::string> entry_names() {
  std::vector<std::string> v;
#define LVAR_NAME(name) v.emplace_back(#name);
  LVAR_ENTRIES(LVAR_NAME)
#undef LVAR_NAME
  return v;
}

// addresses in the order of entry_names()
void bind(const std::vector<uintptr_t>& a) {
  TORCH_CHECK(a.size() == entry_names().size(), "lvar_amd: wrong number of entry points");
  size_t i = 0;
#define LVAR_SET(name) api.name = reinterpret_cast<decltype(&::name)>(a[i++]);
  LVAR_ENTRIES(LVAR_SET)
#undef LVAR_SET
  bound = true;
}

bool plain(const at::Tensor& t) {
  return t.defined() && t.is_cuda() && t.dim() == 4 && t.scalar_type() == at::kBFloat16 && t.is_contiguous() &&
         (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15u) == 0;
}

lvar_tensor_t view(const at::Tensor& t) {
  lvar_tensor_t v;
  v.ptr = t.data_ptr();
  v.stride_b = t.stride(0);
  v.stride_h = t.stride(1);
  v.stride_row = t.stride(2);
  return v;
}

// ---- argument helpers: each returns false / null for what the Python path has to look at ----
const at::Tensor* tensor(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

// rows of a 4-d bf16 tensor that the kernels can read in place: unit stride on d, 16-byte aligned rows
bool rows_ok(const at::Tensor* t, int dev) {
  if (!t || !t->is_cuda() || t->get_device() != dev || t->dim() != 4 || t->scalar_type() != at::kBFloat16) return false;
  const auto st = t->strides();
  return st[3] == 1 && ((st[0] | st[1] | st[2]) & 7) == 0 && st[2] > 0 && (reinterpret_cast<uintptr_t>(t->data_ptr()) & 15u) == 0;
}

// contiguous tensor of a dtype on the device
bool packed(const at::Tensor* t, int dev, at::ScalarType ty) {
  return t && t->is_cuda() && t->get_device() == dev && t->scalar_type() == ty && t->is_contiguous();
}

bool as_long(PyObject* o, int64_t& v) {
  if (!PyLong_CheckExact(o)) return false;
  v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
  return true;
}

bool as_bool(PyObject* o, bool& v) {
  if (!PyBool_Check(o)) return false;
  v = o == Py_True;
  return true;
}

bool as_double(PyObject* o, double& v) {
  if (PyFloat_CheckExact(o)) { v = PyFloat_AS_DOUBLE(o); return true; }
  int64_t i;
  if (!as_long(o, i)) return false;
  v = static_cast<double>(i);
  return true;
}

// softmax scale: None = 1/sqrt(d)
bool as_scale(PyObject* o, int64_t d, float& s) {
  if (o == Py_None) { s = static_cast<float>(1.0 / std::sqrt(static_cast<double>(d))); return true; }
  double v;
  if (!as_double(o, v)) return false;
  s = static_cast<float>(v);
  return true;
}

struct Qkv {
  const at::Tensor *q, *k, *v;
  int dev, B, H, Hkv, Lq, Lk, d;
  void* stream;
};

// q, k and (unless `v` is null) v of one attention call on the current device; `gqa`: fewer key heads than query heads
bool qkv_ok(Qkv& a, PyObject* q, PyObject* k, PyObject* v, bool gqa) {
  a.q = tensor(q); a.k = tensor(k); a.v = v ? tensor(v) : a.k;
  if (!bound || !a.q || !a.q->is_cuda()) return false;
  a.dev = a.q->get_device();
  if (!rows_ok(a.q, a.dev) || !rows_ok(a.k, a.dev) || !rows_ok(a.v, a.dev)) return false;
  const auto qs = a.q->sizes(), ks = a.k->sizes();
  if (a.v != a.k && a.v->sizes() != ks) return false;
  if (qs[0] != ks[0] || qs[3] != ks[3] || (qs[3] != 64 && qs[3] != 128 && qs[3] != 256)) return false;
  if (qs[0] <= 0 || qs[1] <= 0 || qs[2] <= 0 || ks[1] <= 0 || ks[2] <= 0 || qs[2] > INT32_MAX || ks[2] > INT32_MAX) return false;
  if (qs[1] != ks[1] && !(gqa && qs[1] % ks[1] == 0)) return false;
  if (c10::hip::current_device() != a.dev) return false;
  a.B = static_cast<int>(qs[0]); a.H = static_cast<int>(qs[1]); a.Hkv = static_cast<int>(ks[1]);
  a.Lq = static_cast<int>(qs[2]); a.Lk = static_cast<int>(ks[2]); a.d = static_cast<int>(qs[3]);
  a.stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(a.dev)).stream();
  return true;
}

at::Tensor empty(at::IntArrayRef sizes, at::ScalarType ty, int dev) {
  return at::Tensor(at::detail::empty_cuda(sizes, ty, at::Device(at::kCUDA, static_cast<c10::DeviceIndex>(dev)), std::nullopt));
}
at::Tensor empty_o(const Qkv& a) { return empty({a.B, a.H, a.Lq, a.d}, at::kBFloat16, a.dev); }
at::Tensor empty_stat(const Qkv& a) { return empty({a.B, a.H, a.Lq, 1}, at::kFloat, a.dev); }

// M and L in one allocation: L is a view of the storage behind M
void empty_stats(const Qkv& a, at::Tensor& M, at::Tensor& L) {
  const int64_t rows = int64_t(a.B) * a.H * a.Lq;
  M = empty({2, a.B, a.H, a.Lq, 1}, at::kFloat, a.dev);
  L = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(M.storage()), M.key_set(), M.dtype());
  L.unsafeGetTensorImpl()->set_sizes_contiguous({a.B, a.H, a.Lq, 1});
  L.unsafeGetTensorImpl()->set_storage_offset(rows);
  M.unsafeGetTensorImpl()->set_sizes_contiguous({a.B, a.H, a.Lq, 1});
}

PyObject* none() { Py_RETURN_NONE; }

template <class... T>
PyObject* tuple(T&&... t) {
  PyObject* r = PyTuple_New(sizeof...(t));
  if (!r) return nullptr;
  Py_ssize_t i = 0;
  (PyTuple_SET_ITEM(r, i++, THPVariable_Wrap(std::forward<T>(t))), ...);
  return r;
}

#define LVAR_FAST(name) PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n)
#define LVAR_NEED(cond) do { if (!(cond)) return none(); } while (0)

// (q, k, v, scale) -> (o, M, L)
LVAR_FAST(fast_dense_attn) {
  HANDLE_TH_ERRORS
  Qkv x;
  float scale;
  LVAR_NEED(n == 4 && qkv_ok(x, a[0], a[1], a[2], true) && as_scale(a[3], x.d, scale));
  at::Tensor o = empty_o(x), M, L;
  empty_stats(x, M, L);
  LVAR_NEED(api.lvar_dense_attn_fwd(view(*x.q), view(*x.k), view(*x.v), view(o), M.data_ptr<float>(), L.data_ptr<float>(), nullptr,
                                    x.B, x.H, x.Hkv, x.Lq, x.Lk, x.d, scale, x.stream) == LVAR_OK);
  return tuple(std::move(o), std::move(M), std::move(L));
  END_HANDLE_TH_ERRORS
}

int64_t groups_of(int64_t Lq, int64_t rows) { return (Lq + rows - 1) / rows; }

// (q, k, v, scale, group rows) -> (o, cs, M, L)
LVAR_FAST(fast_dense_colsum_attn) {
  HANDLE_TH_ERRORS
  Qkv x;
  float scale;
  int64_t bm;
  LVAR_NEED(n == 5 && qkv_ok(x, a[0], a[1], a[2], true) && as_scale(a[3], x.d, scale) && as_long(a[4], bm) && bm > 0 && bm % 32 == 0);
  at::Tensor o = empty_o(x), lse2 = empty_stat(x), M, L;
  empty_stats(x, M, L);
  at::Tensor cs = empty({x.B, x.H, groups_of(x.Lq, bm), x.Lk}, at::kFloat, x.dev);
  LVAR_NEED(api.lvar_dense_attn_fwd(view(*x.q), view(*x.k), view(*x.v), view(o), M.data_ptr<float>(), L.data_ptr<float>(), lse2.data_ptr<float>(),
                                    x.B, x.H, x.Hkv, x.Lq, x.Lk, x.d, scale, x.stream) == LVAR_OK);
  LVAR_NEED(api.lvar_colsum_fwd(view(*x.q), view(*x.k), lse2.data_ptr<float>(), cs.data_ptr<float>(), nullptr, x.B, x.H, x.Hkv, x.Lq, x.Lk, x.d,
                                static_cast<int>(bm), scale, x.stream) == LVAR_OK);
  return tuple(std::move(o), std::move(cs), std::move(M), std::move(L));
  END_HANDLE_TH_ERRORS
}

// (q, k, scale, group rows, M | None, L | None, want block sums, want columns) -> (cs | None, block sums | None)
LVAR_FAST(fast_colsum) {
  HANDLE_TH_ERRORS
  Qkv x;
  float scale;
  int64_t bm;
  bool want_bs, want_cs;
  LVAR_NEED(n == 8 && qkv_ok(x, a[0], a[1], nullptr, true) && as_scale(a[2], x.d, scale) && as_long(a[3], bm) && bm > 0 && bm % 32 == 0 &&
            as_bool(a[6], want_bs) && as_bool(a[7], want_cs) && (want_bs || want_cs));
  const bool given = a[4] != Py_None;
  const int64_t rows = int64_t(x.B) * x.H * x.Lq, G = groups_of(x.Lq, bm);
  const at::Tensor *M = nullptr, *L = nullptr;
  if (given) {
    M = tensor(a[4]); L = tensor(a[5]);
    LVAR_NEED(packed(M, x.dev, at::kFloat) && packed(L, x.dev, at::kFloat) && M->numel() == rows && L->numel() == rows);
  }
  at::Tensor lse2 = empty_stat(x), cs, bs;
  if (given) {
    LVAR_NEED(api.lvar_lse2_from_stats(M->data_ptr<float>(), L->data_ptr<float>(), lse2.data_ptr<float>(), rows, x.stream) == LVAR_OK);
  } else {
    // (block sums alone: the keys stay uncut, see _colsum_block_scores)
    const int64_t bytes = want_cs ? api.lvar_row_lse_scratch_bytes(x.B, x.H, x.Lq, x.Lk) : 0;
    at::Tensor scratch;
    if (bytes > 0) scratch = empty({bytes}, at::kByte, x.dev);
    LVAR_NEED(api.lvar_row_lse_fwd(view(*x.q), view(*x.k), lse2.data_ptr<float>(), bytes > 0 ? scratch.data_ptr() : nullptr, bytes > 0 ? bytes : 0,
                                   x.B, x.H, x.Hkv, x.Lq, x.Lk, x.d, scale, x.stream) == LVAR_OK);
  }
  if (want_cs) cs = empty({x.B, x.H, G, x.Lk}, at::kFloat, x.dev);
  if (want_bs) bs = empty({x.B, x.H, G, (x.Lk + 63) / 64}, at::kFloat, x.dev);
  LVAR_NEED(api.lvar_colsum_fwd(view(*x.q), view(*x.k), lse2.data_ptr<float>(), want_cs ? cs.data_ptr<float>() : nullptr,
                                want_bs ? bs.data_ptr<float>() : nullptr, x.B, x.H, x.Hkv, x.Lq, x.Lk, x.d, static_cast<int>(bm), scale, x.stream) == LVAR_OK);
  return tuple(std::move(cs), std::move(bs));   // (an undefined tensor wraps as None)
  END_HANDLE_TH_ERRORS
}

// key lists of a token-list call: int32, rows of one (batch, head) packed
bool lists_ok(const Qkv& x, const at::Tensor* idx, const at::Tensor* cnt, int64_t bm) {
  if (!idx || !packed(cnt, x.dev, at::kInt) || !idx->is_cuda() || idx->get_device() != x.dev || idx->scalar_type() != at::kInt) return false;
  if (idx->dim() != 4 || cnt->dim() != 3 || bm <= 0) return false;
  const auto s = idx->sizes(), st = idx->strides();
  if (s[0] != x.B || s[1] != x.H || s[2] <= 0 || s[2] > INT32_MAX || s[2] * bm < x.Lq) return false;
  if (cnt->size(0) != s[0] || cnt->size(1) != s[1] || cnt->size(2) != s[2]) return false;
  return st[3] == 1 && st[1] == s[2] * st[2] && st[0] == s[1] * st[1];
}

int csp_launch(const Qkv& x, const at::Tensor& idx, const at::Tensor& cnt, int64_t bm, const at::Tensor* accum, int up_src, int up_dst,
               const at::Tensor& o, float o_scale, float scale) {
  const lvar_tensor_t av = accum ? view(*accum) : lvar_tensor_t{};
  const int G = static_cast<int>(idx.size(2));
  if (up_src > 0)
    return api.lvar_csp_attn_upsample_fwd(view(*x.q), view(*x.k), view(*x.v), av, up_src, up_dst, view(o), nullptr, nullptr, idx.data_ptr<int32_t>(),
                                          cnt.data_ptr<int32_t>(), G, idx.stride(2), static_cast<int>(bm), x.B, x.H, x.Lq, x.Lk, x.d, o_scale, scale, x.stream);
  return api.lvar_csp_attn_fwd(view(*x.q), view(*x.k), view(*x.v), av, view(o), nullptr, nullptr, idx.data_ptr<int32_t>(), cnt.data_ptr<int32_t>(), G,
                               idx.stride(2), static_cast<int>(bm), x.B, x.H, x.Lq, x.Lk, x.d, o_scale, scale, x.stream);
}

// o_accum of a token-list call: shaped like q, or the coarse grid of `up_src` x `up_src` tokens
bool accum_ok(const Qkv& x, const at::Tensor* t, int64_t up_src, int64_t up_dst) {
  if (!rows_ok(t, x.dev) || t->size(0) != x.B || t->size(1) != x.H || t->size(3) != x.d) return false;
  return up_src > 0 ? (t->size(2) == up_src * up_src && up_dst * up_dst == x.Lq) : t->size(2) == x.Lq;
}

// (q, k, v, scale, indices, counts, o_accum, o_scale, group rows, up_src, up_dst) -> o
LVAR_FAST(fast_csp_attn) {
  HANDLE_TH_ERRORS
  Qkv x;
  float scale;
  double o_scale;
  int64_t bm, up_src, up_dst;
  LVAR_NEED(n == 11 && qkv_ok(x, a[0], a[1], a[2], false) && as_scale(a[3], x.d, scale) && as_double(a[7], o_scale) && as_long(a[8], bm) &&
            as_long(a[9], up_src) && as_long(a[10], up_dst) && up_src >= 0 && up_src < 32768 && up_dst < 32768);
  const at::Tensor *idx = tensor(a[4]), *cnt = tensor(a[5]), *acc = tensor(a[6]);
  LVAR_NEED(lists_ok(x, idx, cnt, bm) && idx->size(3) == x.Lk && accum_ok(x, acc, up_src, up_dst));
  at::Tensor o = empty_o(x);
  LVAR_NEED(csp_launch(x, *idx, *cnt, bm, acc, static_cast<int>(up_src), static_cast<int>(up_dst), o, static_cast<float>(o_scale), scale) == LVAR_OK);
  return THPVariable_Wrap(std::move(o));
  END_HANDLE_TH_ERRORS
}

// Decision-scale step of a column-sparse layer (models/sparvar/sparse_attn.py:991-1051): dense attention, column sums,
// top-k key lists and, if wanted, the output cache O - delta(O).
// (q, k, v, scale, group rows, keys per list, want cache) -> (o, indices, counts, cache | None)
LVAR_FAST(fast_full_step) {
  HANDLE_TH_ERRORS
  Qkv x;
  float scale;
  int64_t bm, keep;
  bool want_cache;
  LVAR_NEED(n == 7 && qkv_ok(x, a[0], a[1], a[2], false) && as_scale(a[3], x.d, scale) && as_long(a[4], bm) && bm > 0 && bm % 32 == 0 &&
            as_long(a[5], keep) && keep >= 0 && keep <= x.Lk && as_bool(a[6], want_cache));
  const int64_t G = groups_of(x.Lq, bm);
  at::Tensor o = empty_o(x), lse2 = empty_stat(x), cs = empty({x.B, x.H, G, x.Lk}, at::kFloat, x.dev);
  at::Tensor idx = empty({x.B, x.H, G, x.Lk}, at::kInt, x.dev), cnt = empty({x.B, x.H, G}, at::kInt, x.dev), cache;
  if (want_cache) cache = empty_o(x);
  LVAR_NEED(api.lvar_dense_attn_fwd(view(*x.q), view(*x.k), view(*x.v), view(o), nullptr, nullptr, lse2.data_ptr<float>(),
                                    x.B, x.H, x.Hkv, x.Lq, x.Lk, x.d, scale, x.stream) == LVAR_OK);
  LVAR_NEED(api.lvar_colsum_fwd(view(*x.q), view(*x.k), lse2.data_ptr<float>(), cs.data_ptr<float>(), nullptr, x.B, x.H, x.Hkv, x.Lq, x.Lk, x.d,
                                static_cast<int>(bm), scale, x.stream) == LVAR_OK);
  LVAR_NEED(api.lvar_topk_token_lists(cs.data_ptr<float>(), x.Lk, idx.data_ptr<int32_t>(), x.Lk, cnt.data_ptr<int32_t>(),
                                      static_cast<int>(int64_t(x.B) * x.H * G), x.Lk, static_cast<int>(keep), static_cast<int>(keep), x.stream) == LVAR_OK);
  if (want_cache) LVAR_NEED(csp_launch(x, idx, cnt, bm, &o, 0, 0, cache, -1.f, scale) == LVAR_OK);
  return tuple(std::move(o), std::move(idx), std::move(cnt), std::move(cache));
  END_HANDLE_TH_ERRORS
}

// key list of a sparse step: remapped decision-scale lists, then the local run (see remap_concat_lists)
bool remap(const at::Tensor& src, int64_t count, int64_t Gk, int64_t k_len, const at::Tensor* local, int64_t pad, int64_t out_len, bool zero_tail,
           int dev, void* stream, at::Tensor& idx, at::Tensor& cnt) {
  const int64_t B = src.size(0), H = src.size(1), Gs = src.size(2), Ks = src.size(3);
  const int64_t c = std::max(pad, (count + pad - 1) / pad * pad), L = local ? local->size(1) : 0;
  if (c + L > out_len || out_len > INT32_MAX) return false;
  idx = empty({B, H, Gk, out_len}, at::kInt, dev);
  cnt = empty({B, H, Gk}, at::kInt, dev);
  return api.lvar_remap_concat_lists(src.data_ptr<int32_t>(), Ks, static_cast<int>(Ks), local ? local->data_ptr<int64_t>() : nullptr, L, static_cast<int>(L),
                                     idx.data_ptr<int32_t>(), out_len, cnt.data_ptr<int32_t>(), static_cast<int>(B * H), static_cast<int>(Gs),
                                     static_cast<int>(Gk), static_cast<int>(c), static_cast<int>(k_len), static_cast<int>(zero_tail ? out_len : c + L), stream) == LVAR_OK;
}

// Step of a column-sparse layer after the decision scale (models/sparvar/sparse_attn.py:1053-1144): lists remapped to
// this scale's query groups + local run, then token-list attention on top of the upsampled output cache.
// Lists that no later step reads are not written (head_dim 64 and 128, groups of a multiple of 192 rows).
// (q, k, v, scale, src indices, src count, local, group rows, pad, cache, up_src, up_dst, keep lists) -> (o, indices | None, counts | None)
LVAR_FAST(fast_sparse_step) {
  HANDLE_TH_ERRORS
  Qkv x;
  float scale;
  int64_t count, bm, pad, up_src, up_dst;
  bool keep;
  LVAR_NEED(n == 13 && as_bool(a[12], keep) && qkv_ok(x, a[0], a[1], a[2], false) && as_scale(a[3], x.d, scale) && as_long(a[5], count) && as_long(a[7], bm) && bm > 0 &&
            as_long(a[8], pad) && pad > 0 && as_long(a[10], up_src) && as_long(a[11], up_dst) && up_src > 0 && up_src < 32768 && up_dst < 32768);
  const at::Tensor *src = tensor(a[4]), *local = tensor(a[6]), *cache = tensor(a[9]);
  const int64_t Gk = groups_of(x.Lq, bm);
  LVAR_NEED(packed(src, x.dev, at::kInt) && src->dim() == 4 && src->size(0) == x.B && src->size(1) == x.H && src->size(2) > 0 && count >= 0);
  LVAR_NEED(packed(local, x.dev, at::kLong) && local->dim() == 2 && local->size(0) == Gk && accum_ok(x, cache, up_src, up_dst));
  at::Tensor idx, cnt, o = empty_o(x);
  const int64_t c = std::max(pad, (count + pad - 1) / pad * pad), L = local->size(1), Ks = src->size(3);
  if (!keep && c <= Ks && c + L <= x.Lk) {
    const int st = api.lvar_csp_attn_remap_fwd(view(*x.q), view(*x.k), view(*x.v), view(*cache), static_cast<int>(up_src), static_cast<int>(up_dst), view(o),
                                               src->data_ptr<int32_t>(), Ks, static_cast<int>(Ks), static_cast<int>(src->size(2)), static_cast<int>(c),
                                               L > 0 ? local->data_ptr<int64_t>() : nullptr, L, static_cast<int>(L), static_cast<int>(bm), x.B, x.H, x.Lq,
                                               x.Lk, x.d, 1.f, scale, x.stream);
    if (st == LVAR_OK) return tuple(std::move(o), std::move(idx), std::move(cnt));
    LVAR_NEED(st == LVAR_EUNSUPPORTED);
  }
  LVAR_NEED(remap(*src, count, Gk, x.Lk, local, pad, x.Lk, false, x.dev, x.stream, idx, cnt));
  LVAR_NEED(csp_launch(x, idx, cnt, bm, cache, static_cast<int>(up_src), static_cast<int>(up_dst), o, 1.f, scale) == LVAR_OK);
  return tuple(std::move(o), std::move(idx), std::move(cnt));
  END_HANDLE_TH_ERRORS
}

// (q, k, v, kv_num_blocks, kv_indices, block_q, block_k, scale, want statistics) -> (o, M | None, L | None)
LVAR_FAST(fast_block_sparse_attn) {
  HANDLE_TH_ERRORS
  Qkv x;
  float scale;
  int64_t bq, bk;
  bool stats;
  LVAR_NEED(n == 9 && qkv_ok(x, a[0], a[1], a[2], false) && as_long(a[5], bq) && as_long(a[6], bk) && as_scale(a[7], x.d, scale) && as_bool(a[8], stats));
  LVAR_NEED((bq == 64 || (bq > 0 && bq % 128 == 0 && bq <= INT32_MAX)) && (bk == 64 || bk == 128 || bk == 256));
  const at::Tensor *num = tensor(a[3]), *idx = tensor(a[4]);
  LVAR_NEED(packed(num, x.dev, at::kInt) && packed(idx, x.dev, at::kInt) && num->dim() == 3 && idx->dim() == 4);
  const auto ns = num->sizes(), is = idx->sizes();
  const int64_t nQ = groups_of(x.Lq, bq);
  LVAR_NEED(ns[2] == nQ && is[2] == nQ && (ns[0] == 1 || ns[0] == x.B) && (ns[1] == 1 || ns[1] == x.H) && is[0] == ns[0] && is[1] == ns[1] &&
            is[3] > 0 && is[3] <= INT32_MAX);
  const bool per_b = ns[0] == x.B && x.B > 1, per_h = ns[1] == x.H && x.H > 1;
  at::Tensor o = empty_o(x), M, L;
  if (stats) empty_stats(x, M, L);
  LVAR_NEED(api.lvar_block_sparse_attn_fwd(view(*x.q), view(*x.k), view(*x.v), view(o), stats ? M.data_ptr<float>() : nullptr, stats ? L.data_ptr<float>() : nullptr,
                                           num->data_ptr<int32_t>(), per_b ? num->stride(0) : 0, per_h ? num->stride(1) : 0, idx->data_ptr<int32_t>(),
                                           per_b ? idx->stride(0) : 0, per_h ? idx->stride(1) : 0, is[3], static_cast<int>(is[3]), static_cast<int>(bq),
                                           static_cast<int>(bk), x.B, x.H, x.Lq, x.Lk, x.d, scale, x.stream) == LVAR_OK);
  return tuple(std::move(o), std::move(M), std::move(L));
  END_HANDLE_TH_ERRORS
}

// device and stream of a list-building call: `t` lives on the current device
bool list_call(const at::Tensor* t, int& dev, void*& stream) {
  if (!bound || !t || !t->is_cuda()) return false;
  dev = t->get_device();
  if (c10::hip::current_device() != dev) return false;
  stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream();
  return true;
}

// (block scores, target, base mask | None) -> (kv_num_blocks, kv_indices)
LVAR_FAST(fast_block_topk_lists) {
  HANDLE_TH_ERRORS
  const at::Tensor* s = n == 3 ? tensor(a[0]) : nullptr;
  int dev;
  void* stream;
  int64_t target;
  LVAR_NEED(list_call(s, dev, stream) && packed(s, dev, at::kFloat) && s->dim() == 4 && s->numel() > 0 && as_long(a[1], target) && target >= 0 && target <= INT32_MAX);
  const int64_t B = s->size(0), H = s->size(1), nQ = s->size(2), nK = s->size(3);
  const at::Tensor* base = a[2] == Py_None ? nullptr : tensor(a[2]);
  if (a[2] != Py_None) LVAR_NEED(base && base->dim() == 2 && base->size(0) == nQ && base->size(1) == nK && (packed(base, dev, at::kBool) || packed(base, dev, at::kByte)));
  LVAR_NEED(nK <= 2048 && B * H * nQ <= INT32_MAX);
  at::Tensor num = empty({B, H, nQ}, at::kInt, dev), idx = empty({B, H, nQ, nK}, at::kInt, dev);
  LVAR_NEED(api.lvar_block_topk_lists(s->data_ptr<float>(), base ? static_cast<const uint8_t*>(base->data_ptr()) : nullptr, num.data_ptr<int32_t>(),
                                      idx.data_ptr<int32_t>(), static_cast<int>(B), static_cast<int>(H), static_cast<int>(nQ), static_cast<int>(nK),
                                      static_cast<int>(target), stream) == LVAR_OK);
  return tuple(std::move(num), std::move(idx));
  END_HANDLE_TH_ERRORS
}

// (scores, k, out_len, zero_tail) -> (indices, counts)
LVAR_FAST(fast_topk_token_lists) {
  HANDLE_TH_ERRORS
  const at::Tensor* s = n == 4 ? tensor(a[0]) : nullptr;
  int dev;
  void* stream;
  int64_t k, out_len;
  bool zero_tail;
  LVAR_NEED(list_call(s, dev, stream) && packed(s, dev, at::kFloat) && s->dim() >= 1 && s->numel() > 0 && as_long(a[1], k) && as_long(a[2], out_len) && as_bool(a[3], zero_tail));
  const int64_t n_col = s->size(-1), rows = s->numel() / n_col;
  LVAR_NEED(k >= 0 && k <= n_col && out_len >= k && out_len <= INT32_MAX && rows <= INT32_MAX && n_col <= INT32_MAX);
  std::vector<int64_t> shape = s->sizes().vec();
  shape.back() = out_len;
  at::Tensor idx = empty(shape, at::kInt, dev);
  shape.pop_back();
  at::Tensor cnt = empty(shape, at::kInt, dev);
  LVAR_NEED(api.lvar_topk_token_lists(s->data_ptr<float>(), n_col, idx.data_ptr<int32_t>(), out_len, cnt.data_ptr<int32_t>(), static_cast<int>(rows),
                                      static_cast<int>(n_col), static_cast<int>(k), static_cast<int>(zero_tail ? out_len : k), stream) == LVAR_OK);
  return tuple(std::move(idx), std::move(cnt));
  END_HANDLE_TH_ERRORS
}

// (src indices, src count, query groups, k_len, local | None, pad, out_len, zero_tail) -> (indices, counts)
LVAR_FAST(fast_remap_concat_lists) {
  HANDLE_TH_ERRORS
  const at::Tensor* src = n == 8 ? tensor(a[0]) : nullptr;
  int dev;
  void* stream;
  int64_t count, Gk, k_len, pad, out_len;
  bool zero_tail;
  LVAR_NEED(list_call(src, dev, stream) && packed(src, dev, at::kInt) && src->dim() == 4 && src->numel() > 0 && as_long(a[1], count) && as_long(a[2], Gk) &&
            as_long(a[3], k_len) && as_long(a[5], pad) && as_long(a[6], out_len) && as_bool(a[7], zero_tail) && count >= 0 && Gk > 0 && pad > 0 && k_len > 0);
  const at::Tensor* local = a[4] == Py_None ? nullptr : tensor(a[4]);
  if (a[4] != Py_None) LVAR_NEED(packed(local, dev, at::kLong) && local->dim() == 2 && local->size(0) == Gk);
  at::Tensor idx, cnt;
  LVAR_NEED(remap(*src, count, Gk, k_len, local, pad, out_len, zero_tail, dev, stream, idx, cnt));
  return tuple(std::move(idx), std::move(cnt));
  END_HANDLE_TH_ERRORS
}

// (bool mask, multiple) -> (counts, indices)
LVAR_FAST(fast_mask_to_lists) {
  HANDLE_TH_ERRORS
  const at::Tensor* m = n == 2 ? tensor(a[0]) : nullptr;
  int dev;
  void* stream;
  int64_t mult;
  LVAR_NEED(list_call(m, dev, stream) && packed(m, dev, at::kBool) && m->dim() >= 1 && m->numel() > 0 && as_long(a[1], mult) && mult > 0 && mult <= INT32_MAX);
  const int64_t n_col = m->size(-1), rows = m->numel() / n_col;
  LVAR_NEED(n_col <= INT32_MAX && rows <= INT32_MAX);
  at::Tensor idx = empty(m->sizes(), at::kInt, dev), cnt = empty(m->sizes().slice(0, m->dim() - 1), at::kInt, dev);
  LVAR_NEED(api.lvar_mask_to_lists(static_cast<const uint8_t*>(m->data_ptr()), n_col, idx.data_ptr<int32_t>(), n_col, cnt.data_ptr<int32_t>(),
                                   static_cast<int>(rows), static_cast<int>(n_col), static_cast<int>(mult), stream) == LVAR_OK);
  return tuple(std::move(cnt), std::move(idx));
  END_HANDLE_TH_ERRORS
}

// (q, k, window keys, pool kernel size, max pool, scale, keep) -> keep > 0: the kept positions, int64 [B,H,keep+W], the
// `keep` best-scoring keys and the window keys in ascending order; keep = 0: the scores, fp32 [B,H,Lk]
LVAR_FAST(fast_window_keys) {
  HANDLE_TH_ERRORS
  Qkv x;
  float scale;
  int64_t ksize, keep;
  bool maxpool;
  LVAR_NEED(n == 7 && qkv_ok(x, a[0], a[1], nullptr, false) && as_long(a[3], ksize) && as_bool(a[4], maxpool) && as_scale(a[5], x.d, scale) && as_long(a[6], keep));
  const at::Tensor* win = tensor(a[2]);
  LVAR_NEED(packed(win, x.dev, at::kLong) && win->dim() == 3 && win->size(0) == x.B && win->size(1) == x.H && win->size(2) > 0 && win->size(2) <= 65535);
  LVAR_NEED(x.Lq <= x.Lk && ksize % 2 == 1 && ksize >= 1 && ksize <= 33 && keep >= 0 && keep <= x.Lk);
  const int W = static_cast<int>(win->size(2));
  if (keep > 0) LVAR_NEED(x.Lk <= 16384);
  at::Tensor scores = empty({x.B, x.H, x.Lk}, at::kFloat, x.dev), out;
  if (keep > 0) out = empty({x.B, x.H, keep + W}, at::kLong, x.dev);
  LVAR_NEED(api.lvar_window_key_scores(view(*x.q), view(*x.k), win->data_ptr<int64_t>(), W, scores.data_ptr<float>(), x.B, x.H, x.Lq, x.Lk, x.d,
                                       static_cast<int>(ksize), maxpool ? 1 : 0, scale, x.stream) == LVAR_OK);
  if (keep == 0) return THPVariable_Wrap(std::move(scores));
  LVAR_NEED(api.lvar_topk_union_lists(scores.data_ptr<float>(), x.Lk, win->data_ptr<int64_t>(), W, out.data_ptr<int64_t>(), x.B * x.H, x.Lk,
                                      static_cast<int>(keep), x.stream) == LVAR_OK);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// rows are read with 16-byte accesses: anything else is copied into a plain tensor first
at::Tensor as_plain(const at::Tensor& t, const char* name) {
  TORCH_CHECK(t.dim() == 4, name, " must be [B,H,L,d], got ", t.sizes());
  TORCH_CHECK(t.scalar_type() == at::kBFloat16, name, " must be bfloat16, got ", t.scalar_type());
  TORCH_CHECK(t.is_cuda(), name, " must live on a HIP device; lvar_amd has no CPU path");
  if (plain(t)) return t;
  at::Tensor c = t.contiguous();
  if (reinterpret_cast<uintptr_t>(c.data_ptr()) & 15u) c = c.clone();
  return c;
}

// <ns>::dense_attn(q, k, v) -> [o, 1/(2^M L)]
std::vector<at::Tensor> op_dense_attn(const at::Tensor& q_in, const at::Tensor& k_in, const at::Tensor& v_in) {
  TORCH_CHECK(bound, "lvar_amd: the C-ABI library is not bound");
  const at::Tensor q = as_plain(q_in, "q"), k = as_plain(k_in, "k"), v = as_plain(v_in, "v");
  const int64_t B = q.size(0), H = q.size(1), Lq = q.size(2), d = q.size(3), Lk = k.size(2);
  TORCH_CHECK(k.sizes() == v.sizes(), "k/v shape mismatch: ", k.sizes(), " vs ", v.sizes());
  const int64_t Hkv = k.size(1);
  TORCH_CHECK(k.size(0) == B && Hkv > 0 && H % Hkv == 0 && k.size(3) == d, "q/k batch, head or head_dim mismatch: ", q.sizes(), " vs ", k.sizes());
  TORCH_CHECK(q.get_device() == k.get_device() && q.get_device() == v.get_device(), "q, k, v must be on the same device");
  TORCH_CHECK(Lq <= INT32_MAX && Lk <= INT32_MAX, "sequence too long");
  const c10::DeviceGuard guard(q.device());   // the tensors' device is current for the allocations and the launch
  at::Tensor o = at::empty_like(q);
  at::Tensor rcp = at::empty({B, H, Lq, 1}, q.options().dtype(at::kFloat));
  void* stream = c10::hip::getCurrentHIPStream(q.get_device()).stream();
  const int st = api.lvar_dense_attn_rcp_fwd(view(q), view(k), view(v), view(o), rcp.data_ptr<float>(), static_cast<int>(B), static_cast<int>(H), static_cast<int>(Hkv),
                             static_cast<int>(Lq), static_cast<int>(Lk), static_cast<int>(d), 1.0f, stream);
  TORCH_CHECK(st == LVAR_OK, "lvar_dense_attn_rcp_fwd failed with status ", st,
              st == LVAR_EUNSUPPORTED ? " (unsupported head_dim)" : st == LVAR_EINVAL ? " (invalid argument)" : " (launch failed)");
  return {o, rcp};
}

// Libraries registered by register_dense_attn live until the process ends (as a TORCH_LIBRARY block's would).
std::vector<std::unique_ptr<torch::Library>>& libraries() {
  static std::vector<std::unique_ptr<torch::Library>> libs;
  return libs;
}

void register_dense_attn(const std::string& ns) {
  auto lib = std::make_unique<torch::Library>(torch::Library::FRAGMENT, ns, std::nullopt, __FILE__, __LINE__);
  lib->def("dense_attn(Tensor q, Tensor k, Tensor v) -> Tensor[]");
  lib->impl("dense_attn", torch::dispatch(c10::DispatchKey::CUDA, TORCH_FN(op_dense_attn)));
  libraries().push_back(std::move(lib));
}

#define LVAR_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef fast_methods[] = {
    LVAR_METHOD(fast_dense_attn), LVAR_METHOD(fast_dense_colsum_attn), LVAR_METHOD(fast_colsum), LVAR_METHOD(fast_csp_attn),
    LVAR_METHOD(fast_full_step), LVAR_METHOD(fast_sparse_step), LVAR_METHOD(fast_block_sparse_attn), LVAR_METHOD(fast_block_topk_lists),
    LVAR_METHOD(fast_topk_token_lists), LVAR_METHOD(fast_remap_concat_lists), LVAR_METHOD(fast_mask_to_lists), LVAR_METHOD(fast_window_keys),
    {nullptr, nullptr, 0, nullptr}};

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
  m.def("entry_names", &entry_names, "names of the C-ABI entry points that bind() takes the addresses of");
  m.def("bind", &bind);
  m.def("register_dense_attn", &register_dense_attn, "define and implement <ns>::dense_attn natively");
  if (PyModule_AddFunctions(m.ptr(), fast_methods) != 0) throw pybind11::error_already_set();
}
