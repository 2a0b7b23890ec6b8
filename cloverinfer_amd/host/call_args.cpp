// call_args.cpp - the argument blocks of the C ABI from tensors, in native code.
//
// kernels.py checks a call's tensors and copies some twenty-five pointers,
// sizes and strides into a ctypes structure. In Python that is most of the
// host's share of a small call: a KV append of 16 rows took 10 us a call with
// a kernel of 2 us. These functions make the same checks and fill the same
// structure in one call; they return false where any check fails or an object
// is not a plain tensor, and the Python code then does it all again and raises
// its own error (or takes what this one does not).
#include "call_args.h"

#include <clover_attn.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/extension.h>

#include <cmath>
#include <cstddef>
#include <limits>

namespace clv_host {
namespace {

// A plain strided device tensor (torch.Tensor or Parameter, no subclass that
// may override its methods), or null.
const at::Tensor *plain(const py::object &o) {
  if (!THPVariable_CheckExact(o.ptr())) return nullptr;
  const at::Tensor &t = THPVariable_Unpack(o.ptr());
  if (!t.defined() || t.layout() != at::kStrided || !t.has_storage() ||
      t.device().type() != at::kCUDA)
    return nullptr;
  return &t;
}

bool fits32(int64_t x) { return x >= 0 && x <= std::numeric_limits<int32_t>::max(); }

bool dtype_code(at::ScalarType t, int32_t *out) {
  switch (t) {
    case at::kFloat: *out = CLV_F32; return true;
    case at::kHalf: *out = CLV_F16; return true;
    case at::kBFloat16: *out = CLV_BF16; return true;
    default: return false;
  }
}

// [num_blocks, block_size, num_kv_heads, head_dim] pools of one shape, dtype
// and strides.
bool pools_ok(const at::Tensor &k, const at::Tensor &v) {
  return k.dim() == 4 && v.sizes() == k.sizes() && v.strides() == k.strides() &&
         k.stride(3) == 1 && v.scalar_type() == k.scalar_type() && fits32(k.size(0)) &&
         fits32(k.size(1)) && fits32(k.size(2)) && fits32(k.size(3));
}

// dtype rules shared by queries / new rows (x) and pools: equal, or e4m3
// pools; *fp8 tells which.
bool dtypes_ok(const at::Tensor &x, const at::Tensor &k, bool *fp8) {
  *fp8 = k.scalar_type() == at::kFloat8_e4m3fn;
  return *fp8 || x.scalar_type() == k.scalar_type();
}

bool int_vector(const at::Tensor &t, at::ScalarType dt, int64_t n) {
  return t.scalar_type() == dt && t.dim() == 1 && t.size(0) == n && t.is_contiguous();
}

bool int_matrix(const at::Tensor &t, int64_t rows) {
  return t.scalar_type() == at::kInt && t.dim() == 2 && t.size(0) == rows && t.is_contiguous() &&
         fits32(t.size(1));
}

// q and out: [rows, num_heads, head_dim] with a contiguous last dimension.
bool rows_ok(const at::Tensor &q, const at::Tensor &out) {
  return q.dim() == 3 && out.sizes() == q.sizes() && out.scalar_type() == q.scalar_type() &&
         q.stride(2) == 1 && out.stride(2) == 1 && fits32(q.size(0)) && fits32(q.size(1));
}

// The softmax scale: 1/sqrt(head_dim) for None.
bool scale_of(const py::object &scale, int64_t head_dim, float *out) {
  if (scale.is_none()) {
    *out = (float)(1.0 / std::sqrt((double)head_dim));
    return true;
  }
  const double x = PyFloat_AsDouble(scale.ptr());
  if (x == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  *out = (float)x;
  return true;
}

template <typename... Ts>
bool same_device(const at::Tensor &a, const Ts &...ts) {
  return ((ts.device() == a.device()) && ...);
}

}  // namespace

bool fill_decode_args(uintptr_t dst, py::object out_, py::object q_, py::object k_, py::object v_,
                      py::object bt_, py::object cl_, int64_t block_size, int64_t max_context_len,
                      py::object scale) {
  const at::Tensor *out = plain(out_), *q = plain(q_), *k = plain(k_), *v = plain(v_),
                   *bt = plain(bt_), *cl = plain(cl_);
  if (!out || !q || !k || !v || !bt || !cl || !same_device(*out, *q, *k, *v, *bt, *cl))
    return false;
  bool fp8;
  clv_decode_args a{};
  if (!rows_ok(*q, *out) || !pools_ok(*k, *v) || !dtypes_ok(*q, *k, &fp8) ||
      !dtype_code(q->scalar_type(), &a.dtype) || (fp8 && a.dtype == CLV_F32) ||
      !scale_of(scale, q->size(2), &a.scale))
    return false;
  if (k->size(3) != q->size(2) || k->size(1) != block_size || k->size(2) == 0 ||
      q->size(1) % k->size(2) != 0 || !fits32(max_context_len))
    return false;
  if (!int_matrix(*bt, q->size(0)) || !int_vector(*cl, at::kInt, q->size(0))) return false;
  a.out = out->data_ptr();
  a.q = q->data_ptr();
  a.k_cache = k->data_ptr();
  a.v_cache = v->data_ptr();
  a.block_tables = (const int32_t *)bt->data_ptr();
  a.context_lens = (const int32_t *)cl->data_ptr();
  a.q_stride_seq = q->stride(0);
  a.q_stride_head = q->stride(1);
  a.out_stride_seq = out->stride(0);
  a.out_stride_head = out->stride(1);
  a.kv_stride_block = k->stride(0);
  a.kv_stride_token = k->stride(1);
  a.kv_stride_head = k->stride(2);
  a.num_seqs = (int32_t)q->size(0);
  a.num_heads = (int32_t)q->size(1);
  a.num_kv_heads = (int32_t)k->size(2);
  a.head_dim = (int32_t)q->size(2);
  a.block_size = (int32_t)block_size;
  a.max_blocks_per_seq = (int32_t)bt->size(1);
  a.max_context_len = (int32_t)max_context_len;
  a.num_blocks = (int32_t)k->size(0);
  *reinterpret_cast<clv_decode_args *>(dst) = a;
  return true;
}

bool fill_prefill_args(uintptr_t dst, py::object out_, py::object q_, py::object k_, py::object v_,
                       py::object bt_, py::object cl_, py::object qsl_, int64_t max_query_len,
                       py::object scale) {
  const at::Tensor *out = plain(out_), *q = plain(q_), *k = plain(k_), *v = plain(v_),
                   *bt = plain(bt_), *cl = plain(cl_), *qsl = plain(qsl_);
  if (!out || !q || !k || !v || !bt || !cl || !qsl ||
      !same_device(*out, *q, *k, *v, *bt, *cl, *qsl))
    return false;
  bool fp8;
  clv_prefill_args a{};
  if (!rows_ok(*q, *out) || !pools_ok(*k, *v) || !dtypes_ok(*q, *k, &fp8) || fp8 ||
      !dtype_code(q->scalar_type(), &a.dtype) || !scale_of(scale, q->size(2), &a.scale))
    return false;
  if (k->size(3) != q->size(2) || k->size(2) == 0 || q->size(1) % k->size(2) != 0 ||
      cl->dim() != 1 || !fits32(max_query_len))
    return false;
  const int64_t num_seqs = cl->size(0);
  if (!fits32(num_seqs) || !int_matrix(*bt, num_seqs) || !int_vector(*cl, at::kInt, num_seqs) ||
      !int_vector(*qsl, at::kInt, num_seqs + 1))
    return false;
  a.out = out->data_ptr();
  a.q = q->data_ptr();
  a.k_cache = k->data_ptr();
  a.v_cache = v->data_ptr();
  a.block_tables = (const int32_t *)bt->data_ptr();
  a.context_lens = (const int32_t *)cl->data_ptr();
  a.query_start_loc = (const int32_t *)qsl->data_ptr();
  a.q_stride_token = q->stride(0);
  a.q_stride_head = q->stride(1);
  a.out_stride_token = out->stride(0);
  a.out_stride_head = out->stride(1);
  a.kv_stride_block = k->stride(0);
  a.kv_stride_token = k->stride(1);
  a.kv_stride_head = k->stride(2);
  a.num_seqs = (int32_t)num_seqs;
  a.num_tokens = (int32_t)q->size(0);
  a.num_heads = (int32_t)q->size(1);
  a.num_kv_heads = (int32_t)k->size(2);
  a.head_dim = (int32_t)q->size(2);
  a.block_size = (int32_t)k->size(1);
  a.max_blocks_per_seq = (int32_t)bt->size(1);
  a.max_query_len = (int32_t)max_query_len;
  a.num_blocks = (int32_t)k->size(0);
  *reinterpret_cast<clv_prefill_args *>(dst) = a;
  return true;
}

bool fill_cache_args(uintptr_t dst, py::object key_, py::object value_, py::object k_,
                     py::object v_, py::object slots_) {
  const at::Tensor *key = plain(key_), *value = plain(value_), *k = plain(k_), *v = plain(v_),
                   *slots = plain(slots_);
  if (!key || !value || !k || !v || !slots || !same_device(*key, *value, *k, *v, *slots))
    return false;
  bool fp8;
  clv_cache_args a{};
  if (!pools_ok(*k, *v) || key->dim() != 3 || value->sizes() != key->sizes() ||
      key->size(1) != k->size(2) || key->size(2) != k->size(3) || !fits32(key->size(0)) ||
      value->scalar_type() != key->scalar_type() || !dtypes_ok(*key, *k, &fp8) ||
      !dtype_code(key->scalar_type(), &a.dtype) || key->stride(2) != 1 || value->stride(2) != 1 ||
      !int_vector(*slots, at::kLong, key->size(0)))
    return false;
  a.key = key->data_ptr();
  a.value = value->data_ptr();
  a.k_cache = k->data_ptr();
  a.v_cache = v->data_ptr();
  a.slot_mapping = (const int64_t *)slots->data_ptr();
  a.key_stride_token = key->stride(0);
  a.key_stride_head = key->stride(1);
  a.value_stride_token = value->stride(0);
  a.value_stride_head = value->stride(1);
  a.kv_stride_block = k->stride(0);
  a.kv_stride_token = k->stride(1);
  a.kv_stride_head = k->stride(2);
  a.num_tokens = (int32_t)key->size(0);
  a.num_kv_heads = (int32_t)k->size(2);
  a.head_dim = (int32_t)k->size(3);
  a.block_size = (int32_t)k->size(1);
  a.num_blocks = (int32_t)k->size(0);
  *reinterpret_cast<clv_cache_args *>(dst) = a;
  return true;
}

py::tuple call_args_layout() {
  return py::make_tuple(
      (size_t)CLV_ABI_VERSION, sizeof(clv_decode_args), offsetof(clv_decode_args, dtype),
      offsetof(clv_decode_args, scale), sizeof(clv_prefill_args), offsetof(clv_prefill_args, dtype),
      offsetof(clv_prefill_args, scale), sizeof(clv_cache_args), offsetof(clv_cache_args, dtype));
}

}  // namespace clv_host
