// The framework's calls on torch tensors, without the interpreter between their steps: the ordinary form of each entry point of the
// Python package is checked, allocated for and launched here. A function returns None, with nothing done, where a call is of any
// other form (another device than the current one, a dtype, shape or stride that the checks below do not name, a tensor subclass, a
// dispatch mode, a transform); the Python code then takes it, or refuses it with its own error.
//
// What bounds a small call is the host: a decode of 1 x 1320 keys is 10.8 us of kernels, and was 16.1 us of calls (two launches 7.2, two
// torch.empty 3.1, 33 arguments through ctypes 1.5, the rest Python).
#include <Python.h>

#include <torch/csrc/Device.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ops/empty.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/Allocator.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <climits>
#include <initializer_list>
#include <utility>

#include "tdist.h"

namespace {

PyObject* g_error = nullptr;   // TdistError

// ---- ordinary arguments --------------------------------------------------------------------------------------
// Nothing between a call and its tensors: no __torch_function__ or dispatch mode, no transform, no tracing.
bool plain_state() {
  constexpr c10::DispatchKeySet kUsual({c10::DispatchKey::BackendSelect, c10::DispatchKey::ADInplaceOrView});
  return kUsual.has_all(c10::impl::tls_local_dispatch_key_set().included_) && !at::impl::torch_function_mode_enabled();
}

// A strided tensor of the GPU `device` that is a plain torch.Tensor, else NULL.
const at::Tensor* tensor_of(PyObject* o, int device) {
  constexpr c10::DispatchKeySet kUsual({c10::DispatchKey::CUDA, c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutogradCUDA,
                                        c10::DispatchKey::AutocastCUDA});
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.defined() || !kUsual.has_all(t.key_set()) || t.layout() != c10::kStrided || !t.has_storage() || t.get_device() != device) return nullptr;
  for (int64_t n : t.sizes())
    if (n > INT_MAX) return nullptr;
  return &t;
}
const at::Tensor* tensor_of(PyObject* o, int device, c10::ScalarType type, int64_t dim) {
  const at::Tensor* t = tensor_of(o, device);
  return t && t->scalar_type() == type && t->dim() == dim ? t : nullptr;
}
// `o` is None (`*t` NULL) or a contiguous tensor of this type.
bool optional_of(PyObject* o, int device, c10::ScalarType type, const at::Tensor** t) {
  *t = nullptr;
  if (o == Py_None) return true;
  *t = tensor_of(o, device);
  return *t && (*t)->scalar_type() == type && (*t)->is_contiguous();
}
bool int_of(PyObject* o, int* v) {
  if (!PyLong_CheckExact(o)) return false;
  int overflow = 0;
  const long x = PyLong_AsLongAndOverflow(o, &overflow);
  if (overflow || x < INT_MIN || x > INT_MAX) return false;
  *v = (int)x;
  return true;
}
bool float_of(PyObject* o, float* v) {
  if (PyFloat_CheckExact(o)) return *v = (float)PyFloat_AS_DOUBLE(o), true;
  int i;
  return int_of(o, &i) && (*v = (float)i, true);
}
bool code_of(c10::ScalarType t, int* code) {
  switch (t) {
    case c10::ScalarType::BFloat16: *code = TDIST_BF16; return true;
    case c10::ScalarType::Half: *code = TDIST_F16; return true;
    case c10::ScalarType::Float8_e4m3fn: *code = TDIST_F8E4M3; return true;
    default: return false;
  }
}
bool aligned16(const at::Tensor& t) { return ((uintptr_t)t.data_ptr() & 15) == 0; }
void* ptr(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }
int32_t* i32(const at::Tensor* t) { return (int32_t*)t->data_ptr(); }
// an optional workspace's address and size
bool workspace_of(PyObject* o, int device, void** p, int64_t* bytes) {
  *p = nullptr, *bytes = 0;
  if (o == Py_None) return true;
  const at::Tensor* t = tensor_of(o, device);
  return t && (*p = t->data_ptr(), *bytes = t->numel() * t->element_size(), true);
}

at::Tensor empty_on(int device, c10::ScalarType type, at::IntArrayRef sizes) {
  return at::empty(sizes, at::TensorOptions().dtype(type).device(c10::Device(c10::kCUDA, (c10::DeviceIndex)device)));
}
void* stream_of(int device) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

// Runs `launch` without the GIL; raises TdistError and returns false where it fails.
template <typename F>
bool run(F&& launch) {
  int rc;
  Py_BEGIN_ALLOW_THREADS
  rc = launch();
  Py_END_ALLOW_THREADS
  if (rc == TDIST_OK) return true;
  PyObject* e = PyObject_CallFunction(g_error, "is", rc, tdist_last_error_string());
  if (e) PyErr_SetObject(g_error, e);
  Py_XDECREF(e);
  return false;
}

// `first`: an argument that is a tensor of the GPU in an ordinary call (the runtime is not asked for a device before one is seen)
#define TDIST_ARGS(n, first)                                                                                             \
  HANDLE_TH_ERRORS                                                                                                       \
  if (nargs != n) return PyErr_Format(PyExc_TypeError, "%d arguments, not %zd", n, nargs);                                \
  if (!plain_state() || !THPVariable_CheckExact(o[first]) || !THPVariable_Unpack(o[first]).is_cuda()) Py_RETURN_NONE;     \
  const int device = (int)c10::hip::current_device()
#define TDIST_ORDINARY(cond) \
  do {                       \
    if (!(cond)) Py_RETURN_NONE; \
  } while (0)

// ---- decode --------------------------------------------------------------------------------------------------
struct Decode {
  const at::Tensor *q, *k, *v, *table;
  float scale, soft_cap;
  int batch, q_heads, kv_heads, dk, dv, page, code;
  int64_t workspace;
};
// q, k_cache, v_cache and the page table (o[0], o[1], o[2], o[3]), scale and soft cap (o[4], o[5])
bool decode_of(PyObject* const* o, int device, Decode& d) {
  d.q = tensor_of(o[0], device), d.k = tensor_of(o[1], device), d.v = tensor_of(o[2], device);
  d.table = tensor_of(o[3], device, c10::ScalarType::Int, 2);
  if (!d.q || !d.k || !d.v || !d.table || !float_of(o[4], &d.scale) || !float_of(o[5], &d.soft_cap)) return false;
  const at::Tensor &q = *d.q, &k = *d.k, &v = *d.v;
  const auto type = q.scalar_type();
  if (type != c10::ScalarType::BFloat16 && type != c10::ScalarType::Half) return false;
  if (k.scalar_type() != type || v.scalar_type() != type || q.dim() != 3 || k.dim() != 4 || v.dim() != 4) return false;
  if (q.stride(2) != 1 || k.stride(3) != 1 || v.stride(3) != 1 || d.table->stride(1) != 1) return false;
  d.batch = (int)q.size(0), d.q_heads = (int)q.size(1), d.dk = (int)q.size(2);
  d.page = (int)v.size(1), d.kv_heads = (int)v.size(2), d.dv = (int)v.size(3);
  if (k.size(1) != d.page || k.size(2) != d.kv_heads || k.size(3) != d.dk) return false;
  if (d.batch <= 0 || d.kv_heads <= 0 || d.q_heads <= 0 || d.q_heads % d.kv_heads != 0) return false;
  const bool even = d.dk == d.dv && d.dk > 0 && d.dk <= 256 && d.dk % 8 == 0;
  if (!even && !(d.dk == 192 && d.dv == 128) && !(d.dk == 576 && d.dv == 512)) return false;
  // (these heads stream where the value is a view of the key only)
  if (d.dk > 256 && (k.data_ptr() != v.data_ptr() || k.strides() != v.strides())) return false;
  d.workspace = tdist_decode_stream_workspace_bytes(d.batch, d.q_heads, d.kv_heads, d.dk, d.dv);
  return d.workspace > 0 && code_of(type, &d.code);
}

// decode(q, k_cache, v_cache, block_table, scale, soft_cap, kv_lens) -> out
PyObject* decode(PyObject*, PyObject* const* o, Py_ssize_t nargs) {
  TDIST_ARGS(7, 0);
  Decode d;
  TDIST_ORDINARY(decode_of(o, device, d));
  const at::Tensor* lens = tensor_of(o[6], device, c10::ScalarType::Int, 1);
  TDIST_ORDINARY(lens && lens->is_contiguous());
  const at::Tensor &q = *d.q, &k = *d.k, &v = *d.v;
  at::Tensor out = empty_on(device, q.scalar_type(), {d.batch, d.q_heads, d.dv});
  const c10::DataPtr workspace = c10::GetAllocator(c10::kCUDA)->allocate(d.workspace);
  void* const stream = stream_of(device);
  if (!run([&] {
        return tdist_decode_stream(q.data_ptr(), k.data_ptr(), v.data_ptr(), d.scale, d.soft_cap, (const int32_t*)d.table->data_ptr(),
                                   (const int32_t*)lens->data_ptr(), d.batch, d.q_heads, d.kv_heads, d.dk, d.dv, d.page, q.stride(0), q.stride(1),
                                   k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2), d.table->stride(0), d.code, nullptr,
                                   0, workspace.get(), d.workspace, out.data_ptr(), d.code, out.stride(0), out.stride(1), nullptr, stream);
      })) return nullptr;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// decode_ranks(q, k_cache, v_cache, block_table, scale, soft_cap, global_kv_lens, rank, num_ranks, q_heads, v_head_dim, max_batch, all_out,
// all_lse) -> out
PyObject* decode_ranks(PyObject*, PyObject* const* o, Py_ssize_t nargs) {
  TDIST_ARGS(14, 0);
  Decode d;
  int rank, ranks, q_heads, dv, max_batch, out_code;
  TDIST_ORDINARY(decode_of(o, device, d) && int_of(o[7], &rank) && int_of(o[8], &ranks) && int_of(o[9], &q_heads) && int_of(o[10], &dv) &&
                 int_of(o[11], &max_batch));
  const at::Tensor* lens = tensor_of(o[6], device, c10::ScalarType::Int, 2);
  const at::Tensor *all_out = tensor_of(o[12], device), *all_lse = tensor_of(o[13], device, c10::ScalarType::Float, 3);
  TDIST_ORDINARY(lens && lens->is_contiguous() && lens->size(0) == ranks && lens->size(1) == d.batch && rank >= 0 && rank < ranks);
  TDIST_ORDINARY(q_heads == d.q_heads && dv == d.dv && d.batch <= max_batch);
  TDIST_ORDINARY(all_out && all_out->dim() == 4 && all_out->size(0) == ranks && all_out->size(1) == d.batch && all_out->size(2) == d.q_heads &&
                 all_out->size(3) == d.dv && all_out->stride(3) == 1 &&
                 (all_out->scalar_type() == c10::ScalarType::BFloat16 || all_out->scalar_type() == c10::ScalarType::Half ||
                  all_out->scalar_type() == c10::ScalarType::Float));
  out_code = all_out->scalar_type() == c10::ScalarType::Float ? TDIST_F32 : all_out->scalar_type() == c10::ScalarType::Half ? TDIST_F16 : TDIST_BF16;
  TDIST_ORDINARY(all_lse && all_lse->size(0) == ranks && all_lse->size(1) == d.batch && all_lse->size(2) == d.q_heads && all_lse->stride(2) == 1 &&
                 all_lse->stride(1) == d.q_heads);
  const at::Tensor &q = *d.q, &k = *d.k, &v = *d.v;
  const c10::DataPtr workspace = c10::GetAllocator(c10::kCUDA)->allocate(d.workspace);
  at::Tensor out = empty_on(device, q.scalar_type(), {d.batch, d.q_heads, d.dv});
  void* const stream = stream_of(device);
  if (!run([&] {
        return tdist_decode_stream_ranks(q.data_ptr(), k.data_ptr(), v.data_ptr(), d.scale, d.soft_cap, (const int32_t*)d.table->data_ptr(),
                                         (const int32_t*)lens->data_ptr(), rank, ranks, d.batch, d.q_heads, d.kv_heads, d.dk, d.dv, d.page, q.stride(0),
                                         q.stride(1), k.stride(0), k.stride(1), k.stride(2), v.stride(0), v.stride(1), v.stride(2), d.table->stride(0),
                                         d.code, workspace.get(), d.workspace, all_out->data_ptr(), out_code, all_out->stride(0), all_out->stride(1),
                                         all_out->stride(2), (float*)all_lse->data_ptr(), all_lse->stride(0), out.data_ptr(), d.code, stream);
      })) return nullptr;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ---- GEMMs ---------------------------------------------------------------------------------------------------
// The table of every rank's shard: `own` at `rank`, the others from a dict rank -> tensor.
bool shards_of(const at::Tensor& own, PyObject* peers, int rank, int ranks, int device, const void** table) {
  if (!PyDict_CheckExact(peers) || ranks < 2 || ranks > TDIST_GATHER_MAX_RANKS || rank < 0 || rank >= ranks || !aligned16(own)) return false;
  int found = 1;
  table[rank] = own.data_ptr();
  PyObject *key, *value;
  for (Py_ssize_t pos = 0; PyDict_Next(peers, &pos, &key, &value);) {
    int r;
    if (!int_of(key, &r) || r < 0 || r >= ranks) return false;
    if (r == rank) continue;
    const at::Tensor* t = tensor_of(value, device);
    if (!t || !aligned16(*t)) return false;
    table[r] = t->data_ptr();
    ++found;
  }
  return found == ranks;
}
// a and b [rows, K] of one GEMM type with contiguous rows (a: whole), the type's code and the type of the results
bool operands_of(PyObject* ao, PyObject* bo, int device, const at::Tensor** a, const at::Tensor** b, int* code, c10::ScalarType* out) {
  *a = tensor_of(ao, device), *b = tensor_of(bo, device);
  if (!*a || !*b || (*a)->dim() != 2 || (*b)->dim() != 2 || (*a)->scalar_type() != (*b)->scalar_type()) return false;
  if (!(*a)->is_contiguous() || (*b)->stride(1) != 1 || (*a)->size(1) != (*b)->size(1) || (*a)->numel() == 0 || (*b)->numel() == 0) return false;
  if (!code_of((*a)->scalar_type(), code)) return false;
  *out = *code == TDIST_F16 ? c10::ScalarType::Half : c10::ScalarType::BFloat16;
  return true;
}

// ag_gemm(a, b, peer_shards, rank, num_ranks, workspace, status, sk_workspace, stream, row_scale, col_scale) -> c. `stream`: the context's,
// as an address.
PyObject* ag_gemm(PyObject*, PyObject* const* o, Py_ssize_t nargs) {
  TDIST_ARGS(11, 0);
  const at::Tensor *a, *b, *row_scale, *col_scale;
  int code, rank, ranks;
  c10::ScalarType out_type;
  TDIST_ORDINARY(operands_of(o[0], o[1], device, &a, &b, &code, &out_type) && int_of(o[3], &rank) && int_of(o[4], &ranks));
  const void* shards[TDIST_GATHER_MAX_RANKS];
  TDIST_ORDINARY(shards_of(*a, o[2], rank, ranks, device, shards));
  const at::Tensor *workspace = tensor_of(o[5], device), *status = tensor_of(o[6], device, c10::ScalarType::Int, 1);
  const int64_t bytes = a->numel() * a->element_size(), M = a->size(0), K = a->size(1), N = b->size(0);
  TDIST_ORDINARY(workspace && workspace->numel() * workspace->element_size() >= ranks * bytes && bytes % 16 == 0 && M * ranks <= INT_MAX);
  TDIST_ORDINARY(status && status->numel() == 4 && status->is_contiguous());
  void* sk;
  int64_t sk_bytes;
  TDIST_ORDINARY(workspace_of(o[7], device, &sk, &sk_bytes));
  TDIST_ORDINARY(optional_of(o[9], device, c10::ScalarType::Float, &row_scale) && optional_of(o[10], device, c10::ScalarType::Float, &col_scale));
  TDIST_ORDINARY(code == TDIST_F8E4M3 || (!row_scale && !col_scale));
  void* const stream = stream_of(device);
  TDIST_ORDINARY(PyLong_CheckExact(o[8]) && PyLong_AsVoidPtr(o[8]) == stream && !PyErr_Occurred());
  at::Tensor c = empty_on(device, out_type, {M * ranks, N});
  int32_t* const st = (int32_t*)status->data_ptr();
  if (!run([&] {
        return tdist_ag_gemm_rows(code, shards, ranks, (int)M, workspace->data_ptr(), b->data_ptr(), b->stride(0), c.data_ptr(), N, (int)N, (int)K,
                                  (const float*)ptr(row_scale), (const float*)ptr(col_scale), st, st + 2, sk, sk_bytes, stream);
      })) return nullptr;
  return THPVariable_Wrap(std::move(c));
  END_HANDLE_TH_ERRORS
}

// gemm_rs(a, b, rank, num_ranks, own_buffer, buffer_addresses, sk_workspace, row_scale, col_scale) -> own rows of the sum
PyObject* gemm_rs(PyObject*, PyObject* const* o, Py_ssize_t nargs) {
  TDIST_ARGS(9, 0);
  const at::Tensor *a, *b, *row_scale, *col_scale;
  int code, rank, ranks;
  c10::ScalarType out_type;
  TDIST_ORDINARY(operands_of(o[0], o[1], device, &a, &b, &code, &out_type) && int_of(o[2], &rank) && int_of(o[3], &ranks));
  const int64_t M = a->size(0), K = a->size(1), N = b->size(0);
  TDIST_ORDINARY(M % 256 == 0 && N % 256 == 0 && K % 256 == 0 && rank >= 0 && rank < ranks && M % ranks == 0);
  const at::Tensor *own = tensor_of(o[4], device, out_type, 2), *addresses = tensor_of(o[5], device, c10::ScalarType::Long, 1);
  TDIST_ORDINARY(own && own->is_contiguous() && own->size(0) >= M && own->size(1) == N);
  TDIST_ORDINARY(addresses && addresses->is_contiguous() && addresses->numel() == ranks);
  void* sk;
  int64_t sk_bytes;
  TDIST_ORDINARY(workspace_of(o[6], device, &sk, &sk_bytes));
  TDIST_ORDINARY(optional_of(o[7], device, c10::ScalarType::Float, &row_scale) && optional_of(o[8], device, c10::ScalarType::Float, &col_scale));
  TDIST_ORDINARY(code == TDIST_F8E4M3 || (!row_scale && !col_scale));
  void* const stream = stream_of(device);
  at::Tensor out = empty_on(device, out_type, {M / ranks, N});
  if (!run([&] {
        return tdist_gemm_rs(code, a->data_ptr(), K, b->data_ptr(), b->stride(0), (void* const*)addresses->data_ptr(), own->data_ptr(), out.data_ptr(),
                             (int)M, (int)N, (int)K, (const float*)ptr(row_scale), (const float*)ptr(col_scale), rank, ranks, sk, sk_bytes, stream);
      })) return nullptr;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ---- grouped GEMMs of the MoE tensor-parallel layer -----------------------------------------------------------
// A call's sorted routing and the memory that its row blocks are joined into.
struct Blocks {
  const at::Tensor *sorted, *experts, *padded;
  int block_size, entries;
  int64_t at[4];   // addresses: sorted ids, experts, segments, padded total
  int count, rows;
  int tail_most, tail_count;   // experts' last rows in blocks of their own, of TDIST_GROUP_TAIL_BLOCK rows, one array behind the other from tail_ids on
  int32_t *tail_ids, *tail_experts, *tail_segments, *tail_padded;
};
// o[0..4]: sorted ids, experts and padded total of the align / sort, its block size, entries; o[5..13]: a RowBlocks, field by field
bool blocks_of(PyObject* const* o, int device, Blocks& b) {
  b.sorted = tensor_of(o[0], device, c10::ScalarType::Int, 1), b.experts = tensor_of(o[1], device, c10::ScalarType::Int, 1);
  b.padded = tensor_of(o[2], device, c10::ScalarType::Int, 1);
  if (!b.sorted || !b.experts || !b.padded || !b.sorted->is_contiguous() || !b.experts->is_contiguous() || b.padded->numel() < 1) return false;
  if (!int_of(o[3], &b.block_size) || b.block_size <= 0 || !int_of(o[4], &b.entries) || !int_of(o[9], &b.count) || !int_of(o[10], &b.rows)) return false;
  for (int i = 0; i < 4; ++i)
    if (!PyLong_CheckExact(o[5 + i]) || (b.at[i] = PyLong_AsLongLong(o[5 + i])) <= 0) return PyErr_Clear(), false;
  int64_t tail;
  if (!int_of(o[11], &b.tail_most) || !int_of(o[13], &b.tail_count) || b.tail_most < 0 || b.tail_count < 0 || !PyLong_CheckExact(o[12]) ||
      (tail = PyLong_AsLongLong(o[12])) < 0) return PyErr_Clear(), false;
  b.tail_ids = (int32_t*)tail;
  if ((b.tail_most > 0) != (tail != 0 && b.tail_count > 0)) return false;
  b.tail_experts = b.tail_ids + (int64_t)b.tail_count * TDIST_GROUP_TAIL_BLOCK;
  b.tail_segments = b.tail_experts + b.tail_count;
  b.tail_padded = b.tail_segments + b.tail_count;
  return true;
}
// weights [E, K, N] whose rows are contiguous along K, for rows of `k` elements of this type
const at::Tensor* weights_of(PyObject* o, int device, const at::Tensor& a, int64_t rows) {
  const at::Tensor* b = tensor_of(o, device);
  if (!b || b->dim() != 3 || b->scalar_type() != a.scalar_type() || b->size(1) != a.size(1) || b->stride(1) != 1 || b->numel() == 0) return nullptr;
  // (offsets of 32 bits in the forms that take blocks of any size)
  const int64_t e = a.element_size();
  return rows * a.size(1) * e < 1ll << 32 && b->size(2) * b->stride(2) * e < 1ll << 31 ? b : nullptr;
}
int join_and_multiply(const Blocks& k, int code, const void* const* shards, int ranks, int64_t rows, const at::Tensor& a, const at::Tensor& b, void* c, int topk,
                      int32_t* status, void* sk, int64_t sk_bytes, void* stream, bool* joined) {
  const int blocks = (int)std::min(k.experts->numel(), k.sorted->numel() / k.block_size), N = (int)b.size(2);
  int32_t *const ids = (int32_t*)k.at[0], *const experts = (int32_t*)k.at[1], *const segments = (int32_t*)k.at[2], *const padded = (int32_t*)k.at[3];
  const int64_t room = (int64_t)k.count * k.rows;
  int rc = k.tail_most > 0
               ? tdist_moe_join_blocks_tails(i32(k.sorted), i32(k.experts), i32(k.padded), blocks, k.block_size, k.entries, (int)b.size(0), k.rows, ids, room,
                                             experts, segments, padded, k.tail_most, TDIST_GROUP_TAIL_BLOCK, N, k.tail_ids, (int64_t)k.tail_count * TDIST_GROUP_TAIL_BLOCK,
                                             k.tail_experts, k.tail_segments, k.tail_padded, stream)
               : tdist_moe_join_blocks(i32(k.sorted), i32(k.experts), i32(k.padded), blocks, k.block_size, k.entries, (int)b.size(0), k.rows, ids, room,
                                       experts, segments, padded, stream);
  *joined = rc != TDIST_ERR_UNSUPPORTED;   // (nothing has been launched then)
  if (rc != TDIST_OK) return *joined ? rc : TDIST_OK;
  int32_t* const first_error = status ? status + 2 : nullptr;
  if (k.tail_most > 0)
    return tdist_group_gemm_rows_tails(code, shards, ranks, (int)rows, b.data_ptr(), b.stride(2), b.stride(0), c, N, N, (int)a.size(1), ids, experts,
                                       segments, padded, k.count, k.rows, k.entries, topk, k.tail_ids, k.tail_experts, k.tail_segments, k.tail_padded,
                                       k.tail_count, status, first_error, sk, sk_bytes, stream);
  return tdist_group_gemm_rows(code, shards, ranks, (int)rows, b.data_ptr(), b.stride(2), b.stride(0), c, N, N, (int)a.size(1), ids, experts, segments,
                               padded, k.count, k.rows, k.entries, topk, status, first_error, sk, sk_bytes, stream);
}

// ag_group_gemm(a, b, peer_shards, rank, num_ranks, topk, workspace, status, sk_workspace, blocks...) -> c, where the rows can be read where
// they lie
PyObject* ag_group_gemm(PyObject*, PyObject* const* o, Py_ssize_t nargs) {
  TDIST_ARGS(23, 0);
  const at::Tensor* a = tensor_of(o[0], device);
  int code, rank, ranks, topk;
  TDIST_ORDINARY(a && a->dim() == 2 && a->is_contiguous() && a->numel() > 0 && code_of(a->scalar_type(), &code) && int_of(o[3], &rank) &&
                 int_of(o[4], &ranks) && int_of(o[5], &topk) && topk > 0);
  const int64_t M = a->size(0), row_bytes = a->size(1) * a->element_size();
  const void* shards[TDIST_GATHER_MAX_RANKS];
  TDIST_ORDINARY(shards_of(*a, o[2], rank, ranks, device, shards) && M * row_bytes % 16 == 0 && M * ranks <= INT_MAX);
  const at::Tensor *b = weights_of(o[1], device, *a, M * ranks), *workspace = tensor_of(o[6], device), *status = tensor_of(o[7], device, c10::ScalarType::Int, 1);
  TDIST_ORDINARY(b && workspace && workspace->numel() * workspace->element_size() >= ranks * M * row_bytes && status && status->numel() == 4 &&
                 status->is_contiguous());
  TDIST_ORDINARY(tdist_shards_in_reach(shards, ranks, (int)M, M * row_bytes));
  void* sk;
  int64_t sk_bytes;
  Blocks k;
  TDIST_ORDINARY(workspace_of(o[8], device, &sk, &sk_bytes) && blocks_of(o + 9, device, k) && k.entries <= topk * M * ranks);
  void* const stream = stream_of(device);
  at::Tensor c = empty_on(device, code == TDIST_F16 ? c10::ScalarType::Half : c10::ScalarType::BFloat16, {topk * M * ranks, b->size(2)});
  bool joined = true;
  if (!run([&] {
        return join_and_multiply(k, code, shards, ranks, M, *a, *b, c.data_ptr(), topk, i32(status), sk, sk_bytes, stream, &joined);
      })) return nullptr;
  TDIST_ORDINARY(joined);
  return THPVariable_Wrap(std::move(c));
  END_HANDLE_TH_ERRORS
}

// reduce_rs(a, b, rank, world, weights, rows_buffer, rank_buffer, sk_workspace, blocks...) -> this rank's rows of the sum
PyObject* reduce_rs(PyObject*, PyObject* const* o, Py_ssize_t nargs) {
  TDIST_ARGS(22, 0);
  const at::Tensor *a = tensor_of(o[0], device), *weight = tensor_of(o[4], device, c10::ScalarType::Float, 2);
  const at::Tensor *rows = tensor_of(o[5], device, c10::ScalarType::BFloat16, 2), *slab = tensor_of(o[6], device, c10::ScalarType::BFloat16, 2);
  int code, rank, world;
  // (the products of f16 rows are f16, and the buffers hold bf16)
  TDIST_ORDINARY(a && a->dim() == 2 && a->is_contiguous() && a->numel() > 0 && aligned16(*a) && code_of(a->scalar_type(), &code) && code != TDIST_F16 &&
                 int_of(o[2], &rank) && int_of(o[3], &world) && world > 0 && weight && weight->is_contiguous());
  const int64_t M = weight->size(0), topk = weight->size(1), row_bytes = a->size(1) * a->element_size();
  TDIST_ORDINARY(a->size(0) == M * topk && M >= world && row_bytes > 128);
  const at::Tensor* b = weights_of(o[1], device, *a, M * topk);
  TDIST_ORDINARY(b && rows && slab && rows->is_contiguous() && slab->is_contiguous() && rows->size(1) == b->size(2) && slab->size(1) == b->size(2) &&
                 rows->size(0) >= M * topk && slab->size(0) >= M);
  void* sk;
  int64_t sk_bytes;
  Blocks k;
  TDIST_ORDINARY(workspace_of(o[7], device, &sk, &sk_bytes) && blocks_of(o + 8, device, k) && k.entries <= M * topk);
  void* const stream = stream_of(device);
  const int64_t m_per = M / world, hidden = b->size(2);
  const at::Tensor sums = empty_on(device, c10::ScalarType::BFloat16, {M, hidden});
  at::Tensor out = empty_on(device, c10::ScalarType::BFloat16, {m_per, hidden});
  const void* const all[1] = {a->data_ptr()};
  bool joined = true;
  if (!run([&] {
        const int rc = join_and_multiply(k, code, all, 1, a->size(0), *a, *b, rows->data_ptr(), 1, nullptr, sk, sk_bytes, stream, &joined);
        if (rc != TDIST_OK || !joined) return rc;
        return tdist_moe_combine_reduce(rows->data_ptr(), (const float*)weight->data_ptr(), m_per * world, (int)topk, (int)hidden, rank, world,
                                        slab->data_ptr(), sums.data_ptr(), out.data_ptr(), stream);
      })) return nullptr;
  TDIST_ORDINARY(joined);
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// ---- MoE dispatch / combine ----------------------------------------------------------------------------------
// The attributes of an AllToAllContext that are read or written here.
enum Attr { kCallCount, kModValue, kIndexCalls, kIndexKey, kIndexSets, kIndexWorkspace, kLastIndex, kHalves, kSplitBuf, kRecvBuf, kScaleBuf, kDtype,
            kHidden, kEleSize, kMaxM, kWorld, kPerRank, kExperts, kGroupSize, kNumAttrs };
constexpr const char* kAttrNames[kNumAttrs] = {"call_count", "MOD_VALUE", "index_calls", "index_key", "index_sets", "index_workspace", "last_index",
                                               "halves", "split_recv_buf", "recv_buf", "scale_recv_buf", "dtype", "hidden", "ele_size", "max_m",
                                               "WORLD_SIZE", "experts_per_rank", "num_tot_experts", "fp8_group_size"};
PyObject* g_attr[kNumAttrs];

// A reference that is given back.
struct Ref {
  PyObject* o;
  explicit Ref(PyObject* o) : o(o) {}
  Ref(const Ref&) = delete;
  ~Ref() { Py_XDECREF(o); }
  operator PyObject*() const { return o; }
};
PyObject* get(PyObject* ctx, Attr a) {
  PyObject* o = PyObject_GetAttr(ctx, g_attr[a]);
  if (!o) PyErr_Clear();
  return o;
}
bool get_int(PyObject* ctx, Attr a, int* v) {
  const Ref o(get(ctx, a));
  return o.o && int_of(o, v);
}
bool set_int(PyObject* ctx, Attr a, int v) {
  const Ref o(PyLong_FromLong(v));
  return o.o && PyObject_SetAttr(ctx, g_attr[a], o) == 0;
}
bool int_is(PyObject* o, uintptr_t v) {
  const bool same = PyLong_CheckExact(o) && PyLong_AsSize_t(o) == v;
  if (PyErr_Occurred()) return PyErr_Clear(), false;
  return same;
}

// Places in AllToAllContext.halves: the halves, the buffers, their addresses, rows of a half and experts.
enum Half { kHalfBufs = 2, kHalfAddresses = 5, kHalfRows = 8, kHalfExperts = 9, kHalfFields = 10 };
struct Slots {
  int hidden, ele, max_m, world, per_rank, experts, calls, mod;
  c10::ScalarType type;
  at::Tensor splits, recv, scales;   // the next call's half of the receive buffers: see AllToAllContext.next_half
};
bool slots_of(PyObject* ctx, int device, Slots& s) {
  if (!get_int(ctx, kHidden, &s.hidden) || !get_int(ctx, kEleSize, &s.ele) || !get_int(ctx, kMaxM, &s.max_m) || !get_int(ctx, kWorld, &s.world) ||
      !get_int(ctx, kPerRank, &s.per_rank) || !get_int(ctx, kExperts, &s.experts) || !get_int(ctx, kCallCount, &s.calls) ||
      !get_int(ctx, kModValue, &s.mod) || s.mod <= 0 || s.calls < 0) return false;
  const Ref dtype(get(ctx, kDtype)), halves(get(ctx, kHalves));
  if (!dtype.o || !THPDtype_Check(dtype) || !halves.o || !PyTuple_CheckExact(halves) || PyTuple_GET_SIZE(halves.o) != kHalfFields) return false;
  s.type = ((THPDtype*)dtype.o)->scalar_type;
  const Attr bufs[3] = {kSplitBuf, kRecvBuf, kScaleBuf};
  for (int i = 0; i < 3; ++i) {
    const Ref buf(get(ctx, bufs[i]));
    if (!buf.o || buf != PyTuple_GET_ITEM(halves.o, kHalfBufs + i)) return false;
    const at::Tensor* t = tensor_of(buf, device);
    if (!t || !int_is(PyTuple_GET_ITEM(halves.o, kHalfAddresses + i), (uintptr_t)t->data_ptr())) return false;
  }
  if (!int_is(PyTuple_GET_ITEM(halves.o, kHalfRows), (uintptr_t)s.world * s.max_m) || !int_is(PyTuple_GET_ITEM(halves.o, kHalfExperts), s.experts)) return false;
  PyObject* const half = PyTuple_GET_ITEM(halves.o, s.calls % 2);
  if (!PyTuple_CheckExact(half) || PyTuple_GET_SIZE(half) != 3) return false;
  at::Tensor* const out[3] = {&s.splits, &s.recv, &s.scales};
  for (int i = 0; i < 3; ++i) {
    const at::Tensor* t = tensor_of(PyTuple_GET_ITEM(half, i), device);
    if (!t) return false;
    *out[i] = t->detach();
  }
  return true;
}

struct IndexSet {
  PyObject* set;   // borrowed from the context's list
  int calls;
  const at::Tensor* t[5];
};
// The set of index tensors whose turn it is, where the context has seen this shape.
bool index_set_of(PyObject* ctx, int device, int64_t T, int64_t topk, int64_t experts, IndexSet& s) {
  const Ref key(get(ctx, kIndexKey)), sets(get(ctx, kIndexSets));
  if (!key.o || !sets.o || !PyTuple_CheckExact(key) || PyTuple_GET_SIZE(key.o) != 4 || !PyList_CheckExact(sets) || PyList_GET_SIZE(sets.o) != 2) return false;
  if (!int_is(PyTuple_GET_ITEM(key.o, 0), T) || !int_is(PyTuple_GET_ITEM(key.o, 1), topk) || !int_is(PyTuple_GET_ITEM(key.o, 2), experts)) return false;
  PyObject* const dev = PyTuple_GET_ITEM(key.o, 3);
  if (!THPDevice_Check(dev) || ((THPDevice*)dev)->device != c10::Device(c10::kCUDA, (c10::DeviceIndex)device)) return false;
  if (!get_int(ctx, kIndexCalls, &s.calls) || s.calls < 0) return false;
  s.set = PyList_GET_ITEM(sets.o, s.calls % 2);   // (the context holds the list)
  if (!PyTuple_CheckExact(s.set) || PyTuple_GET_SIZE(s.set) != 5) return false;
  for (int i = 0; i < 5; ++i)
    if (!(s.t[i] = tensor_of(PyTuple_GET_ITEM(s.set, i), device)) || s.t[i]->scalar_type() != c10::ScalarType::Int) return false;
  return true;
}
// contiguous ids [T, topk] of 32 or 64 bits
const at::Tensor* ids_of(PyObject* o, int device) {
  const at::Tensor* t = tensor_of(o, device);
  return t && t->dim() == 2 && t->is_contiguous() && t->numel() > 0 &&
                 (t->scalar_type() == c10::ScalarType::Int || t->scalar_type() == c10::ScalarType::Long) ? t : nullptr;
}
PyObject* three(at::Tensor splits, at::Tensor recv, at::Tensor scales, bool with_scales) {
  Ref a(THPVariable_Wrap(std::move(splits))), b(THPVariable_Wrap(std::move(recv)));
  Ref c(with_scales ? THPVariable_Wrap(std::move(scales)) : Py_NewRef(Py_None));
  PyObject* list = a.o && b.o && c.o ? PyList_New(3) : nullptr;
  if (!list) return nullptr;
  PyList_SET_ITEM(list, 0, std::exchange(a.o, nullptr));
  PyList_SET_ITEM(list, 1, std::exchange(b.o, nullptr));
  PyList_SET_ITEM(list, 2, std::exchange(c.o, nullptr));
  return list;
}

// preprocess(ctx, ids, num_experts) -> (splits, cumsum, scatter, gather)
PyObject* preprocess(PyObject*, PyObject* const* o, Py_ssize_t nargs) {
  TDIST_ARGS(3, 1);
  int experts;
  const at::Tensor* ids = ids_of(o[1], device);
  TDIST_ORDINARY(ids && int_of(o[2], &experts));
  IndexSet s;
  TDIST_ORDINARY(index_set_of(o[0], device, ids->size(0), ids->size(1), experts, s));
  const Ref workspace(get(o[0], kIndexWorkspace));
  void* ws;
  int64_t ws_bytes;
  TDIST_ORDINARY(workspace.o && workspace_of(workspace, device, &ws, &ws_bytes) && ws);
  const Ref out(PyTuple_GetSlice(s.set, 0, 4));
  if (!out.o) return nullptr;
  void* const stream = stream_of(device);
  bool unsupported = false;
  if (!run([&] {
        const int64_t n = ids->numel();
        const int topk = (int)ids->size(1);
        if (ids->scalar_type() == c10::ScalarType::Int)
          return tdist_moe_scatter_index(i32(ids), n, topk, experts, i32(s.t[0]), i32(s.t[1]), i32(s.t[2]), i32(s.t[3]), nullptr, ws, ws_bytes, stream);
        const int rc = tdist_moe_scatter_index64((const int64_t*)ids->data_ptr(), n, topk, experts, i32(s.t[0]), i32(s.t[1]), i32(s.t[2]), i32(s.t[3]),
                                                 nullptr, ws, ws_bytes, stream);
        unsupported = rc == TDIST_ERR_UNSUPPORTED;   // (ids of this many are converted first)
        return unsupported ? TDIST_OK : rc;
      })) return nullptr;
  TDIST_ORDINARY(!unsupported);
  if (!set_int(o[0], kIndexCalls, s.calls + 1)) return nullptr;
  return Py_NewRef(out.o);
  END_HANDLE_TH_ERRORS
}

// dispatch_ids(ctx, tokens, token_scales, expert_ids) -> [splits, recv, scales or None]
PyObject* dispatch_ids(PyObject*, PyObject* const* o, Py_ssize_t nargs) {
  TDIST_ARGS(4, 1);
  PyObject* const ctx = o[0];
  const at::Tensor *x = tensor_of(o[1], device), *scale, *ids = ids_of(o[3], device);
  int group;
  TDIST_ORDINARY(x && x->dim() == 2 && x->is_contiguous() && ids && ids->size(0) == x->size(0) && get_int(ctx, kGroupSize, &group) && group == 0);
  TDIST_ORDINARY(optional_of(o[2], device, c10::ScalarType::Float, &scale));
  Slots s;
  TDIST_ORDINARY(slots_of(ctx, device, s) && x->size(1) == s.hidden && x->scalar_type() == s.type);
  const int64_t T = ids->size(0), topk = ids->size(1), row_bytes = (int64_t)s.hidden * s.ele;
  TDIST_ORDINARY(tdist_moe_dispatch_from_ids_takes(T, (int)topk, row_bytes, s.experts));
  IndexSet set;
  TDIST_ORDINARY(index_set_of(ctx, device, T, topk, s.experts, set));
  const Ref last(PyTuple_GetSlice(set.set, 0, 4));
  if (!last.o || !set_int(ctx, kIndexCalls, set.calls + 1)) return nullptr;
  void* const stream = stream_of(device);
  if (!run([&] {
        auto call = [&](auto entry, auto* p) {
          return entry(x->data_ptr(), row_bytes, (const float*)ptr(scale), p, (int)topk, T, s.world, s.per_rank, s.max_m, s.recv.data_ptr(),
                       scale ? (float*)s.scales.data_ptr() : nullptr, i32(&s.splits), i32(set.t[0]), i32(set.t[1]), i32(set.t[2]), i32(set.t[3]), stream);
        };
        return ids->scalar_type() == c10::ScalarType::Int ? call(tdist_moe_dispatch_tokens_from_ids, (const int32_t*)ids->data_ptr())
                                                          : call(tdist_moe_dispatch_tokens_from_ids64, (const int64_t*)ids->data_ptr());
      })) return nullptr;
  if (PyObject_SetAttr(ctx, g_attr[kLastIndex], last) != 0 || !set_int(ctx, kCallCount, (s.calls + 1) % s.mod)) return nullptr;
  return three(std::move(s.splits), std::move(s.recv), std::move(s.scales), scale != nullptr);
  END_HANDLE_TH_ERRORS
}

// dispatch_quant(ctx, tokens, cumsum, scatter_index) -> [splits, recv, scales]
PyObject* dispatch_quant(PyObject*, PyObject* const* o, Py_ssize_t nargs) {
  TDIST_ARGS(4, 1);
  PyObject* const ctx = o[0];
  const at::Tensor *x = tensor_of(o[1], device, c10::ScalarType::BFloat16, 2), *cumsum = tensor_of(o[2], device, c10::ScalarType::Int, 1);
  const at::Tensor* scatter = tensor_of(o[3], device, c10::ScalarType::Int, 2);
  int group;
  TDIST_ORDINARY(x && x->is_contiguous() && cumsum && cumsum->is_contiguous() && scatter && scatter->is_contiguous() && scatter->size(0) == x->size(0));
  Slots s;
  TDIST_ORDINARY(get_int(ctx, kGroupSize, &group) && group > 0 && slots_of(ctx, device, s) && s.type == c10::ScalarType::Float8_e4m3fn &&
                 x->size(1) == s.hidden && cumsum->numel() == (int64_t)s.experts + 1);
  void* const stream = stream_of(device);
  if (!run([&] {
        return tdist_moe_dispatch_tokens_quant(x->data_ptr(), s.hidden, group, i32(scatter), (int)scatter->size(1), i32(cumsum), x->size(0), s.world,
                                               s.per_rank, s.max_m, s.recv.data_ptr(), (float*)s.scales.data_ptr(), i32(&s.splits), stream);
      })) return nullptr;
  if (!set_int(ctx, kCallCount, (s.calls + 1) % s.mod)) return nullptr;
  return three(std::move(s.splits), std::move(s.recv), std::move(s.scales), true);
  END_HANDLE_TH_ERRORS
}

// combine(ctx, rows, row_scale, scatter_index, weights, cumsum) -> y, from the slots of the context
PyObject* combine(PyObject*, PyObject* const* o, Py_ssize_t nargs) {
  TDIST_ARGS(6, 1);
  const at::Tensor *rows = tensor_of(o[1], device), *scale, *scatter = tensor_of(o[3], device, c10::ScalarType::Int, 2), *weight;
  const at::Tensor* cumsum = tensor_of(o[5], device, c10::ScalarType::Int, 1);
  TDIST_ORDINARY(rows && rows->dim() == 2 && rows->is_contiguous() && rows->size(1) > 0 && scatter && scatter->is_contiguous() && cumsum && cumsum->is_contiguous());
  TDIST_ORDINARY(rows->scalar_type() == c10::ScalarType::Float8_e4m3fn || rows->scalar_type() == c10::ScalarType::BFloat16);
  TDIST_ORDINARY(optional_of(o[2], device, c10::ScalarType::Float, &scale) && optional_of(o[4], device, c10::ScalarType::Float, &weight));
  TDIST_ORDINARY(!weight || weight->sizes() == scatter->sizes());
  int world, per_rank, max_m, group = 0;
  TDIST_ORDINARY(get_int(o[0], kWorld, &world) && get_int(o[0], kPerRank, &per_rank) && get_int(o[0], kMaxM, &max_m));
  const int64_t T = scatter->size(0), hidden = rows->size(1);
  if (scale && scale->dim() == 2) {
    TDIST_ORDINARY(scale->size(1) > 0 && hidden % scale->size(1) == 0);
    group = (int)(hidden / scale->size(1));
  }
  void* const stream = stream_of(device);
  at::Tensor out = empty_on(device, c10::ScalarType::BFloat16, {T, hidden});
  if (!run([&] {
        return tdist_moe_combine(rows->data_ptr(), rows->scalar_type() == c10::ScalarType::BFloat16 ? TDIST_BF16 : TDIST_F8E4M3, (const float*)ptr(scale),
                                 i32(scatter), (const float*)ptr(weight), i32(cumsum), T, (int)scatter->size(1), (int)hidden, world, per_rank, max_m,
                                 group, out.data_ptr(), stream);
      })) return nullptr;
  return THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// align(ids, num_experts, num_ranks, block_size, starts, sizes, total, workspace, workspace_bytes) -> the five results, views of one tensor
// of `total` elements
PyObject* align(PyObject*, PyObject* const* o, Py_ssize_t nargs) {
  TDIST_ARGS(9, 0);
  const at::Tensor* ids = ids_of(o[0], device);
  int experts, ranks, block, total, bytes, starts[5], sizes[5];
  TDIST_ORDINARY(ids && int_of(o[1], &experts) && int_of(o[2], &ranks) && int_of(o[3], &block) && int_of(o[6], &total) && int_of(o[8], &bytes));
  TDIST_ORDINARY(ranks > 0 && ids->numel() % ranks == 0);
  for (int i = 0; i < 5; ++i)
    TDIST_ORDINARY(PyTuple_CheckExact(o[4]) && PyTuple_GET_SIZE(o[4]) == 5 && PyTuple_CheckExact(o[5]) && PyTuple_GET_SIZE(o[5]) == 5 &&
                   int_of(PyTuple_GET_ITEM(o[4], i), &starts[i]) && int_of(PyTuple_GET_ITEM(o[5], i), &sizes[i]));
  void* ws;
  int64_t ws_bytes;
  TDIST_ORDINARY(workspace_of(o[7], device, &ws, &ws_bytes) && ws && ws_bytes >= bytes);
  void* const stream = stream_of(device);
  const at::Tensor flat = empty_on(device, c10::ScalarType::Int, {total});
  int32_t* const at = i32(&flat);
  if (!run([&] {
        return tdist_moe_align_block_size(ids->data_ptr(), ids->scalar_type() == c10::ScalarType::Long, ids->numel(), experts, ranks, ids->numel() / ranks,
                                          block, at + starts[0], sizes[0], at + starts[1], at + starts[2], at + starts[3], at + starts[4], ws, bytes,
                                          stream);
      })) return nullptr;
  Ref out(PyTuple_New(5));
  if (!out.o) return nullptr;
  for (int i = 0; i < 5; ++i) {
    PyObject* t = THPVariable_Wrap(flat.narrow(0, starts[i], sizes[i]));
    if (!t) return nullptr;
    PyTuple_SET_ITEM(out.o, i, t);
  }
  return std::exchange(out.o, nullptr);
  END_HANDLE_TH_ERRORS
}

// set_error(class): what a call that fails raises, TdistError(code, message)
PyObject* set_error(PyObject*, PyObject* cls) {
  Py_INCREF(cls);
  Py_XDECREF(std::exchange(g_error, cls));
  Py_RETURN_NONE;
}

#define TDIST_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {TDIST_METHOD(decode), TDIST_METHOD(decode_ranks), TDIST_METHOD(ag_gemm), TDIST_METHOD(gemm_rs), TDIST_METHOD(ag_group_gemm),
                          TDIST_METHOD(reduce_rs), TDIST_METHOD(preprocess),
                          TDIST_METHOD(dispatch_ids), TDIST_METHOD(dispatch_quant), TDIST_METHOD(combine), TDIST_METHOD(align),
                          {"set_error", set_error, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "tdist_torch", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_tdist_torch() {
  for (int i = 0; i < kNumAttrs; ++i)
    if (!(g_attr[i] = PyUnicode_InternFromString(kAttrNames[i]))) return nullptr;
  PyObject* const m = PyModule_Create(&kModule);
  if (m && PyModule_AddStringConstant(m, "torch_version", TDIST_TORCH_VERSION) != 0) return Py_DECREF(m), nullptr;
  return m;
}
