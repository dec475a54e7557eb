// The hot operators as a CPython module: tensor checks, output allocation and the C ABI's call in one step.
//
// A decode linear takes 6 us on the GPU; the Python wrappers (argument checks one by one, three to four torch.empty, two
// ctypes calls of some twenty arguments) took 26 us of host time around it.  Each function here handles the common case of
// one wrapper and returns None for every other -- another dtype, layout, device, an empty tensor -- so that the wrapper's
// own checks and messages decide those.  Nothing is kept between calls but the Python function found at import.
#include <Python.h>

#include <ATen/ATen.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/maxfp8.h"

namespace {

PyObject* g_raw_stream = nullptr;  // torch._C._cuda_getCurrentRawStream

bool stream_of(const at::Tensor& t, void** stream) {
  PyObject* index = PyLong_FromLong(t.device().index());
  if (!index) return false;
  PyObject* handle = PyObject_CallOneArg(g_raw_stream, index);
  Py_DECREF(index);
  if (!handle) return false;
  *stream = PyLong_AsVoidPtr(handle);
  Py_DECREF(handle);
  return !PyErr_Occurred();
}

// the exception class the Python wrappers raise for a status of the C ABI
PyObject* raise(int status) {
  PyObject* kind = status == MAXFP8_ERR_DTYPE ? PyExc_TypeError : status == MAXFP8_ERR_LAUNCH ? PyExc_RuntimeError : PyExc_ValueError;
  PyErr_SetString(kind, maxfp8_last_error());
  return nullptr;
}

const at::Tensor* tensor(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }
bool on_gpu(const at::Tensor& t, const at::Tensor& like) { return t.is_cuda() && t.device() == like.device(); }
bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
int64_t row_stride(const at::Tensor& t) { return t.size(0) > 1 ? t.stride(0) : t.size(1); }
// bf16 rows a kernel can read 16 bytes at a time
bool bf16_rows(const at::Tensor& t) {
  return t.is_cuda() && t.scalar_type() == at::kBFloat16 && t.dim() == 2 && t.size(0) > 0 && t.size(1) > 0 && t.stride(1) == 1 &&
         row_stride(t) >= t.size(1) && row_stride(t) % 8 == 0 && aligned16(t.data_ptr());
}
bool fp8_rows(const at::Tensor& t) {
  return t.is_cuda() && t.scalar_type() == at::kFloat8_e4m3fn && t.dim() == 2 && t.size(0) > 0 && t.size(1) > 0 && t.stride(1) == 1 &&
         row_stride(t) >= t.size(1) && row_stride(t) % 16 == 0 && aligned16(t.data_ptr());
}
// weight scales of w in the granularity's layout: [ceil(N/128), K/128] with contiguous rows, or a contiguous [N, 1]
bool weight_scales_ok(const at::Tensor& s, const at::Tensor& w, int granularity) {
  if (!on_gpu(s, w) || s.scalar_type() != at::kFloat || s.dim() != 2) return false;
  const int64_t N = w.size(0), K = w.size(1);
  if (granularity == MAXFP8_GRAN_BLOCK) return K % 128 == 0 && s.size(0) == (N + 127) / 128 && s.size(1) == K / 128 && s.is_contiguous();
  return s.size(0) == N && s.size(1) == 1 && s.is_contiguous() && K % 16 == 0;
}
at::Tensor bytes_on(const at::Tensor& like, size_t n) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte)); }

// An operator's allocations and launches without the interpreter lock, as torch's own calls and ctypes make them: an allocation
// may reach the driver, a launch waits where the queue is full, and other threads go on meanwhile.  (The lock is back before an
// exception of the call leaves.)
struct Unlocked {
  PyThreadState* state = PyEval_SaveThread();
  ~Unlocked() { PyEval_RestoreThread(state); }
};
template <class Call>
int unlocked(Call call) {
  const Unlocked released;
  return call();
}

// y = quantise(x) . w^T: [M, N] bf16; a status of the C ABI.  (Without the lock, like what the operators below do inside `unlocked`.)
int linear_of(at::Tensor& y, const at::Tensor& x, const at::Tensor& w, const at::Tensor& s, int granularity, float scale_ub, void* stream) {
  const int64_t M = x.size(0), K = x.size(1), N = w.size(0);
  y = at::empty({M, N}, x.options());
  const size_t need = maxfp8_linear_workspace_bytes(M, N, K, granularity);
  at::Tensor ws;
  if (need) ws = bytes_on(x, need);
  return maxfp8_linear_dynamic_scaled_fp8(y.data_ptr(), x.data_ptr(), w.data_ptr(), s.data_ptr(), M, N, K, row_stride(x), row_stride(w), N,
      granularity, s.size(1), scale_ub, need ? ws.data_ptr() : nullptr, need, stream);
}
bool linear_ok(const at::Tensor& x, const at::Tensor& w, const at::Tensor& s, int granularity) {
  return bf16_rows(x) && fp8_rows(w) && on_gpu(w, x) && w.size(1) == x.size(1) && weight_scales_ok(s, w, granularity);
}

#define NEED_ARGS(n)                                                                        \
  if (nargs != (n)) {                                                                       \
    PyErr_Format(PyExc_TypeError, "%s takes %d arguments, got %zd", __func__, (n), nargs);  \
    return nullptr;                                                                         \
  }
// a C++ exception (a tensor without memory of its own is asked for its pointer, an allocation fails) becomes Python's RuntimeError
using Function = PyObject*(PyObject*, PyObject* const*, Py_ssize_t);
template <Function* F>
PyObject* guarded(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
  try {
    return F(self, args, nargs);
  } catch (const std::exception& e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}

// linear(x, w, w_scales, granularity, scale_ub) -> y
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  NEED_ARGS(5)
  const at::Tensor *x = tensor(args[0]), *w = tensor(args[1]), *s = tensor(args[2]);
  const int granularity = (int)PyLong_AsLong(args[3]);
  const float ub = (float)PyFloat_AsDouble(args[4]);
  if (PyErr_Occurred()) return nullptr;
  if (!x || !w || !s || !linear_ok(*x, *w, *s, granularity)) Py_RETURN_NONE;
  void* stream;
  if (!stream_of(*x, &stream)) return nullptr;
  at::Tensor y;
  const int status = unlocked([&] { return linear_of(y, *x, *w, *s, granularity, ub, stream); });
  if (status != MAXFP8_OK) return raise(status);
  return THPVariable_Wrap(std::move(y));
}

// linear_static(x, w, input_scale, weight_scale) -> y; the scales are tensors of one float on the CPU
PyObject* linear_static(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  NEED_ARGS(4)
  const at::Tensor *x = tensor(args[0]), *w = tensor(args[1]), *si = tensor(args[2]), *sw = tensor(args[3]);
  // (a tensor on the meta device, or one that only has a shape while a program is traced, has no value to read)
  auto scalar = [](const at::Tensor* t) -> const float* {
    const bool ok = t && t->device().is_cpu() && t->scalar_type() == at::kFloat && t->numel() == 1 && t->dim() <= 1;
    return ok ? static_cast<const float*>(t->data_ptr()) : nullptr;
  };
  const float *pi = scalar(si), *pw = scalar(sw);
  if (!x || !w || !pi || !pw || !bf16_rows(*x) || !fp8_rows(*w) || !on_gpu(*w, *x) || w->size(1) != x->size(1) || x->size(1) % 16 != 0)
    Py_RETURN_NONE;
  void* stream;
  if (!stream_of(*x, &stream)) return nullptr;
  const float input_scale = *pi, weight_scale = *pw;
  const int64_t M = x->size(0), K = x->size(1), N = w->size(0);
  at::Tensor y;
  const int status = unlocked([&] {
    y = at::empty({M, N}, x->options());
    const size_t need = maxfp8_linear_workspace_bytes(M, N, K, MAXFP8_GRAN_TENSOR);
    at::Tensor ws;
    if (need) ws = bytes_on(*x, need);
    return maxfp8_linear_static_scaled_fp8(y.data_ptr(), x->data_ptr(), w->data_ptr(), M, N, K, row_stride(*x), row_stride(*w), N,
        input_scale, weight_scale, need ? ws.data_ptr() : nullptr, need, stream);
  });
  if (status != MAXFP8_OK) return raise(status);
  return THPVariable_Wrap(std::move(y));
}

PyObject* pair(at::Tensor a, at::Tensor b) {
  PyObject* first = THPVariable_Wrap(std::move(a));
  PyObject* second = first ? THPVariable_Wrap(std::move(b)) : nullptr;
  PyObject* out = second ? PyTuple_Pack(2, first, second) : nullptr;
  Py_XDECREF(first);
  Py_XDECREF(second);
  return out;
}

// quantize(x, group or -1 for a whole row, whether the scales' rows are padded to 16 bytes, scale_ub) -> (q, scales); float32 scales
PyObject* quantize(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  NEED_ARGS(4)
  const at::Tensor* x = tensor(args[0]);
  int64_t group = PyLong_AsLongLong(args[1]);
  const bool padded = PyLong_AsLong(args[2]) != 0;
  const float ub = (float)PyFloat_AsDouble(args[3]);
  if (PyErr_Occurred()) return nullptr;
  if (!x || !bf16_rows(*x)) Py_RETURN_NONE;
  if (group == -1) group = x->size(1);
  if (group <= 0 || x->size(1) % group != 0) Py_RETURN_NONE;
  void* stream;
  if (!stream_of(*x, &stream)) return nullptr;
  const int64_t M = x->size(0), K = x->size(1), ld = padded ? (M + 3) / 4 * 4 : M;
  at::Tensor q, s;
  const int status = unlocked([&] {
    q = at::empty({M, K}, x->options().dtype(at::kFloat8_e4m3fn));
    s = at::empty({K / group, ld}, x->options().dtype(at::kFloat));
    return maxfp8_quantize_dynamic_scaled_fp8(q.data_ptr(), s.data_ptr(), x->data_ptr(), M, K, row_stride(*x), K, group, ld, MAXFP8_BF16,
        MAXFP8_F32, ub, stream);
  });
  if (status != MAXFP8_OK) return raise(status);
  return pair(std::move(q), std::move(s));
}

// rms_norm_quantize(x, gamma, epsilon, weight_offset, scale_ub) -> (q, scales [1, rows])
PyObject* rms_norm_quantize(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  NEED_ARGS(5)
  const at::Tensor *x = tensor(args[0]), *g = tensor(args[1]);
  const float eps = (float)PyFloat_AsDouble(args[2]), offset = (float)PyFloat_AsDouble(args[3]), ub = (float)PyFloat_AsDouble(args[4]);
  if (PyErr_Occurred()) return nullptr;
  if (!x || !g || !bf16_rows(*x) || !on_gpu(*g, *x) || g->scalar_type() != at::kBFloat16 || g->dim() != 1 || g->size(0) != x->size(1) || !g->is_contiguous())
    Py_RETURN_NONE;
  void* stream;
  if (!stream_of(*x, &stream)) return nullptr;
  const int64_t M = x->size(0), K = x->size(1);
  at::Tensor q, s;
  const int status = unlocked([&] {
    q = at::empty({M, K}, x->options().dtype(at::kFloat8_e4m3fn));
    s = at::empty({1, M}, x->options().dtype(at::kFloat));
    return maxfp8_rms_norm_fused_quantize_dynamic_scaled_fp8(q.data_ptr(), s.data_ptr(), x->data_ptr(), g->data_ptr(), M, K, row_stride(*x),
        K, MAXFP8_BF16, MAXFP8_F32, eps, offset, ub, stream);
  });
  if (status != MAXFP8_OK) return raise(status);
  return pair(std::move(q), std::move(s));
}

// matmul(a, b, a_scales, b_scales, granularity of b) -> c [M, N] bf16; float32 block or per-token x per-channel scales
PyObject* matmul(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  NEED_ARGS(5)
  const at::Tensor *a = tensor(args[0]), *b = tensor(args[1]), *sa = tensor(args[2]), *sb = tensor(args[3]);
  const int granularity = (int)PyLong_AsLong(args[4]);
  if (PyErr_Occurred()) return nullptr;
  if (!a || !b || !sa || !sb || !fp8_rows(*a) || !fp8_rows(*b) || !on_gpu(*b, *a) || a->size(1) != b->size(1) || !weight_scales_ok(*sb, *b, granularity) ||
      !on_gpu(*sa, *a) || sa->scalar_type() != at::kFloat || sa->dim() != 2 || sa->stride(1) != 1 || sa->size(1) < a->size(0) ||
      row_stride(*sa) < sa->size(1))
    Py_RETURN_NONE;
  const bool block = granularity == MAXFP8_GRAN_BLOCK;
  if (sa->size(0) != (block ? a->size(1) / 128 : 1)) Py_RETURN_NONE;
  void* stream;
  if (!stream_of(*a, &stream)) return nullptr;
  const int64_t M = a->size(0), K = a->size(1), N = b->size(0);
  at::Tensor c;
  const int status = unlocked([&] {
    c = at::empty({M, N}, a->options().dtype(at::kBFloat16));
    const size_t need = maxfp8_matmul_auto_workspace_bytes(M, N, K);
    at::Tensor ws;
    if (need) ws = bytes_on(*a, need);
    return maxfp8_matmul_dynamic_scaled_fp8(
        c.data_ptr(), a->data_ptr(), b->data_ptr(), sa->data_ptr(), sb->data_ptr(), M, N, K, row_stride(*a), row_stride(*b), N,
        block ? MAXFP8_GRAN_BLOCK : MAXFP8_GRAN_COLWISE, granularity, block ? 1 : -1, block ? 128 : -1, block ? 128 : -1, row_stride(*sa), sb->size(1),
        MAXFP8_BF16, MAXFP8_F32, MAXFP8_ALGO_AUTO, need ? ws.data_ptr() : nullptr, need, stream);
  });
  if (status != MAXFP8_OK) return raise(status);
  return THPVariable_Wrap(std::move(c));
}

// batched_quantize(x [B, M, K] with contiguous channels, group, scale_ub) -> (q [B, M, K], scales [B, K / group, M_pad])
PyObject* batched_quantize(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  NEED_ARGS(3)
  const at::Tensor* x = tensor(args[0]);
  const int64_t group = PyLong_AsLongLong(args[1]);
  const float ub = (float)PyFloat_AsDouble(args[2]);
  if (PyErr_Occurred()) return nullptr;
  if (!x || !x->is_cuda() || x->scalar_type() != at::kBFloat16 || x->dim() != 3 || x->numel() == 0 || x->stride(2) != 1 || group <= 0 ||
      x->size(2) % group != 0)
    Py_RETURN_NONE;
  void* stream;
  if (!stream_of(*x, &stream)) return nullptr;
  const int64_t B = x->size(0), M = x->size(1), K = x->size(2), ld = (M + 3) / 4 * 4;
  at::Tensor q, s;
  const int status = unlocked([&] {
    q = at::empty({B, M, K}, x->options().dtype(at::kFloat8_e4m3fn));
    s = at::empty({B, K / group, ld}, x->options().dtype(at::kFloat));
    return maxfp8_batched_quantize_dynamic_scaled_fp8(
        q.data_ptr(), s.data_ptr(), x->data_ptr(), B, M, K, B > 1 ? x->stride(0) : M * K, M > 1 ? x->stride(1) : K, M * K, K, group, (K / group) * ld, ld,
        MAXFP8_BF16, MAXFP8_F32, ub, stream);
  });
  if (status != MAXFP8_OK) return raise(status);
  return pair(std::move(q), std::move(s));
}

// batched_matmul(a, b, a_scales, b_scales) -> c [B, M, N] bf16; contiguous operands, block scaling
PyObject* batched_matmul(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  NEED_ARGS(4)
  const at::Tensor *a = tensor(args[0]), *b = tensor(args[1]), *sa = tensor(args[2]), *sb = tensor(args[3]);
  auto ok = [](const at::Tensor* t, at::ScalarType kind) { return t && t->is_cuda() && t->scalar_type() == kind && t->dim() == 3 && t->is_contiguous() && t->numel() > 0; };
  if (!ok(a, at::kFloat8_e4m3fn) || !ok(b, at::kFloat8_e4m3fn) || !ok(sa, at::kFloat) || !ok(sb, at::kFloat)) Py_RETURN_NONE;
  const int64_t B = a->size(0), M = a->size(1), K = a->size(2), N = b->size(1), kb = (K + 127) / 128, nb = (N + 127) / 128;
  if (!on_gpu(*b, *a) || !on_gpu(*sa, *a) || !on_gpu(*sb, *a) || b->size(0) != B || b->size(2) != K || sa->size(0) != B || sa->size(1) != kb ||
      sa->size(2) < M || sb->size(0) != B || sb->size(1) != nb || sb->size(2) != kb)
    Py_RETURN_NONE;
  void* stream;
  if (!stream_of(*a, &stream)) return nullptr;
  const int64_t ld = sa->size(2);
  at::Tensor c;
  const int status = unlocked([&] {
    c = at::empty({B, M, N}, a->options().dtype(at::kBFloat16));
    return maxfp8_batched_matmul_dynamic_scaled_fp8(
        c.data_ptr(), a->data_ptr(), b->data_ptr(), sa->data_ptr(), sb->data_ptr(), B, M, N, K, M * K, K, N * K, K, M * N, N, 1, 128, 128, kb * ld, ld,
        nb * kb, kb, MAXFP8_BF16, MAXFP8_F32, MAXFP8_ALGO_AUTO, stream);
  });
  if (status != MAXFP8_OK) return raise(status);
  return THPVariable_Wrap(std::move(c));
}

// silu(gate) * up of every row, rounded twice to bf16, and the down linear: see MLP
bool silu_group_ok(int64_t rows, int64_t inter, int granularity) {
  // (the rule of moe_kernels.silu_quantize_group)
  return inter % 128 == 0 && (granularity == MAXFP8_GRAN_BLOCK || (inter > 128 && inter <= (rows >= 128 ? 32768 : 14336)));
}

// mlp(x, gate_up, gate_up_scales, down, down_scales, granularity, row_offsets [0, rows], scale_ub) -> y
PyObject* mlp(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  NEED_ARGS(8)
  const at::Tensor *x = tensor(args[0]), *gu = tensor(args[1]), *sgu = tensor(args[2]), *d = tensor(args[3]), *sd = tensor(args[4]), *rows = tensor(args[6]);
  const int granularity = (int)PyLong_AsLong(args[5]);
  const float ub = (float)PyFloat_AsDouble(args[7]);
  if (PyErr_Occurred()) return nullptr;
  if (!x || !gu || !sgu || !d || !sd || !rows || !linear_ok(*x, *gu, *sgu, granularity) || gu->size(0) % 2 != 0 || !fp8_rows(*d) || !on_gpu(*d, *x) ||
      d->size(1) * 2 != gu->size(0) || !weight_scales_ok(*sd, *d, granularity) || !on_gpu(*rows, *x) || rows->numel() != 2 ||
      rows->scalar_type() != at::kUInt32 || !silu_group_ok(x->size(0), d->size(1), granularity))
    Py_RETURN_NONE;
  void* stream;
  if (!stream_of(*x, &stream)) return nullptr;
  const int64_t M = x->size(0), F = d->size(1), H = d->size(0);
  const bool block = granularity == MAXFP8_GRAN_BLOCK;
  const int64_t group = block ? 128 : F, ld = block ? (M + 3) / 4 * 4 : M;
  // one buffer: the quantised product, its scales, the down matmul's partial sums
  const size_t at_scales = ((size_t)M * (size_t)F + 255) / 256 * 256, at_partial = at_scales + ((size_t)(F / group) * (size_t)ld * 4 + 255) / 256 * 256;
  at::Tensor y;
  const int status = unlocked([&] {
    at::Tensor both;
    int rc = linear_of(both, *x, *gu, *sgu, granularity, ub, stream);
    if (rc != MAXFP8_OK) return rc;
    const size_t partial = maxfp8_matmul_auto_workspace_bytes(M, H, F);
    at::Tensor ws = bytes_on(*x, at_partial + partial);
    uint8_t* q = static_cast<uint8_t*>(ws.data_ptr());
    rc = maxfp8_silu_quantize_dynamic_scaled_fp8(q, q + at_scales, both.data_ptr(), static_cast<const uint32_t*>(rows->data_ptr()), 2, M, F, 2 * F, F,
        group, ld, MAXFP8_BF16, 1, ub, stream);
    if (rc != MAXFP8_OK) return rc;
    y = at::empty({M, H}, x->options());
    return maxfp8_matmul_dynamic_scaled_fp8(y.data_ptr(), q, d->data_ptr(), q + at_scales, sd->data_ptr(), M, H, F, F, row_stride(*d), H,
        block ? MAXFP8_GRAN_BLOCK : MAXFP8_GRAN_COLWISE, granularity, block ? 1 : -1, block ? 128 : -1,
        block ? 128 : -1, ld, sd->size(1), MAXFP8_BF16, MAXFP8_F32, MAXFP8_ALGO_AUTO,
        partial ? q + at_partial : nullptr, partial, stream);
  });
  if (status != MAXFP8_OK) return raise(status);
  return THPVariable_Wrap(std::move(y));
}

// qkv_linear(x, wqkv, w_scales, granularity, scale_ub, row_offsets, kv_blocks, cache_lengths, lookup_table, bias or None, layer, q_dim) -> q
PyObject* qkv_linear(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  NEED_ARGS(12)
  const at::Tensor *x = tensor(args[0]), *w = tensor(args[1]), *s = tensor(args[2]), *offsets = tensor(args[5]), *blocks = tensor(args[6]),
                   *lengths = tensor(args[7]), *table = tensor(args[8]), *bias = tensor(args[9]);
  const int granularity = (int)PyLong_AsLong(args[3]);
  const float ub = (float)PyFloat_AsDouble(args[4]);
  const int64_t layer = PyLong_AsLongLong(args[10]), q_dim = PyLong_AsLongLong(args[11]);
  if (PyErr_Occurred()) return nullptr;
  auto u32 = [&](const at::Tensor* t, int64_t dim) {
    return t && on_gpu(*t, *x) && (t->scalar_type() == at::kInt || t->scalar_type() == at::kUInt32) && t->dim() == dim && t->is_contiguous();
  };
  if (!x || !w || !s || !linear_ok(*x, *w, *s, granularity) || !w->is_contiguous() || !u32(offsets, 1) || !u32(lengths, 1) || !u32(table, 2) ||
      !blocks || !on_gpu(*blocks, *x) || blocks->scalar_type() != at::kBFloat16 || blocks->dim() != 6 || !blocks->is_contiguous() || q_dim <= 0)
    Py_RETURN_NONE;
  const int64_t T = x->size(0), K = x->size(1), N = w->size(0), batch = offsets->size(0) - 1;
  if (batch < 1 || lengths->size(0) < batch || table->size(0) < batch) Py_RETURN_NONE;
  if (args[9] != Py_None && (!bias || !on_gpu(*bias, *x) || bias->scalar_type() != at::kBFloat16 || bias->numel() != N || !bias->is_contiguous()))
    Py_RETURN_NONE;
  void* stream;
  if (!stream_of(*x, &stream)) return nullptr;
  at::Tensor q;
  const int status = unlocked([&] {
    q = at::empty({T, q_dim}, x->options());
    const size_t need = maxfp8_linear_qkv_workspace_bytes(T, N, K, granularity);
    at::Tensor ws;
    if (need) ws = bytes_on(*x, need);
    return maxfp8_linear_qkv_ragged_paged_scale(
        q.data_ptr(), x->data_ptr(), row_stride(*x), static_cast<const uint32_t*>(offsets->data_ptr()), w->data_ptr(), s->data_ptr(), blocks->data_ptr(),
        static_cast<const uint32_t*>(lengths->data_ptr()), static_cast<const uint32_t*>(table->data_ptr()), bias ? bias->data_ptr() : nullptr, T, N, K,
        q_dim, batch, blocks->size(0), blocks->size(1), blocks->size(2), layer, blocks->size(3), blocks->size(4), blocks->size(5), table->size(1),
        granularity, s->size(1), ub, need ? ws.data_ptr() : nullptr, need, stream);
  });
  if (status != MAXFP8_OK) return raise(status);
  return THPVariable_Wrap(std::move(q));
}

// moe_experts(x, router [seq, k] int32, gate_up [E, 2I, H], its scales, down [E, H, I], its scales, scale_ub, host_sync) -> [seq, k, H]
PyObject* moe_experts(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
  NEED_ARGS(8)
  const at::Tensor *x = tensor(args[0]), *r = tensor(args[1]), *gu = tensor(args[2]), *sgu = tensor(args[3]), *d = tensor(args[4]), *sd = tensor(args[5]);
  const float ub = (float)PyFloat_AsDouble(args[6]);
  const bool host_sync = PyObject_IsTrue(args[7]) > 0;
  if (PyErr_Occurred()) return nullptr;
  auto ok = [&](const at::Tensor* t, at::ScalarType kind) { return t && on_gpu(*t, *x) && t->scalar_type() == kind && t->dim() == 3 && t->is_contiguous() && t->numel() > 0; };
  if (!x || !bf16_rows(*x) || !r || !on_gpu(*r, *x) || r->scalar_type() != at::kInt || r->dim() != 2 || !r->is_contiguous() || r->size(0) != x->size(0) ||
      r->size(1) < 1 || !ok(gu, at::kFloat8_e4m3fn) || !ok(sgu, at::kFloat) || !ok(d, at::kFloat8_e4m3fn) || !ok(sd, at::kFloat))
    Py_RETURN_NONE;
  const int64_t seq = x->size(0), H = x->size(1), k = r->size(1), E = gu->size(0), F = d->size(2), T = seq * k, ld = (T + 3) / 4 * 4;
  if (gu->size(1) != 2 * F || gu->size(2) != H || d->size(0) != E || d->size(1) != H || H % 128 != 0 || F % 128 != 0 || E > 65535 ||
      sgu->size(0) != E || sgu->size(1) != (2 * F) / 128 || sgu->size(2) != H / 128 || sd->size(0) != E || sd->size(1) != H / 128 || sd->size(2) != F / 128 ||
      !aligned16(gu->data_ptr()) || !aligned16(d->data_ptr()))
    Py_RETURN_NONE;
  void* stream;
  if (!stream_of(*x, &stream)) return nullptr;
  at::Tensor y;
  const int status = unlocked([&] {
    // the grouping: order [T], restore [T], starts [E + 1], expert ids [E], usage [2]
    at::Tensor idx = at::empty({2 * T + 2 * E + 8}, x->options().dtype(at::kInt));
    uint32_t* order = static_cast<uint32_t*>(idx.data_ptr());
    uint32_t *restore = order + T, *start = restore + T, *ids = start + E + 1, *usage = ids + E;
    const int32_t* expert_ids = reinterpret_cast<const int32_t*>(ids);
    int rc = maxfp8_moe_create_indices(order, start, restore, reinterpret_cast<int32_t*>(ids), usage, r->data_ptr(), T, E, stream);
    if (rc != MAXFP8_OK) return rc;
    // the two host scalars of the grouped matmuls: copied, which waits for the grouping (12 us of the 2300 that 4096 tokens of 8
    // experts take), or their bounds (every row on one expert, every expert in use)
    int64_t most = T, active = E;
    if (host_sync) {
      const at::Tensor stats = idx.narrow(0, usage - order, 2).cpu();
      most = static_cast<const int32_t*>(stats.data_ptr())[0];
      active = static_cast<const int32_t*>(stats.data_ptr())[1];
    }
    // every token quantised once and stored to its k rows of the grouped order
    at::Tensor q = at::empty({T, H}, x->options().dtype(at::kFloat8_e4m3fn)), s = at::empty({H / 128, ld}, x->options().dtype(at::kFloat));
    rc = maxfp8_quantize_dynamic_scaled_fp8_scatter(q.data_ptr(), s.data_ptr(), x->data_ptr(), restore, k, seq, H, T, row_stride(*x), H, 128, ld,
        MAXFP8_BF16, MAXFP8_F32, ub, stream);
    if (rc != MAXFP8_OK) return rc;
    at::Tensor both = at::empty({T, 2 * F}, x->options());
    rc = maxfp8_grouped_matmul_dynamic_scaled_fp8(both.data_ptr(), q.data_ptr(), gu->data_ptr(), s.data_ptr(), sgu->data_ptr(), start, expert_ids,
        T, 2 * F, H, E, most, active, ld, MAXFP8_BF16, MAXFP8_F32, MAXFP8_ALGO_AUTO, stream);
    if (rc != MAXFP8_OK) return rc;
    at::Tensor hq = at::empty({T, F}, x->options().dtype(at::kFloat8_e4m3fn)), hs = at::empty({F / 128, ld}, x->options().dtype(at::kFloat));
    rc = maxfp8_silu_quantize_dynamic_scaled_fp8(hq.data_ptr(), hs.data_ptr(), both.data_ptr(), start, E + 1, T, F, 2 * F, F, 128, ld, MAXFP8_BF16, 0,
        ub, stream);
    if (rc != MAXFP8_OK) return rc;
    y = at::empty({seq, k, H}, x->options());
    return maxfp8_grouped_matmul_dynamic_scaled_fp8_scatter(y.data_ptr(), order, hq.data_ptr(), d->data_ptr(), hs.data_ptr(), sd->data_ptr(), start,
        expert_ids, T, H, F, E, most, active, ld, MAXFP8_BF16, MAXFP8_F32, MAXFP8_ALGO_AUTO, stream);
  });
  if (status != MAXFP8_OK) return raise(status);
  return THPVariable_Wrap(std::move(y));
}

#define METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&guarded<name>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(linear), METHOD(linear_static), METHOD(quantize), METHOD(rms_norm_quantize), METHOD(matmul),
                         METHOD(batched_quantize), METHOD(batched_matmul), METHOD(mlp), METHOD(qkv_linear), METHOD(moe_experts),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "The hot operators of modular_amd, checks and allocation included.", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__native() {
  PyObject* torch_c = PyImport_ImportModule("torch._C");
  if (!torch_c) return nullptr;
  g_raw_stream = PyObject_GetAttrString(torch_c, "_cuda_getCurrentRawStream");
  Py_DECREF(torch_c);
  if (!g_raw_stream) return nullptr;
  return PyModule_Create(&module);
}
