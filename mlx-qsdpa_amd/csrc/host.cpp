// The per-call host path of the torch wrappers (mlx_qsdpa_amd/kernels.py):
// reads the tensors, fills the C ABI's argument structs and calls it.
//
// A decode step makes two such calls and six views.  In Python (shape checks,
// ctypes structs, slicing) they took 13 us (update), 9 us (views) and 13 us
// (attention) of host time, more than the kernels of every short step: one
// sequence over 4096 keys 35.2 us a step against 18.7 here, a window of four
// 36.7 against 19.6; a decode under a mask tensor (two sequences of 16 / 4
// 128-wide heads over 2000 keys) 25.3 against 10.1.
//
// Every function takes only what it can check in full: plain strided tensors
// on one GPU with the shapes, types and strides the wrapper would accept as
// they are.  For anything else it returns None before doing anything, and the
// wrapper goes on with its general path, which converts or raises.  C++
// exceptions (an allocation that fails) become Python ones; every other
// failure is the C ABI's negative code, returned.  No tensor, address or
// geometry is kept from one call to the next.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <ATen/ATen.h>
#include <ATen/TensorSubclassLikeUtils.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <hip/hip_runtime_api.h>

#include <algorithm>
#include <vector>

#include "../../include/qsdpa.h"

namespace {

// A plain CUDA (ROCm) tensor of 4 dimensions with contiguous rows, or null.
const at::Tensor* plain(PyObject* o) {
  if (!THPVariable_CheckExact(o)) return nullptr;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.is_cuda() || t.layout() != at::kStrided || t.is_conj() || t.is_neg() || at::isTensorSubclassLike(t))
    return nullptr;
  return &t;
}

const at::Tensor* plain4(PyObject* o) {
  const at::Tensor* t = plain(o);
  return t && t->dim() == 4 && (t->stride(3) == 1 || t->size(3) <= 1) ? t : nullptr;
}

bool shaped(const at::Tensor& t, int64_t b, int64_t h, int64_t n, int64_t w) {
  return t.size(0) == b && t.size(1) == h && t.size(2) == n && t.size(3) == w;
}

qsdpa_view view(const at::Tensor& t) { return {t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)}; }

bool fits32(std::initializer_list<int64_t> xs) {
  for (int64_t x : xs)
    if (x < 0 || x > INT32_MAX) return false;
  return true;
}

bool as_int(PyObject* o, int64_t& x) {
  if (!PyLong_CheckExact(o)) return false;
  x = PyLong_AsLongLong(o);
  if (x == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    return false;
  }
  return true;
}

int dtype_of(const at::Tensor& t) {
  return t.scalar_type() == at::kHalf ? QSDPA_F16 : t.scalar_type() == at::kBFloat16 ? QSDPA_BF16 : -1;
}

void* stream_of(int64_t x) { return reinterpret_cast<void*>(static_cast<intptr_t>(x)); }

// The interpreter's lock is released over a launch, which may wait for room in
// the stream's queue (as ctypes releases it on the general path).
template <typename F>
auto unlocked(F&& launch) {
  struct Lock {
    PyThreadState* state = PyEval_SaveThread();
    ~Lock() { PyEval_RestoreThread(state); }
  } lock;
  return launch();
}

bool capturing(void* stream) {
  hipStreamCaptureStatus st = hipStreamCaptureStatusNone;
  return hipStreamIsCapturing(static_cast<hipStream_t>(stream), &st) != hipSuccess || st != hipStreamCaptureStatusNone;
}

// One quantize job: src [B, H, S, D] into columns [t0, t0 + S) of the
// (packed, scales, biases) buffers; false if it is not such a job.
bool quantize_job(PyObject* src_o, PyObject* dst_o, int64_t t0, int64_t bits, int64_t gs, qsdpa_quantize_args& j) {
  const at::Tensor* src = plain4(src_o);
  if (!src || !PyTuple_CheckExact(dst_o) || PyTuple_GET_SIZE(dst_o) != 3) return false;
  const at::Tensor* d[3];
  for (int i = 0; i < 3; ++i)
    if (!(d[i] = plain4(PyTuple_GET_ITEM(dst_o, i))) || d[i]->device() != src->device()) return false;
  const int64_t B = src->size(0), H = src->size(1), S = src->size(2), D = src->size(3), cap = d[0]->size(2);
  const int dt = dtype_of(*src);
  if (dt < 0 || (bits != 4 && bits != 8) || gs <= 0 || D <= 0 || D % gs || t0 < 0 || S > cap || t0 > cap - S)
    return false;
  if (!shaped(*d[0], B, H, cap, D * bits / 32) || !shaped(*d[1], B, H, cap, D / gs) ||
      !shaped(*d[2], B, H, cap, D / gs))
    return false;
  if (d[0]->scalar_type() != at::kUInt32 || d[1]->scalar_type() != src->scalar_type() ||
      d[2]->scalar_type() != src->scalar_type() || !fits32({B, H, cap, D, gs}))
    return false;
  j.B = B; j.H = H; j.S = S; j.D = D;
  j.bits = bits; j.group_size = gs; j.dtype = dt; j.t0 = t0;
  j.src = view(*src);
  j.dst_packed = view(*d[0]); j.dst_scales = view(*d[1]); j.dst_biases = view(*d[2]);
  return true;
}

// quantize_kv(keys, values, kdst, vdst, t0, bits, group_size, stream):
// the code of qsdpa_quantize_batch, or None.
PyObject* quantize_kv(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t t0, bits, gs, stream;
  qsdpa_quantize_args j[2];
  if (n != 8 || !as_int(a[4], t0) || !as_int(a[5], bits) || !as_int(a[6], gs) || !as_int(a[7], stream) ||
      !quantize_job(a[0], a[2], t0, bits, gs, j[0]) || !quantize_job(a[1], a[3], t0, bits, gs, j[1]) ||
      j[0].dtype != j[1].dtype || THPVariable_Unpack(a[0]).device() != THPVariable_Unpack(a[1]).device())
    Py_RETURN_NONE;
  return PyLong_FromLong(unlocked([&] { return qsdpa_quantize_batch(j, 2, stream_of(stream)); }));
  END_HANDLE_TH_ERRORS
}

// columns(buffers, n): the first n columns (dim 2) of each tensor of a
// tuple, as a tuple of views, or None.
PyObject* columns(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t cols;
  if (n != 2 || !PyTuple_CheckExact(a[0]) || !as_int(a[1], cols) || cols < 0) Py_RETURN_NONE;
  const Py_ssize_t k = PyTuple_GET_SIZE(a[0]);
  for (Py_ssize_t i = 0; i < k; ++i) {
    PyObject* o = PyTuple_GET_ITEM(a[0], i);
    if (!THPVariable_CheckExact(o) || THPVariable_Unpack(o).dim() != 4) Py_RETURN_NONE;
  }
  THPObjectPtr out(PyTuple_New(k));
  if (!out) return nullptr;
  for (Py_ssize_t i = 0; i < k; ++i) {
    PyObject* v = THPVariable_Wrap(THPVariable_Unpack(PyTuple_GET_ITEM(a[0], i)).slice(2, 0, cols));
    if (!v) return nullptr;
    PyTuple_SET_ITEM(out.get(), i, v);
  }
  return out.release();
  END_HANDLE_TH_ERRORS
}

// grown(keys, values, old, prev, cols, bits, group_size, stream): six new
// buffers of `cols` columns (packed, scales, biases of the keys, then of the
// values): columns [0, prev) from `old` (the six held ones, or None), zeros
// from prev + S on, the S between left for the caller to write.  Their tuple,
// the negative code of qsdpa_move_rows, or None.
PyObject* grown(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t prev, cols, bits, gs, stream;
  const at::Tensor *kv[2], *old[6] = {};
  if (n != 8 || !(kv[0] = plain4(a[0])) || !(kv[1] = plain4(a[1])) || !as_int(a[3], prev) || !as_int(a[4], cols) ||
      !as_int(a[5], bits) || !as_int(a[6], gs) || !as_int(a[7], stream) || (bits != 4 && bits != 8) || gs <= 0)
    Py_RETURN_NONE;
  const int64_t B = kv[0]->size(0), H = kv[0]->size(1), S = kv[0]->size(2);
  for (const at::Tensor* t : kv)
    if (dtype_of(*t) < 0 || t->scalar_type() != kv[0]->scalar_type() || t->device() != kv[0]->device() ||
        !shaped(*t, B, H, S, t->size(3)) || t->size(3) <= 0 || t->size(3) % gs)
      Py_RETURN_NONE;
  if (prev < 0 || B < 1 || H < 1 || S > cols - prev || !fits32({B * H, cols})) Py_RETURN_NONE;
  int64_t width[6];
  at::ScalarType type[6];
  for (int i = 0; i < 6; ++i) {
    const int64_t D = kv[i / 3]->size(3);
    width[i] = i % 3 ? D / gs : D * bits / 32;
    type[i] = i % 3 ? kv[0]->scalar_type() : at::kUInt32;
  }
  if (prev > 0) {
    if (!PyTuple_CheckExact(a[2]) || PyTuple_GET_SIZE(a[2]) != 6) Py_RETURN_NONE;
    for (int i = 0; i < 6; ++i) {
      const at::Tensor* t = old[i] = plain4(PyTuple_GET_ITEM(a[2], i));
      // (batch, head) rows that follow one another, so one move covers them.
      if (!t || t->device() != kv[0]->device() || t->scalar_type() != type[i] || t->size(2) < prev ||
          !shaped(*t, B, H, t->size(2), width[i]) || (B > 1 && t->stride(0) != H * t->stride(1)))
        Py_RETURN_NONE;
    }
  }
  THPObjectPtr out(PyTuple_New(6));
  if (!out) return nullptr;
  qsdpa_row_move moves[12];
  int count = 0;
  for (int i = 0; i < 6; ++i) {
    at::Tensor t = at::empty({B, H, cols, width[i]}, kv[0]->options().dtype(type[i]).requires_grad(false));
    const int64_t es = t.element_size(), row = width[i] * es;
    qsdpa_row_move m = {};
    m.dst_head_stride = cols * row;
    m.dst_token_stride = row;
    m.heads = B * H;
    m.row_bytes = row;
    if (prev + S < cols) {
      m.dst = static_cast<uint8_t*>(t.data_ptr()) + (prev + S) * row;
      m.tokens = cols - prev - S;
      moves[count++] = m;
    }
    if (prev > 0) {
      m.src = old[i]->data_ptr();
      m.src_head_stride = old[i]->stride(1) * es;
      m.src_token_stride = old[i]->stride(2) * es;
      m.dst = t.data_ptr();
      m.tokens = m.copy_end = prev;
      moves[count++] = m;
    }
    PyObject* o = THPVariable_Wrap(std::move(t));
    if (!o) return nullptr;
    PyTuple_SET_ITEM(out.get(), i, o);
  }
  const int rc = unlocked([&] { return qsdpa_move_rows(moves, count, stream_of(stream)); });
  return rc ? PyLong_FromLong(rc) : out.release();
  END_HANDLE_TH_ERRORS
}

// A mask of 1 to 4 dimensions that broadcasts to [B, H, L, N] with its keys
// adjacent, as x's mask; false for any other.
bool mask_view(const at::Tensor& m, int64_t B, int64_t H, int64_t L, int64_t N, qsdpa_decode_args& x) {
  switch (m.scalar_type()) {
    case at::kBool: x.mask_dtype = QSDPA_BOOL; break;
    case at::kHalf: x.mask_dtype = QSDPA_F16; break;
    case at::kBFloat16: x.mask_dtype = QSDPA_BF16; break;
    case at::kFloat: x.mask_dtype = QSDPA_F32; break;
    default: return false;
  }
  const int64_t d = m.dim(), to[4] = {B, H, L, N};
  if (d < 1 || d > 4 || m.size(d - 1) != N || (N > 1 && m.stride(d - 1) != 1)) return false;
  int64_t stride[3] = {0, 0, 0};  // of a broadcast dimension: 0
  for (int64_t i = 4 - d; i < 3; ++i) {
    const int64_t size = m.size(i - (4 - d));
    if (size != 1 && size != to[i]) return false;
    if (size > 1) stride[i] = m.stride(i - (4 - d));
  }
  x.mask = {m.data_ptr(), stride[0], stride[1], 1};
  x.mask_stride_q = stride[2];
  return true;
}

// The counters at a workspace's start (include/qsdpa.h).
constexpr int64_t kCounterBytes = 64 << 10;

// decode(q, packed_k, packed_v, k_scales, v_scales, k_biases, v_biases,
// scale, bits, group_size, kv_start, num_splits, causal, workspace, stream,
// mask): the output of qsdpa_decode; the workspace bytes it has use for
// (positive) when `workspace` (uint8, or None) is smaller: the split-K
// scratch, then a masked prefill's key ranges; its negative code; or None.
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t bits, gs, splits, stream;
  if (n != 16 || !PyFloat_Check(a[7]) || !as_int(a[8], bits) || !as_int(a[9], gs) || !as_int(a[11], splits) ||
      !as_int(a[14], stream) || !PyBool_Check(a[12]) || (bits != 4 && bits != 8) || gs <= 0)
    Py_RETURN_NONE;
  const at::Tensor* t[7];
  for (int i = 0; i < 7; ++i) {
    t[i] = i > 4 && a[i] == Py_None ? nullptr : plain4(a[i]);
    if (!t[i] && (i < 5 || a[i] != Py_None)) Py_RETURN_NONE;
    if (t[i] && t[i]->device() != t[0]->device()) Py_RETURN_NONE;
  }
  if ((t[5] == nullptr) != (t[6] == nullptr)) Py_RETURN_NONE;
  const at::Tensor& q = *t[0];
  const int64_t B = q.size(0), Hq = q.size(1), L = q.size(2), D = q.size(3), Hkv = t[1]->size(1), N = t[1]->size(2);
  const int dt = dtype_of(q);
  if (dt < 0 || D <= 0 || D % gs || D * bits % 32 || L < 1 || Hkv < 1 || Hq % Hkv || !fits32({B, Hq, L, D, N, gs, splits}))
    Py_RETURN_NONE;
  for (int i = 1; i < 7; ++i) {
    if (!t[i]) continue;
    if (!shaped(*t[i], B, Hkv, N, i < 3 ? D * bits / 32 : D / gs) ||
        t[i]->scalar_type() != (i < 3 ? at::kUInt32 : q.scalar_type()))
      Py_RETURN_NONE;
    // Packed rows on 16-byte boundaries (the wrapper copies others).
    if (i < 3 && (reinterpret_cast<uintptr_t>(t[i]->data_ptr()) % 16 || t[i]->stride(0) % 4 || t[i]->stride(1) % 4 ||
                  t[i]->stride(2) % 4))
      Py_RETURN_NONE;
  }
  qsdpa_decode_args x = {};
  x.B = B; x.H_q = Hq; x.H_kv = Hkv; x.N = N; x.D = D;
  x.bits = bits; x.group_size = gs; x.dtype = dt;
  x.scale = static_cast<float>(PyFloat_AS_DOUBLE(a[7]));
  x.q = view(q);
  x.k_packed = view(*t[1]); x.v_packed = view(*t[2]);
  x.k_scales = view(*t[3]); x.v_scales = view(*t[4]);
  if (t[5]) {
    x.k_biases = view(*t[5]);
    x.v_biases = view(*t[6]);
  }
  if (a[10] != Py_None) {
    const at::Tensor* ks = plain(a[10]);
    if (!ks || ks->device() != q.device() || ks->scalar_type() != at::kInt || ks->dim() != 1 || ks->size(0) != B ||
        !ks->is_contiguous())
      Py_RETURN_NONE;
    x.kv_start = ks->data_ptr<int32_t>();
  }
  if (a[15] != Py_None) {
    const at::Tensor* m = plain(a[15]);
    if (!m || m->device() != q.device() || !mask_view(*m, B, Hq, L, N, x)) Py_RETURN_NONE;
  }
  x.num_splits = splits;
  x.q_len = L;
  x.causal = a[12] == Py_True;
  x.out = x.q;  // (planning reads q's strides only; set below)
  int32_t planned = 1;
  const int64_t ws = qsdpa_decode_workspace_size(&x, &planned);
  if (ws < 0) return PyLong_FromLongLong(ws);
  const int64_t rb = x.mask.ptr && L > 1 ? qsdpa_decode_range_bytes(&x) : 0;
  if (rb < 0) return PyLong_FromLongLong(rb);
  const int64_t at_ranges = std::max<int64_t>(ws, kCounterBytes), total = rb > 0 ? at_ranges + rb : ws;
  void* ranges = nullptr;
  if (total > 0) {
    // A captured call takes a workspace of its own (the wrapper's general path).
    if (capturing(stream_of(stream))) Py_RETURN_NONE;
    const at::Tensor* w = a[13] == Py_None ? nullptr : plain(a[13]);
    if (!w || w->device() != q.device() || static_cast<int64_t>(w->nbytes()) < total)
      return PyLong_FromLongLong(total);
    x.workspace = w->data_ptr();
    x.workspace_bytes = ws;
    if (rb > 0) ranges = static_cast<uint8_t*>(w->data_ptr()) + at_ranges;
  }
  at::Tensor out = at::empty(q.sizes(), q.options().requires_grad(false));
  x.out = view(out);
  const int rc = unlocked([&] { return qsdpa_decode_ranges(&x, ranges, rb, stream_of(stream)); });
  return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// The values of a plain CPU int64 vector; false for anything else.
bool positions(PyObject* o, std::vector<int64_t>& x) {
  if (!THPVariable_CheckExact(o)) return false;
  const at::Tensor& t = THPVariable_Unpack(o);
  if (!t.device().is_cpu() || t.layout() != at::kStrided || at::isTensorSubclassLike(t) || t.dim() != 1 ||
      t.scalar_type() != at::kLong)
    return false;
  x.resize(t.numel());
  for (int64_t i = 0; i < t.numel(); ++i) x[i] = t.data_ptr<int64_t>()[i * t.stride(0)];
  return true;
}

// causal_mask(N, start, pad, window, device, stream): the bool mask
// [B, 1, N, max(start) + N] for CPU vectors start and pad (or None), or
// [N, start + N] for an int start and no pad, on GPU `device`; the negative
// code of qsdpa_causal_mask; or None.
PyObject* causal_mask(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t N, first, window = int64_t(1) << 34, device, stream;
  if (n != 6 || !as_int(a[0], N) || !as_int(a[4], device) || !as_int(a[5], stream) ||
      (a[3] != Py_None && !as_int(a[3], window)) || c10::impl::dispatch_mode_enabled())
    Py_RETURN_NONE;
  int current = -1;
  if (hipGetDevice(&current) != hipSuccess || current != device) Py_RETURN_NONE;
  std::vector<int64_t> start, pad;
  const bool one = as_int(a[1], first);
  if (one) start.assign(1, first);
  else if (!positions(a[1], start)) Py_RETURN_NONE;
  if (a[2] != Py_None && (one || !positions(a[2], pad) || pad.size() != start.size())) Py_RETURN_NONE;
  if (start.empty() || N < 1 || window > (int64_t(1) << 34) || window < -(int64_t(1) << 34)) Py_RETURN_NONE;
  for (const auto* v : {&start, &pad})
    for (int64_t x : *v)
      if (x < INT32_MIN || x > INT32_MAX) Py_RETURN_NONE;
  const int64_t B = start.size(), total = *std::max_element(start.begin(), start.end()) + N;
  if (total < 1 || !fits32({B, N, total})) Py_RETURN_NONE;
  const auto options = at::TensorOptions().dtype(at::kBool).device(at::kCUDA, static_cast<c10::DeviceIndex>(device));
  at::Tensor out = one ? at::empty({N, total}, options) : at::empty({B, 1, N, total}, options);
  qsdpa_causal_mask_args x = {};
  x.B = B; x.N = N; x.total = total;
  x.window = window;
  x.start = start.data();
  x.pad = pad.empty() ? nullptr : pad.data();
  x.out = static_cast<uint8_t*>(out.data_ptr());
  const int rc = unlocked([&] { return qsdpa_causal_mask(&x, stream_of(stream)); });
  return rc ? PyLong_FromLong(rc) : THPVariable_Wrap(std::move(out));
  END_HANDLE_TH_ERRORS
}

// A tensor that no gradient, of either mode, is taken through.
bool constant(const at::Tensor& t) {
  return !(c10::GradMode::is_enabled() && t.requires_grad()) && !t._fw_grad(0).defined();
}

// rotate(q, k, start, theta, stream): q and k [B, H, L, D] with the rotary
// positions start (an int, or a CPU tensor of 1 or B of them) + l, as a tuple
// of contiguous tensors; the negative code of qsdpa_rotate; or None.
PyObject* rotate(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  int64_t stream, first = 0;
  if (n != 5 || !PyFloat_Check(a[3]) || !as_int(a[4], stream)) Py_RETURN_NONE;
  const at::Tensor *q = plain4(a[0]), *k = plain4(a[1]);
  if (!q || !k || !constant(*q) || !constant(*k) || q->device() != k->device() || dtype_of(*q) < 0 ||
      k->scalar_type() != q->scalar_type())
    Py_RETURN_NONE;
  int device = -1;
  if (hipGetDevice(&device) != hipSuccess || device != q->device().index()) Py_RETURN_NONE;
  const int64_t B = q->size(0), Hq = q->size(1), L = q->size(2), D = q->size(3), Hkv = k->size(1);
  if (B < 1 || L < 1 || D < 2 || D % 2 || D > 1024 || !shaped(*k, B, Hkv, L, D) || !fits32({B, Hq * D, Hkv * D, L}))
    Py_RETURN_NONE;
  std::vector<int64_t> start(B);
  if (THPVariable_CheckExact(a[2])) {
    const at::Tensor& t = THPVariable_Unpack(a[2]);
    if (!t.device().is_cpu() || t.layout() != at::kStrided || at::isTensorSubclassLike(t) || t.dim() > 1 ||
        t.scalar_type() != at::kLong || (t.numel() != 1 && t.numel() != B))
      Py_RETURN_NONE;
    const int64_t* x = t.data_ptr<int64_t>();
    const int64_t step = t.dim() == 1 && t.numel() == B ? t.stride(0) : 0;
    for (int64_t b = 0; b < B; ++b) start[b] = x[b * step];
  } else if (as_int(a[2], first)) {
    std::fill(start.begin(), start.end(), first);
  } else {
    Py_RETURN_NONE;
  }
  at::Tensor out[2] = {at::empty({B, Hq, L, D}, q->options().requires_grad(false)),
                       at::empty({B, Hkv, L, D}, q->options().requires_grad(false))};
  qsdpa_rotate_args x = {};
  x.B = B; x.H_q = Hq; x.H_kv = Hkv; x.L = L; x.D = D;
  x.dtype = dtype_of(*q);
  x.theta = static_cast<float>(PyFloat_AS_DOUBLE(a[3]));
  x.start = start.data();
  x.q = view(*q); x.k = view(*k);
  x.q_out = view(out[0]); x.k_out = view(out[1]);
  const int rc = unlocked([&] { return qsdpa_rotate(&x, stream_of(stream)); });
  if (rc) return PyLong_FromLong(rc);
  THPObjectPtr pair(PyTuple_New(2));
  if (!pair) return nullptr;
  for (int i = 0; i < 2; ++i) {
    PyObject* o = THPVariable_Wrap(std::move(out[i]));
    if (!o) return nullptr;
    PyTuple_SET_ITEM(pair.get(), i, o);
  }
  return pair.release();
  END_HANDLE_TH_ERRORS
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyCFunction fast() {
  return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F));
}

PyMethodDef methods[] = {
    {"quantize_kv", fast<quantize_kv>(), METH_FASTCALL, nullptr},
    {"columns", fast<columns>(), METH_FASTCALL, nullptr},
    {"grown", fast<grown>(), METH_FASTCALL, nullptr},
    {"decode", fast<decode>(), METH_FASTCALL, nullptr},
    {"causal_mask", fast<causal_mask>(), METH_FASTCALL, nullptr},
    {"rotate", fast<rotate>(), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() {
  if (qsdpa_abi_version() != QSDPA_ABI_VERSION)
    return PyErr_Format(PyExc_ImportError, "_host.so was built for ABI version %d of libqsdpa_hip.so, found %d",
                        QSDPA_ABI_VERSION, qsdpa_abi_version());
  return PyModule_Create(&module);
}
