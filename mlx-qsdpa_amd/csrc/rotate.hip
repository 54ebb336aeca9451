// Rotary positions of an attention layer's queries and keys, one launch.
//
// The half-split layout: element i of a head's first half and element
// i + D / 2 turn by the angle (start[b] + l) * theta^(-2 i / D), in float32,
// rounded to the storage type at the end -- operation for operation what the
// layer's torch expression computes (attention.py::_rope), with the same
// math library's powf, sinf and cosf, so the results are the same bits.
//
// A decode step is bound by its launches: the torch expression is two copies
// of positions to the device and 38 launches for q and k: one layer's step
// (2048 wide, 16 / 4 heads of 128, batch of 2, 4096 keys) 404.9 us, 131.0 with
// this kernel.
//
// One workgroup per token: the angles are shared by all heads, so each is
// computed once (one lane per angle) and read from the LDS by the heads of q
// and then k, in 16-byte pieces of both halves.
#include <algorithm>

#include "abi_internal.h"
#include "common.h"

namespace qsdpa {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxHalf = 512;   // angles per token: head dims to 1024
constexpr int kMaxStarts = 64;  // sequences per launch (positions travel in the kernel arguments)

struct RotatePart {
  const uint16_t* src;
  int64_t sb, sh, sn;
  uint16_t* dst;
  int64_t db, dh, dn;
  int heads;
};

struct RotateParams {
  RotatePart part[2];
  int half;
  float theta, inv_dim;
  int64_t start[kMaxStarts];
};

template <typename Tag, bool VEC>
__global__ __launch_bounds__(kThreads) void rotate_kernel(RotateParams p) {
#pragma clang fp contract(off)
  __shared__ float s_cos[kMaxHalf], s_sin[kMaxHalf];
  const int tid = threadIdx.x;
  const int64_t l = blockIdx.x, b = blockIdx.y;
  const float pos = static_cast<float>(p.start[b] + l);
  for (int i = tid; i < p.half; i += kThreads) {
    const float a = pos * powf(p.theta, -static_cast<float>(2 * i) * p.inv_dim);
    s_cos[i] = cosf(a);
    s_sin[i] = sinf(a);
  }
  __syncthreads();
  constexpr int E = VEC ? 8 : 1;  // elements of each half per unit
  const int per = p.half / E;
#pragma unroll
  for (int k = 0; k < 2; ++k) {
    const RotatePart& t = p.part[k];
    const uint16_t* src = t.src + b * t.sb + l * t.sn;
    uint16_t* dst = t.dst + b * t.db + l * t.dn;
    for (int u = tid; u < t.heads * per; u += kThreads) {
      const int h = u / per, i = (u - h * per) * E;
      const uint16_t* x = src + h * t.sh + i;
      uint16_t* y = dst + h * t.dh + i;
      alignas(16) uint16_t x1[E], x2[E], y1[E], y2[E];
      if constexpr (VEC) {
        *reinterpret_cast<uint4*>(x1) = *reinterpret_cast<const uint4*>(x);
        *reinterpret_cast<uint4*>(x2) = *reinterpret_cast<const uint4*>(x + p.half);
      } else {
        x1[0] = x[0];
        x2[0] = x[p.half];
      }
#pragma unroll
      for (int e = 0; e < E; ++e) {
        const float c = s_cos[i + e], s = s_sin[i + e], f1 = to_f32<Tag>(x1[e]), f2 = to_f32<Tag>(x2[e]);
        y1[e] = from_f32<Tag>(f1 * c - f2 * s);
        y2[e] = from_f32<Tag>(f2 * c + f1 * s);
      }
      if constexpr (VEC) {
        *reinterpret_cast<uint4*>(y) = *reinterpret_cast<const uint4*>(y1);
        *reinterpret_cast<uint4*>(y + p.half) = *reinterpret_cast<const uint4*>(y2);
      } else {
        y[0] = y1[0];
        y[p.half] = y2[0];
      }
    }
  }
}

// 16-byte pieces of a view's rows.
bool pieces(const void* ptr, int64_t sb, int64_t sh, int64_t sn) {
  return reinterpret_cast<uintptr_t>(ptr) % 16 == 0 && sb % 8 == 0 && sh % 8 == 0 && sn % 8 == 0;
}

}  // namespace

int launch_rotate(const qsdpa_rotate_args* a, hipStream_t stream) {
  RotateParams p;
  p.half = a->D / 2;
  p.theta = a->theta;
  p.inv_dim = 1.0f / static_cast<float>(a->D);
  bool vec = p.half % 8 == 0;
  const qsdpa_view *src[2] = {&a->q, &a->k}, *dst[2] = {&a->q_out, &a->k_out};
  const int heads[2] = {a->H_q, a->H_kv};
  for (int k = 0; k < 2; ++k) {
    p.part[k] = {static_cast<const uint16_t*>(src[k]->ptr), src[k]->stride_b, src[k]->stride_h, src[k]->stride_n,
                 static_cast<uint16_t*>(const_cast<void*>(dst[k]->ptr)), dst[k]->stride_b, dst[k]->stride_h,
                 dst[k]->stride_n, heads[k]};
    vec = vec && pieces(src[k]->ptr, src[k]->stride_b, src[k]->stride_h, src[k]->stride_n) &&
          pieces(dst[k]->ptr, dst[k]->stride_b, dst[k]->stride_h, dst[k]->stride_n);
  }
  const bool f16 = a->dtype == QSDPA_F16;
  void (*kernel)(RotateParams) = vec ? (f16 ? rotate_kernel<F16, true> : rotate_kernel<BF16, true>)
                                     : (f16 ? rotate_kernel<F16, false> : rotate_kernel<BF16, false>);
  for (int b0 = 0; b0 < a->B; b0 += kMaxStarts) {
    const int n = std::min(kMaxStarts, a->B - b0);
    for (int i = 0; i < kMaxStarts; ++i) p.start[i] = i < n ? a->start[b0 + i] : 0;
    hipLaunchKernelGGL(kernel, dim3(a->L, n), dim3(kThreads), 0, stream, p);
    const int rc = check_launch("rotate");
    if (rc) return rc;
    for (RotatePart& t : p.part) {
      t.src += n * t.sb;
      t.dst += n * t.db;
    }
  }
  return QSDPA_OK;
}

}  // namespace qsdpa
