// The bool mask of a causal pass over a cache: key k is attended by query i of
// sequence b where start[b] + i - window < k <= start[b] + i and k >= pad[b].
//
// Bound by its bytes, and at a prompt chunk's size by its launch.  As a torch
// expression it is three to five passes over [B, N, total] (comparisons and
// their conjunctions), the positions' copy to the device and two ranges: seven
// launches of 38 us for 8 sequences of 500 x 1500.  Here a thread writes 16
// bytes of the contiguous result, whose rows start at any byte: that chunk with
// its cache update and attention 175.0 us against 208.8.
#include <algorithm>

#include "abi_internal.h"
#include "common.h"

namespace qsdpa {
namespace {

constexpr int kThreads = 256;
constexpr int kMaxRows = 64;  // sequences per launch (positions travel in the kernel arguments)

struct MaskParams {
  uint8_t* out;
  int64_t bytes, window;
  int N, total;
  int64_t start[kMaxRows], pad[kMaxRows];
};

// I: the index type, 32-bit where a launch's bytes fit.
template <typename I>
__global__ __launch_bounds__(kThreads) void causal_mask_kernel(MaskParams p) {
  const I bytes = static_cast<I>(p.bytes), total = static_cast<I>(p.total);
  const I at = (static_cast<I>(blockIdx.x) * kThreads + threadIdx.x) * 16;
  if (at >= bytes) return;
  const I row = at / total;
  int b = static_cast<int>(row / static_cast<I>(p.N)), i = static_cast<int>(row - static_cast<I>(b) * static_cast<I>(p.N));
  int k = static_cast<int>(at - row * total), lo, hi;  // the row's keys [lo, hi]
  auto limits = [&]() {
    const int64_t q = p.start[b] + i;
    lo = static_cast<int>(min(max(max(p.pad[b], q - p.window + 1), int64_t(0)), int64_t(p.total)));
    hi = static_cast<int>(min(max(q, int64_t(-1)), int64_t(p.total)));
  };
  limits();
  const int n = bytes - at < 16 ? static_cast<int>(bytes - at) : 16;
  uint32_t w[4] = {0u, 0u, 0u, 0u};
#pragma unroll
  for (int e = 0; e < 16; ++e) {
    if (e < n) {
      if (k == p.total) {
        k = 0;
        if (++i == p.N) {
          i = 0;
          ++b;
        }
        limits();
      }
      w[e / 4] |= static_cast<uint32_t>(k >= lo && k <= hi) << (8 * (e % 4));
      ++k;
    }
  }
  uint8_t* out = p.out + at;
  if (n == 16) {
    __builtin_memcpy(out, w, 16);
  } else {
#pragma unroll
    for (int e = 0; e < 16; ++e)
      if (e < n) out[e] = static_cast<uint8_t>(w[e / 4] >> (8 * (e % 4)));
  }
}

}  // namespace

int launch_causal_mask(const qsdpa_causal_mask_args* a, hipStream_t stream) {
  MaskParams p;
  p.N = a->N;
  p.total = a->total;
  p.window = a->window;
  const int64_t each = static_cast<int64_t>(a->N) * a->total;
  for (int b0 = 0; b0 < a->B; b0 += kMaxRows) {
    const int n = std::min(kMaxRows, a->B - b0);
    for (int i = 0; i < kMaxRows; ++i) {
      p.start[i] = i < n ? a->start[b0 + i] : 0;
      p.pad[i] = i < n && a->pad ? a->pad[b0 + i] : 0;
    }
    p.out = a->out + b0 * each;
    p.bytes = n * each;
    const int64_t blocks = (p.bytes + 16 * kThreads - 1) / (16 * kThreads);
    const bool narrow = blocks * 16 * kThreads < (int64_t(1) << 32);
    hipLaunchKernelGGL(narrow ? causal_mask_kernel<uint32_t> : causal_mask_kernel<uint64_t>,
                       dim3(static_cast<unsigned>(blocks)), dim3(kThreads), 0, stream, p);
    const int rc = check_launch("causal_mask");
    if (rc) return rc;
  }
  return QSDPA_OK;
}

}  // namespace qsdpa
