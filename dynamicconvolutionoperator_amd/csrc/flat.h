// Flat copies of NCHW tensors (FlatLay, ddpm_common.h) for the kernels that
// stage whole 16-byte chunks.
#pragma once

#include "ddpm_common.h"

namespace ddpm {

// One tensor to lay out flat: src [n][c][H][W] -> dst (flat, cp planes per
// image; planes c .. cp-1 and everything outside the images zero).
struct FlatCopy {
  const void* src;
  void* dst;
  uint32_t c, cp;
  uint32_t chunks;  // 8-element chunks of dst (0: no copy)
};

inline FlatCopy flat_copy_of(const void* src, void* dst, const FlatLay& f, int64_t n, int64_t c,
                             int64_t cp) {
  return FlatCopy{src, dst, (uint32_t)c, (uint32_t)cp, (uint32_t)(flat_elems(f, n * cp) / 8)};
}

// One 8-element chunk of a destination: it lies in one row (P, S and lead are
// multiples of 8), and its source elements are read by two vector loads of
// any alignment, or one by one in the last chunk of a row.
template <typename T>
__device__ __forceinline__ void flat_copy_chunk(const FlatCopy& t, const FlatLay& f, uint32_t idx) {
  const T* __restrict__ src = static_cast<const T*>(t.src);
  T* __restrict__ dst = static_cast<T*>(t.dst) + (size_t)idx * 8;
  typedef T V8 __attribute__((ext_vector_type(8)));
  V8 v = {(T)0.f, (T)0.f, (T)0.f, (T)0.f, (T)0.f, (T)0.f, (T)0.f, (T)0.f};
  const uint32_t lead8 = f.lead / 8;
  if (idx >= lead8) {
    const uint32_t s8 = f.S / 8, p8 = (uint32_t)f.P / 8;
    const uint32_t i = idx - lead8;
    const uint32_t plane = i / s8, k = i - plane * s8;
    const uint32_t n = plane / t.cp, c = plane - n * t.cp;
    const uint32_t h = k / p8, w = (k - h * p8) * 8;
    if (c < t.c && h < (uint32_t)f.H && w < (uint32_t)f.W) {
      const T* __restrict__ s = src + (((size_t)n * t.c + c) * f.H + h) * f.W + w;
      if (w + 8 <= (uint32_t)f.W) {
        __builtin_memcpy(&v, s, sizeof(v));
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e)
          if (w + e < (uint32_t)f.W) v[e] = s[e];
      }
    }
  }
  *reinterpret_cast<V8*>(dst) = v;
}

// Lays out `count` (1 or 2) tensors of `dtype` and the same n, H, W flat in one
// launch.  Defined in flat.hip.
int flat_copy(const FlatCopy* t, int count, const FlatLay& f, int dtype, hipStream_t stream);

// Zeroing of the elements of a flat tensor (`planes` planes in all) that lie
// outside the images, shared out over the workgroups of the launch that
// writes the images.
struct FlatZero {
  void* base;  // null: nothing to do
  FlatLay f;
  int planes;
};

template <typename T>
__device__ __forceinline__ void flat_zero_share(const FlatZero& z, int wg, int wgs, int tid,
                                                int nthreads) {
  T* __restrict__ base = static_cast<T*>(z.base);
  const FlatLay& f = z.f;
  const int stride = wgs * nthreads, first = wg * nthreads + tid;
  const uint32_t tail = f.S - (uint32_t)(f.H * f.P);  // a multiple of 8
  typedef uint32_t V4 __attribute__((ext_vector_type(4)));
  constexpr int VE = 16 / (int)sizeof(T);
  const V4 zero = {0u, 0u, 0u, 0u};
  // the lead and the tail of every plane, 16 bytes at a time
  const uint32_t lv = f.lead / VE, tv = tail / VE;
  for (uint32_t i = first; i < lv; i += stride) reinterpret_cast<V4*>(base)[i] = zero;
  const uint32_t tot = tv * (uint32_t)z.planes;
  for (uint32_t i = first; i < tot; i += stride) {
    const uint32_t pl = i / tv, k = i - pl * tv;
    reinterpret_cast<V4*>(base + f.lead + (size_t)pl * f.S + (size_t)f.H * f.P)[k] = zero;
  }
  // the pad columns of every row
  const uint32_t pad = (uint32_t)(f.P - f.W), rows = (uint32_t)z.planes * (uint32_t)f.H;
  for (uint32_t i = first; i < rows; i += stride) {
    const uint32_t pl = i / (uint32_t)f.H, h = i - pl * (uint32_t)f.H;
    T* __restrict__ d = base + f.lead + (size_t)pl * f.S + (size_t)h * f.P + f.W;
    for (uint32_t e = 0; e < pad; ++e) d[e] = (T)0.f;
  }
}

}  // namespace ddpm
