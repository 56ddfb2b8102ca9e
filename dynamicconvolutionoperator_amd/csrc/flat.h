// Flat copies of NCHW tensors (FlatLay, ddpm_common.h) for the kernels that
// stage whole 16-byte chunks.
#pragma once

#include "ddpm_common.h"

namespace ddpm {

// Planes that one image of a flat concat of 2-byte elements takes (either
// form): its gradient keeps the C x-planes plane-major, since only
// element-wise code reads them, and the 3C branch planes channels-last in
// whole 16-channel blocks.
inline int64_t cl_cat_planes(int64_t c) { return c + (3 * c + 15) / 16 * 16; }

// One tensor to lay out flat: src [n][c][H][W] -> dst (flat, cp planes per
// image; planes c .. cp-1 and everything outside the images zero).
struct FlatCopy {
  const void* src;
  void* dst;
  uint32_t c, cp;
  uint32_t chunks;  // work items (0: no copy): 8 elements, or a position's 16 channels
};

inline FlatCopy flat_copy_of(const void* src, void* dst, const FlatLay& f, int64_t n, int64_t c,
                             int64_t cp, int esz) {
  return FlatCopy{src, dst, (uint32_t)c, (uint32_t)cp,
                  (uint32_t)(flat_elems(f, n * cp, esz) / (esz == 2 ? 16 : 8))};
}

// One item of a copy.  4-byte elements: 8 elements of one row (P, S and lead
// are multiples of 8), read by two vector loads of any alignment, or one by
// one at the end of a row.  2-byte elements: a position of a 16-channel block
// (channels-last), read from 16 planes; neighbouring lanes take neighbouring
// positions of each plane.
template <typename T>
__device__ __forceinline__ void flat_copy_chunk(const FlatCopy& t, const FlatLay& f, uint32_t idx) {
  const T* __restrict__ src = static_cast<const T*>(t.src);
  if constexpr (sizeof(T) == 2) {
    T* __restrict__ dst = static_cast<T*>(t.dst) + (size_t)idx * 16;
    uint32_t v[8] = {0u, 0u, 0u, 0u, 0u, 0u, 0u, 0u};
    if (idx >= f.lead) {
      const uint32_t i = idx - f.lead;
      const uint32_t blk = i / f.S, p = i - blk * f.S;
      const uint32_t n = blk / (t.cp / 16), c0 = (blk - n * (t.cp / 16)) * 16;
      const uint32_t h = p / (uint32_t)f.P, w = p - h * (uint32_t)f.P;
      if (c0 < t.c && h < (uint32_t)f.H && w < (uint32_t)f.W) {
        const size_t hw = (size_t)f.H * f.W;
        const uint16_t* __restrict__ s = reinterpret_cast<const uint16_t*>(src) +
                                         ((size_t)n * t.c + c0) * hw + (size_t)h * f.W + w;
        if (c0 + 16 <= t.c) {
          uint16_t e[16];
#pragma unroll
          for (int k = 0; k < 16; ++k) e[k] = s[k * hw];
#pragma unroll
          for (int k = 0; k < 8; ++k) v[k] = (uint32_t)e[2 * k] | ((uint32_t)e[2 * k + 1] << 16);
        } else {
#pragma unroll
          for (int k = 0; k < 16; ++k)
            if (c0 + k < t.c) v[k >> 1] |= (uint32_t)s[k * hw] << (16 * (k & 1));
        }
      }
    }
    u32x4* __restrict__ o = reinterpret_cast<u32x4*>(dst);
    o[0] = (u32x4){v[0], v[1], v[2], v[3]};
    o[1] = (u32x4){v[4], v[5], v[6], v[7]};
    return;
  } else {
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
}

// The weight gradients of flat tensors sum over whole tiles of positions, so
// those outside the images take part with a gradient of zero; an infinite or
// NaN x (or concat value) beside them makes that product NaN, in the sums of
// taps that meet the value nowhere inside the image.  Masking every fragment
// would cost the vector instructions that bound these kernels, so a workgroup
// whose sums hold a NaN forms them a second time with such positions' products
// replaced by zero: finite inputs pay one vote of a workgroup's waves
// (generator / convolution, us, without -> with: bf16 4x64x135x181 74.0 ->
// 74.0 / 42.5 -> 42.8, fp16 2x128x96x96 31.2 -> 33.1 / 33.5 -> 34.3, fp32
// 4x64x135x181 122.4 -> 123.3 / 100.8 -> 102.3).

// Positions of one row from `pos` (rows start on multiples of 8) that lie
// inside the image, at most 8: none above the last column or row.
__device__ __forceinline__ int flat_inside(const FlatLay& f, int pos) {
  const int row = pos / f.P, n = f.W - (pos - row * f.P);
  return row < f.H && n > 0 ? (n < 8 ? n : 8) : 0;
}

// The first n (from `first` on) of two 2-byte values in a dword, the others zero.
__device__ __forceinline__ uint32_t flat_keep2(uint32_t v, int n, int first) {
  return n >= first + 2 ? v : (n > first ? v & 0xffffu : 0u);
}

// Whether `mine` holds in any lane of the workgroup's NW waves.  votes: NW
// words of LDS that nothing else uses until the call returns.
template <int NW>
__device__ __forceinline__ bool flat_any(bool mine, uint32_t* __restrict__ votes, int wave) {
  const uint32_t any = __builtin_amdgcn_ballot_w64(mine) != 0 ? 1u : 0u;
  if ((threadIdx.x & 63) == 0) votes[wave] = any;
  __syncthreads();
  uint32_t all = 0;
#pragma unroll
  for (int i = 0; i < NW; ++i) all |= votes[i];
  __syncthreads();
  return __builtin_amdgcn_readfirstlane(all) != 0;
}

// Zeroing of the elements of a concat's flat gradient that the input gradient's
// tiles do not cover: the lead, the guard rows after each plane's last tile
// and, for 2-byte elements, the channels past 3C of the last 16-channel block
// and what the buffer holds past the last image.  No kernel reads them, but
// the gradient is a tensor that autograd hands on, and its checks (NaN
// detection, hooks) read all of it.  One item = 16 bytes.
struct FlatGradZero {
  void* base;       // null: nothing to do
  uint32_t n, c;    // images, channels
  uint32_t runs;    // tails per image, in planes: C (or 4C) plane-major ones, then the blocks' 16 each
  uint32_t tail;    // items of one plane's tail
  uint32_t lead;    // items of the lead
  uint32_t spare;   // items per image of the last block's spare channels
  uint32_t end;     // items past the last image
  uint32_t items;   // in all
};

inline FlatGradZero flat_grad_zero(void* grad, const FlatLay& f, int64_t n, int64_t c, int esz) {
  const uint32_t ve = 16 / (uint32_t)esz;  // (lead, S and the tiles are multiples of 8 elements)
  const bool cl = esz == 2;
  FlatGradZero z{grad, (uint32_t)n, (uint32_t)c, 0, 0, 0, 0, 0, 0};
  z.runs = (uint32_t)(cl ? cl_cat_planes(c) : 4 * c);
  z.tail = (f.S - flat_span(f)) / ve;
  z.lead = f.lead / ve;
  z.spare = cl && 3 * c % 16 != 0 ? flat_span(f) : 0;
  z.end = cl ? 15 * f.lead / ve : 0;
  z.items = z.lead + z.end + z.n * (z.runs * z.tail + z.spare);
  return z;
}

template <typename T>
__device__ __forceinline__ void flat_grad_zero_item(const FlatGradZero& z, const FlatLay& f,
                                                    uint32_t i) {
  constexpr uint32_t VE = 16 / (uint32_t)sizeof(T);
  T* __restrict__ base = static_cast<T*>(z.base);
  const uint32_t FS = flat_span(f);
  const size_t img = (size_t)z.runs * f.S;
  size_t o;  // element
  if (i < z.lead) {
    o = (size_t)i * VE;
  } else if ((i -= z.lead) < z.end) {
    o = f.lead + z.n * img + (size_t)i * VE;
  } else {
    i -= z.end;
    const uint32_t per = z.runs * z.tail + z.spare;
    const uint32_t n = i / per, k = i - n * per;
    o = f.lead + n * img;
    if (k < z.runs * z.tail) {
      const uint32_t pl = k / z.tail;
      uint32_t e = k - pl * z.tail;
      if (sizeof(T) == 2 && pl >= z.c) {
        // a block's tail is one run of 16 planes' tails
        const uint32_t blk = (pl - z.c) / 16;
        e += (pl - z.c - 16 * blk) * z.tail;
        o += (size_t)(z.c + 16 * blk) * f.S + (size_t)FS * 16 + (size_t)e * VE;
      } else {
        o += (size_t)pl * f.S + FS + (size_t)e * VE;
      }
    } else {
      o += (size_t)(z.runs - 16) * f.S + (size_t)(k - z.runs * z.tail) * 16 + 8;
    }
  }
  *reinterpret_cast<u32x4*>(base + o) = (u32x4){0u, 0u, 0u, 0u};
}

struct CvPack;
struct YPack;

// Lays out `count` (1 or 2) tensors of `dtype` and the same n, H, W flat in one
// launch, whose first workgroups run a weight packing of the launches that
// follow (optional; ypack: kernel size `ks`) and whose last ones zero the rest
// of the gradient that those write (optional).  Defined in flat.hip.
int flat_copy(const FlatCopy* t, int count, const FlatLay& f, int dtype, hipStream_t stream,
              const CvPack* cpack = nullptr, const YPack* ypack = nullptr, int ks = 0,
              const FlatGradZero* zero = nullptr);

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
  // runs of memory per plane (2-byte elements: per 16-channel block, each
  // position 16 elements)
  constexpr uint32_t EP = sizeof(T) == 2 ? 16 : 1;
  const uint32_t units = (uint32_t)z.planes / EP;
  const int stride = wgs * nthreads, first = wg * nthreads + tid;
  const uint32_t tail = f.S - (uint32_t)(f.H * f.P);  // a multiple of 8
  typedef uint32_t V4 __attribute__((ext_vector_type(4)));
  constexpr int VE = 16 / (int)sizeof(T);
  const V4 zero = {0u, 0u, 0u, 0u};
  // the lead and the tail of every run, 16 bytes at a time
  const uint32_t lv = f.lead * EP / VE, tv = tail * EP / VE;
  for (uint32_t i = first; i < lv; i += stride) reinterpret_cast<V4*>(base)[i] = zero;
  const uint32_t tot = tv * units;
  for (uint32_t i = first; i < tot; i += stride) {
    const uint32_t pl = i / tv, k = i - pl * tv;
    reinterpret_cast<V4*>(base + (f.lead + (size_t)pl * f.S + (size_t)f.H * f.P) * EP)[k] = zero;
  }
  // the pad columns of every row
  const uint32_t pad = (uint32_t)(f.P - f.W), rows = units * (uint32_t)f.H;
  for (uint32_t i = first; i < rows; i += stride) {
    const uint32_t pl = i / (uint32_t)f.H, h = i - pl * (uint32_t)f.H;
    T* __restrict__ d = base + (f.lead + (size_t)pl * f.S + (size_t)h * f.P + f.W) * EP;
    if constexpr (EP == 16) {
      for (uint32_t e = 0; e < 2 * pad; ++e) reinterpret_cast<V4*>(d)[e] = zero;
    } else {
      for (uint32_t e = 0; e < pad; ++e) d[e] = (T)0.f;
    }
  }
}

}  // namespace ddpm
