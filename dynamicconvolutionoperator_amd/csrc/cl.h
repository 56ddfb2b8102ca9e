// Channels-last flat tensors of 2-byte types (bf16, f16): the form in which
// the flat kernels of those types hold the concat, its gradient and their
// copies of x, y and grad_out.
//
// The planes of a flat tensor (FlatLay, ddpm_common.h) are grouped by 16:
// element (plane c, position p) of an image is
//
//   (lead + (c / 16) * S + p) * 16 + c % 16
//
// so a position's 16 channels are 32 bytes.  What that buys the kernels:
//   * an MFMA operand whose K slots are channels (the convolution, dY) is one
//     16-byte LDS read per lane, one whose K slots are positions (the weight
//     gradients) two transposing 8-byte reads, against eight 2-byte reads or
//     five dwords and a realignment from planes;
//   * a tap's shift is a whole number of 32-byte rows, so every shifted
//     window is as aligned as the unshifted one;
//   * a staged window is one run of memory.
#pragma once

#include "flat.h"

namespace ddpm {

constexpr int kClPad = 8;                             // positions staged on either side of a tile
constexpr int kClWin = kFlatTile + 2 * kClPad;        // positions of a staged window
constexpr int kClUnits = 2 * kClWin;                  // its 16-byte units per 16-channel block

// Raw bits of four 2-byte elements per lane, transposed within 16-lane groups:
// lane 16g + 4a + b receives element b of the 8-byte reads of lanes 16g + a +
// 4e, e = 0..3.
__device__ __forceinline__ void cl_read_tr(const char* p, uint32_t& d0, uint32_t& d1) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
  const s16x4 t =
      __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) s16x4*)p);
  const u32x2 d = __builtin_bit_cast(u32x2, t);
  d0 = d[0];
  d1 = d[1];
}

// Products of 8 pairs of 2-byte values (dwords of two), rounded to T: the
// exact product rounded once (f16: one packed multiply rounds the same way).
template <typename T>
struct ClProd;
template <>
struct ClProd<bf16> {
  float g[8];
  __device__ __forceinline__ void set(const u32x4& v) {
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      g[2 * k] = __uint_as_float(v[k] << 16);
      g[2 * k + 1] = __uint_as_float(v[k] & 0xffff0000u);
    }
  }
  __device__ __forceinline__ u32x4 mul(const u32x4& v) const {
    u32x4 o;
#pragma unroll
    for (int k = 0; k < 4; ++k)
      o[k] = pack_bf16x2(g[2 * k] * __uint_as_float(v[k] << 16),
                         g[2 * k + 1] * __uint_as_float(v[k] & 0xffff0000u));
    return o;
  }
};
template <>
struct ClProd<f16> {
  u32x4 g;
  __device__ __forceinline__ void set(const u32x4& v) { g = v; }
  // (element by element: the product of two f16 values is exact in fp32)
  __device__ __forceinline__ u32x4 mul(const u32x4& v) const {
    return __builtin_bit_cast(u32x4, __builtin_bit_cast(f16x8, g) * __builtin_bit_cast(f16x8, v));
  }
};

}  // namespace ddpm
