// Flat copies of NCHW tensors: rows padded with zeros to a 16-byte pitch,
// zero guard rows between planes (FlatLay, ddpm_common.h).
//
// A streaming pass (each source element read once, each destination element
// written once): it buys the staged kernels 16-byte LDS-direct copies, which
// an image whose rows are not whole 16-byte chunks would otherwise stage
// element by element through registers (bf16 2x64x135x181: x and y together
// 7.6 us, against 250 -> 39 us of the generator's weight gradient and 161 -> 29
// us of dY).

#include "flat.h"

#include "gen_bwd.h"

namespace ddpm {

// Workgroups: the packings' units (their few strided loads are the launch's
// longest chain, so they start first), then the chunks of each tensor, then the
// gradient's zeros.
template <typename T>
__global__ __launch_bounds__(256) void flat_copy_kernel(FlatCopy a, FlatCopy b, FlatLay f,
                                                        CvPack cp, YPack yp, int ks,
                                                        FlatGradZero z) {
  uint32_t blk = blockIdx.x;
  const uint32_t pb = (uint32_t)(cp.total + yp.total + 255) / 256, ab = (a.chunks + 255) / 256;
  const uint32_t bb = (b.chunks + 255) / 256;
  if (blk < pb) {
    const int idx = (int)(blk * 256u + threadIdx.x);
    if (idx < cp.total)
      cv_pack_any<T>(cp, idx);
    else if (idx < cp.total + yp.total && ks == 1)
      yt_pack_any<T, 1>(yp, idx - cp.total);
    else if (idx < cp.total + yp.total)
      yt_pack_any<T, 3>(yp, idx - cp.total);
    return;
  }
  blk -= pb;
  if (blk < ab) {
    const uint32_t idx = blk * 256u + threadIdx.x;
    if (idx < a.chunks) flat_copy_chunk<T>(a, f, idx);
  } else if (blk - ab < bb) {
    const uint32_t idx = (blk - ab) * 256u + threadIdx.x;
    if (idx < b.chunks) flat_copy_chunk<T>(b, f, idx);
  } else {
    const uint32_t idx = (blk - ab - bb) * 256u + threadIdx.x;
    if (idx < z.items) flat_grad_zero_item<T>(z, f, idx);
  }
}

int flat_copy(const FlatCopy* t, int count, const FlatLay& f, int dtype, hipStream_t stream,
              const CvPack* cpack, const YPack* ypack, int ks, const FlatGradZero* zero) {
  const FlatCopy none{nullptr, nullptr, 0, 0, 0};
  const FlatGradZero z = zero ? *zero : FlatGradZero{nullptr, 0, 0, 0, 0, 0, 0, 0, 0};
  const FlatCopy &a = t[0], &b = count > 1 ? t[1] : none;
  const CvPack cp = cpack ? *cpack : CvPack{nullptr, nullptr, ConvGeom{}, 0, 0, 0, 0};
  const YPack yp = ypack ? *ypack : YPack{nullptr, nullptr, 0, 0, 0};
  const uint64_t blocks = ((uint64_t)a.chunks + 255) / 256 + ((uint64_t)b.chunks + 255) / 256 +
                          (uint64_t)(cp.total + yp.total + 255) / 256 + ((uint64_t)z.items + 255) / 256;
  if (blocks > 0x7fffffffu) return kUnsupported;
  const dim3 grid((unsigned)blocks);
  switch (dtype) {
    case kF32:
      hipLaunchKernelGGL(flat_copy_kernel<float>, grid, dim3(256), 0, stream, a, b, f, cp, yp, ks,
                         z);
      break;
    case kBF16:
      hipLaunchKernelGGL(flat_copy_kernel<bf16>, grid, dim3(256), 0, stream, a, b, f, cp, yp, ks,
                         z);
      break;
    case kF16:
      hipLaunchKernelGGL(flat_copy_kernel<f16>, grid, dim3(256), 0, stream, a, b, f, cp, yp, ks,
                         z);
      break;
    default:
      return kBadArgument;
  }
  return (int)hipGetLastError();
}

}  // namespace ddpm
