// The channels-last kernels that contract over channels: the fuse
// convolution's forward and input gradient, and the generator's dY.
#pragma once

#include "cl.h"
#include "gen_bwd.h"

namespace ddpm {

struct ClConvGeom {
  int N, M, H, W;   // images, output planes, image size
  FlatLay f;
  int q;            // 16-channel blocks per image of the input
  int64_t in_img;   // elements from one image of the input to the next
  int nc32;         // 32-channel chunks contracted (per branch)
  int nb;           // branches (dY: 3)
  int d0, d1, d2;   // their dilations (the convolution: 1)
  int mgroups;      // groups of 16 * MB output planes
  int gs;           // groups of 64 input channels, ceil(nc32 / 2)
  int ks, gs_per;   // splits of those groups, groups per split (1, gs for dY)
  int pairs;        // > 0: the workgroup runs so many pairs of m groups (a group per half of its
                    // waves, pairs per workgroup dividing their number), ks = 1
  int out;          // kClOutImage, kClOutGrad
  int C;            // kClOutGrad: planes of the first (plane-major) block; dY: channels
  int64_t out_img;  // elements from one image of the output to the next
};

enum ClOut : int {
  kClOutImage = 0,  // [N][M][H][W]
  kClOutGrad = 1,   // a concat gradient: its C x-planes flat, then 3C planes channels-last
};

// Launches the kernel for `dtype` (kBF16, kF16): mode 0 the convolution, 1 dY
// with kernel size ks.  in: the concat / grad_out (mode 0) or x (mode 1),
// channels-last; gout: the concat's gradient (mode 1); pk: the packed A
// operand of MB-block m groups; part: fp32 partials where g.ks > 1.
int cl_conv_launch(int dtype, int mode, int ksize, int mb, const ClConvGeom& g, const void* in,
                   const void* gout, const void* pk, const void* bias, void* out, float* part,
                   const CwReduce& cred, const WReduce& wred, hipStream_t stream);

}  // namespace ddpm
