// The channels-last weight gradients: of the fused generator (dW, db) and of
// the fuse convolution.
#pragma once

#include "cl.h"
#include "gen_bwd.h"

namespace ddpm {

struct ClWGeom {
  int N, C;             // images, channels
  FlatLay f;
  int d0, d1, d2;       // generator: the branches' dilations
  int q;                // generator: 16-channel blocks per image of x; convolution: of the concat
  int64_t x_img;        // elements from one image of x (concat) to the next
  int yq;               // 16-channel blocks per image of y (grad_out)
  int64_t y_img;
  int64_t g_img;        // elements per image of the concat's gradient (generator)
  int blocks;           // generator: 3 * ceil(C / 16) (branch, 16 channels); convolution: 4C / 16
  int halves;           // halves of 64 of the y channels (1 up to 64)
  int splits, steps, steps_per_split;  // steps of 256 positions, N * f.ft in all
  int direct;           // one split: the gradients are written directly
  int dw_blocks;        // workgroups of the weight gradient; any further ones are helpers
};

// Split geometry (at most 16 splits of at least 2 steps each) and bytes of
// the fp32 partials.
void clw_geom(ClWGeom& g, const FlatLay& f, int64_t n, int64_t c, bool generator);
int64_t clw_partial_bytes(const ClWGeom& g, int kk, bool generator);

// Launches the generator's weight gradient (helpers beyond g.dw_blocks run
// `fin`) or the convolution's.
int clw_launch_gen(int dtype, int ksize, const ClWGeom& g, const void* x, const void* y,
                   const void* gout, float* pw, float* pb, void* dw, void* db, int helpers,
                   const BxFinish& fin, hipStream_t stream);
int clw_launch_conv(int dtype, const ClWGeom& g, const void* cat, const void* gout, float* pw,
                    float* pb, void* dw, void* db, hipStream_t stream);

}  // namespace ddpm
