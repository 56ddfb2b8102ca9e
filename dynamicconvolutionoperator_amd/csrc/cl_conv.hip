// Channels-last implicit GEMMs over channels (2-byte types): the 3x3 fuse
// convolution's forward and input gradient, and dY of the fused generator.
//
//   conv: out[m, p] = bias[m] + sum_{k, t} A[m][k][t] * in[k, p + off(t)]
//   dY:   dY[i, p]  = sum_{b, c, t} W[(b,c,t), i] * gO_b[c, p] * x[c, p + off(b, t)]
//
// What bounds the plane-major kernels of these products is LDS instructions
// and, with every wave waiting at one barrier per stage, that LDS reads and
// MFMAs do not overlap (without the stage copies the 256x256 bf16 forward runs
// at 30 of its 40 us, without the MFMA loop at 26).  Here
//   * a workgroup owns 256 positions x 16 * MB output planes; its stages are
//     (64 input channels, kernel row), 8 waves = 4 position groups of 64 x 2
//     halves of the 64 channels: an A fragment read from LDS serves four
//     16-position blocks instead of two, so a stage takes 24 16-byte reads
//     per 48 MFMAs and wave (40 for the plane-major kernel), with two waves
//     per SIMD as before; the halves' sums are added through LDS at the end;
//   * a B fragment is one 16-byte read at any shift (cl.h), free of bank
//     conflicts: the 64 lanes cover two runs of 512 bytes;
//   * dY's gradient values sit in registers for the stages of a branch.

#include "cl_conv.h"

#include <type_traits>

namespace ddpm {

constexpr int kClcThreads = 512;

// What the two groups of four waves (half 0, 1) take of a stage:
enum ClMode : int {
  kClSplitK = 0,  // a stage is (64 input channels, kernel row): half the channels each, sums
                  // added at the end (one group of output planes per workgroup)
  kClGrad = 1,    // the same for dY
  kClSplitM = 2,  // a stage is (32 input channels, kernel row): a group of output planes each;
                  // the workgroup runs its pairs of groups one after another
};

// LDS: kXR windows of a stage in a ring, copied two stages ahead (their
// latency, not their bytes, is what a stage would wait for: 1.6 us per stage
// of the 256x256 bf16 forward with one stage ahead and no compute), and the A
// slices one stage ahead.
template <int KS, int MB, int MODE>
struct ClcLds {
  static constexpr int kXB = MODE == kClSplitM ? 2 : 4;  // 16-channel blocks of a stage
  static constexpr int kXR = MODE == kClSplitM ? 6 : 3;
  static constexpr int kX = kXB * kClUnits * 16;         // bytes: a stage's windows
  static constexpr int kA1 = KS * MB * 1024;             // bytes: one chunk's (or group's) taps
  static constexpr int kAOff = kXR * kX;
  static constexpr int kRP = kFlatTile + 4;              // the halves' sums: floats of a plane
  static constexpr int kRed = MODE == kClSplitM ? 0 : 2 * 16 * MB * kRP * 4;
  static constexpr int kBytes = kAOff + 4 * kA1 > kRed ? kAOff + 4 * kA1 : kRed;
  static_assert(kBytes <= 160 * 1024, "LDS of a CU");
};

// End of a stage: this wave's copies for the next stage have landed (the
// newest `ahead` vector memory operations may still be in flight), its LDS
// reads are done, and all waves are here.
template <bool AHEAD>
__device__ __forceinline__ void clc_barrier() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(AHEAD ? 0x72 : 0x70);  // vmcnt(2 or 0) expcnt(7) lgkmcnt(0)
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

template <typename T, int KS, int MB, int MODE>
__global__ __launch_bounds__(kClcThreads) __attribute__((amdgpu_waves_per_eu(2))) void cl_conv_kernel(
    const T* __restrict__ in, const T* __restrict__ gout, const uint32_t* __restrict__ pk,
    const T* __restrict__ bias, T* __restrict__ out, float* __restrict__ part, ClConvGeom g,
    CwReduce cred, WReduce wred) {
  typedef Mma<T> M;
  typedef typename M::V V;
  typedef ClcLds<KS, MB, MODE> L;
  constexpr bool GRAD = MODE == kClGrad, SM = MODE == kClSplitM;
  constexpr int r = KS / 2;
  extern __shared__ __attribute__((aligned(16))) char clsm[];

  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int mpairs = SM ? g.pairs : 1;
  const int mgw = SM ? (g.mgroups + 1) / 2 / g.pairs : g.mgroups;  // workgroups per (tile, split)
  const int mg0 = SM ? 2 * mpairs * (bid % mgw) : bid % mgw;      // first m group
  const int rest = bid / mgw;
  const int ksplit = rest % g.ks;
  const int tile = rest / g.ks;
  const int n = tile / g.f.ft;
  const int p0 = (tile - n * g.f.ft) * kFlatTile;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int col16 = lane & 15, quad = lane >> 4;
  const int half = wave >> 2, pw = 64 * (wave & 3);  // wave group, first position of the wave
  const int g0 = ksplit * g.gs_per;
  const int gend = SM ? g.nc32 : g.gs;
  const int g1 = SM ? gend : (g0 + g.gs_per < gend ? g0 + g.gs_per : gend);
  const int ng = g1 > g0 ? g1 - g0 : 0;
  const int nst1 = (SM ? 1 : g.nb) * ng * KS;  // stages of one (pair of) group(s) of output planes:
  // (branch, channels, kernel row)
  const int nstage = nst1 * mpairs;
  const bool resident = SM && nst1 <= L::kXR;  // every window stays in its ring slot
  const int nx = resident ? nst1 : nstage;     // window stages to copy

  const BufRes xres = make_buf(in + (int64_t)n * g.in_img,
                               (uint32_t)((g.f.lead + (uint32_t)g.q * g.f.S) * 32u));
  // copies of a stage's windows: unit U = 64 * copy + lane is the 16-byte half
  // U & 1 of position row (U / 2) % kClWin of block U / kClUnits
  constexpr int NX = L::kXB * kClUnits / 64, NXJ = (NX + 7) / 8;
  uint32_t xof[NXJ];
#pragma unroll
  for (int j = 0; j < NXJ; ++j) {
    const int u = 64 * (wave + 8 * j) + lane;
    const int blk = u / kClUnits, px = (u - blk * kClUnits) >> 1;
    xof[j] = ((uint32_t)blk * g.f.S + (uint32_t)px) * 32u + (uint32_t)(u & 1) * 16u;
  }
  // Position of a stage, stepped rather than divided out of the stage number
  // (a scalar division by a runtime count costs a stage some 200 clocks):
  // kernel row, channel group, branch (split M: pair of groups), ring slot.
  struct Pos {
    int ki, gi, b, slot, par;
  };
  auto step = [&](Pos& p) {
    if (++p.ki == KS) {
      p.ki = 0;
      if (++p.gi == g1) {
        p.gi = g0;
        ++p.b;
        if (resident) p.slot = -1;
      }
    }
    if (++p.slot == L::kXR) p.slot = 0;
    p.par ^= 1;
  };
  // a stage's windows -> its ring slot (at least two copies per wave)
  auto stage_x = [&](const Pos& p) {
    const int d = SM ? 1 : dil_of(p.b, g.d0, g.d1, g.d2);
    char* __restrict__ dst = clsm + p.slot * L::kX;
    const uint32_t so = ((uint32_t)(L::kXB * p.gi) * g.f.S +
                         (uint32_t)((int)g.f.lead - kClPad + p0 + (p.ki - r) * d * g.f.P)) * 32u;
#pragma unroll
    for (int j = 0; j < NXJ; ++j) {
      const int cp = wave + 8 * j;
      if (NX % 8 != 0 && cp >= NX) break;
      const uint32_t vo = xof[j];
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          xres, (__attribute__((address_space(3))) void*)(dst + 1024 * cp), 16, vo, so, 0, 0);
    }
  };
  static_assert(NX / 8 >= 2, "the stage barrier leaves two copies in flight");
  // a stage's A slices (both halves') -> its buffer of the two
  auto stage_a = [&](const Pos& p) {
    char* __restrict__ dst = clsm + L::kAOff + p.par * 2 * L::kA1;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int cc = SM ? p.gi : 2 * p.gi + c;
      const int mg = SM ? mg0 + 2 * p.b + c : mg0;
      if (cc >= g.nc32 || mg >= g.mgroups) break;
      const uint32_t* src =
          pk + (((GRAD ? mg * 3 + p.b : mg) * g.nc32 + cc) * KS * KS + p.ki * KS) * (MB * 256);
      const BufRes pres = make_buf(src, (uint32_t)L::kA1);
#pragma unroll
      for (int j = 0; j < (KS * MB + 7) / 8; ++j) {
        const int u = wave + 8 * j;
        if ((KS * MB) % 8 == 0 || u < KS * MB)
          __builtin_amdgcn_raw_ptr_buffer_load_lds(
              pres, (__attribute__((address_space(3))) void*)(dst + c * L::kA1 + 1024 * u), 16,
              (uint32_t)(u * 64 + lane) * 16u, 0, 0, 0);
      }
    }
  };

  // dY: the branch gradient of this lane's 8 channels at its four positions
  constexpr int NB4 = 4;
  ClProd<T> gp[GRAD ? NB4 : 1];
  u32x4 gn[GRAD ? NB4 : 1];
  auto load_g = [&](const Pos& p) {
    if constexpr (GRAD) {
      const int gi = p.gi, b = p.b;
      const int c8 = 8 * gi + 4 * half + quad;  // 8-channel group within the branch
      const int j8 = b * (g.C / 8) + c8;        // and within the gradient's channels-last planes
      const BufRes gres = make_buf(gout + (int64_t)n * g.out_img + (int64_t)g.C * g.f.S,
                                   (uint32_t)((g.f.lead + (uint32_t)((3 * g.C + 15) / 16) * g.f.S * 16u) * 2u));
      // (the lead of the plane-major part is counted in elements)
#pragma unroll
      for (int blk = 0; blk < NB4; ++blk) {
        const uint32_t pos = (uint32_t)(p0 + pw + 16 * blk + col16);
        const uint32_t vo = 8 * c8 < g.C
                                ? (g.f.lead + ((uint32_t)(j8 >> 1) * g.f.S + pos) * 16u + (uint32_t)(j8 & 1) * 8u) * 2u
                                : kOob;
        gn[blk] = __builtin_amdgcn_raw_buffer_load_b128(gres, vo, 0, 0);
      }
    }
  };

  f32x4 acc[NB4][MB];
#pragma unroll
  for (int blk = 0; blk < NB4; ++blk)
#pragma unroll
    for (int ib = 0; ib < MB; ++ib) acc[blk][ib] = f32x4{0.f, 0.f, 0.f, 0.f};

  Pos pc{0, g0, 0, 0, 0}, pn = pc, px2 = pc;  // this stage, the next one, the one after
  if (nstage > 0) {
    stage_x(px2);
    load_g(pc);
    stage_a(pc);
    step(px2);
    if (1 < nx) stage_x(px2);
    step(px2);
    step(pn);
  }
  // a split reduction of the weight gradient that ran before this launch
  if (cred.items > 0) cw_reduce_share<T>(cred, (int)blockIdx.x, (int)gridDim.x, tid, kClcThreads);
  if constexpr (GRAD) {
    if (wred.items > 0) {
      const int per = (wred.items + (int)gridDim.x - 1) / (int)gridDim.x;
      for (int j = tid; j < per; j += kClcThreads) {
        const uint32_t item = (uint32_t)((int)blockIdx.x * per + j);
        if (wred.v4)
          wg_reduce_item<T, 4>(wred.pw, wred.pb, (T*)wred.dw, (T*)wred.db, wred.C, wred.KK,
                               wred.splits, item);
        else
          wg_reduce_item<T, 1>(wred.pw, wred.pb, (T*)wred.dw, (T*)wred.db, wred.C, wred.KK,
                               wred.splits, item);
      }
    }
  }
  __builtin_amdgcn_s_waitcnt(0);
  __syncthreads();

  // One block of 16 positions and 16 output planes from m, straight from the
  // accumulators (input planes unsplit: the pairs of m groups, and the concat
  // gradient).  Whether a block's position lies inside the image (flat outputs
  // hold zero elsewhere):
  bool inside[NB4];
#pragma unroll
  for (int blk = 0; blk < NB4; ++blk) {
    const int pos = p0 + pw + 16 * blk + col16, row = pos / g.f.P;
    inside[blk] = row < g.H && pos - row * g.f.P < g.W;
  }
  auto store = [&](f32x4 v, int m, int blk) {
    const int pos = p0 + pw + 16 * blk + col16;
    if (m >= g.M) return;
    if (g.out == kClOutImage) {
      if (!inside[blk]) return;
      const int row = pos / g.f.P, col = pos - row * g.f.P;
      const size_t hw = (size_t)g.H * g.W;
      T* __restrict__ po = out + ((size_t)n * g.M + m) * hw + (size_t)row * g.W + col;
      float bv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) bv[e] = bias && m + e < g.M ? to_f(bias[m + e]) : 0.f;
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (m + e < g.M) po[e * hw] = from_f<T>(v[e] + bv[e]);
      return;
    }
    // (M = 4C is a multiple of 4)
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = inside[blk] ? v[e] : 0.f;
    T* __restrict__ po = out + (int64_t)n * g.out_img + g.f.lead;
    if (m < g.C) {
#pragma unroll
      for (int e = 0; e < 4; ++e) po[(size_t)(m + e) * g.f.S + pos] = from_f<T>(v[e]);
    } else {
      const int j = m - g.C;
      typedef T T4 __attribute__((ext_vector_type(4)));
      *reinterpret_cast<T4*>(po + (size_t)g.C * g.f.S + ((size_t)(j >> 4) * g.f.S + pos) * 16 + (j & 15)) =
          (T4){from_f<T>(v[0]), from_f<T>(v[1]), from_f<T>(v[2]), from_f<T>(v[3])};
    }
  };
  // the same for a concat gradient of whole 16-channel blocks (C % 16 == 0):
  // lane offsets formed once, the block's in the stores' scalar offset
  const BufRes ores = make_buf(out + (int64_t)n * g.out_img + g.f.lead, (uint32_t)g.out_img * 2u);
  const uint32_t opos = (uint32_t)(p0 + pw + col16);
  const uint32_t ovx = (4u * quad * g.f.S + opos) * 2u, ovc = opos * 32u + 8u * quad;
  auto store_grad = [&](f32x4 v, int mb16, int blk) {  // planes 16 * mb16 ..
#pragma unroll
    for (int e = 0; e < 4; ++e) v[e] = inside[blk] ? v[e] : 0.f;
    const uint32_t d0 = pack2<T>(v[0], v[1]), d1 = pack2<T>(v[2], v[3]);
    if (16 * mb16 < g.C) {
      const uint32_t so = 16u * (uint32_t)mb16 * g.f.S * 2u, vo = ovx + 32u * blk;
      const uint32_t s1 = so + g.f.S * 2u, s2 = s1 + g.f.S * 2u, s3 = s2 + g.f.S * 2u;
      __builtin_amdgcn_raw_buffer_store_b16((unsigned short)d0, ores, vo, so, 0);
      __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(d0 >> 16), ores, vo, s1, 0);
      __builtin_amdgcn_raw_buffer_store_b16((unsigned short)d1, ores, vo, s2, 0);
      __builtin_amdgcn_raw_buffer_store_b16((unsigned short)(d1 >> 16), ores, vo, s3, 0);
    } else {
      typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
      const uint32_t so = ((uint32_t)g.C * g.f.S + (16u * mb16 - (uint32_t)g.C) * g.f.S) * 2u;
      const uint32_t vo = ovc + 512u * blk;
      __builtin_amdgcn_raw_buffer_store_b64((u32x2){d0, d1}, ores, vo, so, 0);
    }
  };
  const bool grad16 = g.out == kClOutGrad && g.C % 16 == 0;
  // sums of 8 positions of plane m into the image (cols: of one row, P % 8 == 0)
  auto store8 = [&](const float (&v)[8], int m, int pos) {
    const int row = pos / g.f.P, col = pos - row * g.f.P;
    if (m >= g.M || row >= g.H || col >= g.W) return;
    T* __restrict__ po = out + (((size_t)n * g.M + m) * g.H + row) * g.W + col;
    typedef T T8 __attribute__((ext_vector_type(8)));
    T8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = from_f<T>(v[e]);
    if (col + 8 <= g.W) {
      __builtin_memcpy(po, &o, sizeof(o));
    } else {
#pragma unroll
      for (int e = 0; e < 8; ++e)
        if (col + e < g.W) po[e] = o[e];
    }
  };

  for (int s = 0; s < nstage; ++s) {
    const int gi = pc.gi;
    const int d = SM ? 1 : dil_of(pc.b, g.d0, g.d1, g.d2);
    if constexpr (GRAD) {
      if (pc.ki == 0) {
        // (opaque: the values are not unpacked, nor waited for, in the stage
        // that loads them)
#pragma unroll
        for (int blk = 0; blk < NB4; ++blk) {
          asm volatile("" : "+v"(gn[blk]));
          gp[blk].set(gn[blk]);
        }
      }
      if (pc.ki == KS - 1 && s + 1 < nstage) load_g(pn);
    }
    const bool ahead = s + 2 < nx;
    // the next copies are issued while the first fragments are on their way
    auto copies = [&]() {
      if (s + 1 < nstage) stage_a(pn);
      if (ahead) stage_x(px2);
    };
    // wave-uniform: an odd chunk count leaves the last stage's second half
    // empty, an odd group count the last pair's
    if (SM ? mg0 + 2 * pc.b + half < g.mgroups : 2 * gi + half < g.nc32) {
      const char* __restrict__ xb =
          clsm + pc.slot * L::kX + ((SM ? 0 : 2 * half) + (quad >> 1)) * kClUnits * 16;
      const char* __restrict__ ab = clsm + L::kAOff + (pc.par * 2 + half) * L::kA1 + lane * 16;
      // tap kj + 1's fragments are read while tap kj's MFMAs run (scheduling
      // groups: one LDS read after every second MFMA)
      V afr[2][MB];
      u32x4 bv[2][NB4];
      auto frags = [&](int kj, int o) {
        const int px = kClPad + pw + col16 + (kj - r) * d;
        const char* __restrict__ xp = xb + px * 32 + (quad & 1) * 16;
#pragma unroll
        for (int ib = 0; ib < MB; ++ib)
          afr[o][ib] = __builtin_bit_cast(V, *reinterpret_cast<const u32x4*>(ab + (kj * MB + ib) * 1024));
#pragma unroll
        for (int blk = 0; blk < NB4; ++blk) bv[o][blk] = *reinterpret_cast<const u32x4*>(xp + 512 * blk);
      };
      frags(0, 0);
      copies();
#pragma unroll
      for (int kj = 0; kj < KS; ++kj) {
        const int o = kj & 1;
        if (kj + 1 < KS) frags(kj + 1, o ^ 1);
#pragma unroll
        for (int blk = 0; blk < NB4; ++blk) {
          u32x4 pv = bv[o][blk];
          if constexpr (GRAD) pv = gp[blk].mul(pv);
          const V bfr = __builtin_bit_cast(V, pv);
#pragma unroll
          for (int ib = 0; ib < MB; ++ib) acc[blk][ib] = M::mac1(afr[o][ib], bfr, acc[blk][ib]);
        }
        if (kj + 1 < KS) {
#pragma unroll
          for (int i = 0; i < MB + NB4; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);                           // LDS read
            if constexpr (GRAD) __builtin_amdgcn_sched_group_barrier(0x002, 10, 0);      // VALU
            __builtin_amdgcn_sched_group_barrier(0x008, MB * NB4 / (MB + NB4), 0);       // MFMA
          }
        }
      }
    } else {
      copies();
    }
    if (ahead)
      clc_barrier<true>();
    else
      clc_barrier<false>();
    const int mpair = pc.b;
    const bool last = SM && pn.b != pc.b;
    pc = pn;
    step(pn);
    step(px2);
    if (last) {
      // the pair's last stage: its sums out, the accumulators cleared
      const int mg = mg0 + 2 * mpair + half;
      if (mg < g.mgroups) {
#pragma unroll
        for (int blk = 0; blk < NB4; ++blk)
#pragma unroll
          for (int ib = 0; ib < MB; ++ib) {
            if (grad16)
              store_grad(acc[blk][ib], mg * MB + ib, blk);
            else
              store(acc[blk][ib], (mg * MB + ib) * 16 + 4 * quad, blk);
            acc[blk][ib] = f32x4{0.f, 0.f, 0.f, 0.f};
          }
      }
    }
  }

  if constexpr (!SM) {
    if (!GRAD && g.out == kClOutGrad) {
      // both halves' sums to the wave that keeps the block
      f32x4* __restrict__ red = reinterpret_cast<f32x4*>(clsm);
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int ib = 0; ib < MB; ++ib)
          red[((wave * 2 + k) * MB + ib) * 64 + lane] = half ? acc[k][ib] : acc[2 + k][ib];
      __syncthreads();
#pragma unroll
      for (int k = 0; k < 2; ++k)
#pragma unroll
        for (int ib = 0; ib < MB; ++ib) {
          const f32x4 o = red[(((wave ^ 4) * 2 + k) * MB + ib) * 64 + lane];
          const int m = (mg0 * MB + ib) * 16 + 4 * quad;
          if (half)
            store(acc[2 + k][ib] + o, m, 2 + k);
          else
            store(acc[k][ib] + o, m, k);
        }
      return;
    }
    // ---- both halves' sums as fp32 planes [half][16 * MB][kRP] in LDS, added
    //      and stored 8 positions of a plane per thread: a wave writes whole
    //      512-byte runs of rows (16 positions x 4 planes per instruction from
    //      the accumulators, and a bias load between the stores of each plane,
    //      took 16 of the kernel's 67 thousand clocks)
    constexpr int RP = L::kRP;
    float* __restrict__ red = reinterpret_cast<float*>(clsm);
#pragma unroll
    for (int blk = 0; blk < NB4; ++blk)
#pragma unroll
      for (int ib = 0; ib < MB; ++ib)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          red[(half * 16 * MB + ib * 16 + 4 * quad + e) * RP + pw + 16 * blk + col16] = acc[blk][ib][e];
    __syncthreads();
#pragma unroll 1
    for (int j = 0; j < MB; ++j) {
      const int task = tid + kClcThreads * j;  // plane task / 32, positions 8 * (task % 32) ..
      const int ml = task >> 5, q8 = 8 * (task & 31);
      const int m = mg0 * MB * 16 + ml;
      const f32x4* __restrict__ ra = reinterpret_cast<const f32x4*>(red + ml * RP + q8);
      const f32x4* __restrict__ rb = reinterpret_cast<const f32x4*>(red + (16 * MB + ml) * RP + q8);
      const f32x4 lo = ra[0] + rb[0], hi = ra[1] + rb[1];
      if (!GRAD && g.ks > 1) {
        if (m >= g.M) continue;
        const uint32_t FS = flat_span(g.f);
        float* __restrict__ po = part + (((size_t)ksplit * g.N + n) * g.M + m) * FS + p0 + q8;
        reinterpret_cast<f32x4*>(po)[0] = lo;
        reinterpret_cast<f32x4*>(po)[1] = hi;
        continue;
      }
      const float bv = bias && m < g.M ? to_f(bias[m]) : 0.f;
      const float v[8] = {lo[0] + bv, lo[1] + bv, lo[2] + bv, lo[3] + bv,
                          hi[0] + bv, hi[1] + bv, hi[2] + bv, hi[3] + bv};
      store8(v, m, p0 + q8);
    }
  }
}

int cl_conv_launch(int dtype, int mode, int ksize, int mb, const ClConvGeom& g, const void* in,
                   const void* gout, const void* pk, const void* bias, void* out, float* part,
                   const CwReduce& cred, const WReduce& wred, hipStream_t stream) {
  const bool split_m = mode == 0 && g.pairs > 0;
  auto go = [&](auto tag, auto ksc, auto mbc, auto modec) {
    using T = decltype(tag);
    constexpr int KS = decltype(ksc)::value, MB = decltype(mbc)::value;
    constexpr int MODE = decltype(modec)::value;
    typedef ClcLds<KS, MB, MODE> L;
    auto kern = cl_conv_kernel<T, KS, MB, MODE>;
    const int ae = allow_dynamic_lds(reinterpret_cast<const void*>(kern), L::kBytes);
    if (ae != 0) return ae;
    const int64_t wgs = (int64_t)g.N * g.f.ft * (MODE == kClSplitM ? (g.mgroups + 1) / 2 / g.pairs : g.mgroups) * g.ks;
    if (wgs > 0x7fffffffLL) return (int)kUnsupported;
    hipLaunchKernelGGL(kern, dim3((unsigned)wgs), dim3(kClcThreads), L::kBytes, stream, (const T*)in,
                       (const T*)gout, (const uint32_t*)pk, (const T*)bias, (T*)out, part, g, cred,
                       wred);
    return (int)hipGetLastError();
  };
  auto by_mb = [&](auto tag) {
    auto pick = [&](auto mbc) {
      typedef std::integral_constant<int, 3> K3;
      if (split_m) return go(tag, K3(), mbc, std::integral_constant<int, kClSplitM>());
      if (mode == 0) return go(tag, K3(), mbc, std::integral_constant<int, kClSplitK>());
      if (ksize == 1)
        return go(tag, std::integral_constant<int, 1>(), mbc, std::integral_constant<int, kClGrad>());
      return go(tag, K3(), mbc, std::integral_constant<int, kClGrad>());
    };
    if (mb == 1) return pick(std::integral_constant<int, 1>());
    if (mb == 2) return pick(std::integral_constant<int, 2>());
    if (mb == 4) return pick(std::integral_constant<int, 4>());
    return (int)kUnsupported;
  };
  if (dtype == kBF16) return by_mb(bf16());
  if (dtype == kF16) return by_mb(f16());
  return kBadArgument;
}

}  // namespace ddpm
