// Channels-last weight gradients (2-byte types), contractions over positions:
//
//   generator:   dW[(b,c,t), i] = sum_p gO_b[c, p] * x[c, p + off(b,t)] * y[i, p],  db = sum_p dK
//   convolution: dW[co, ci, t]  = sum_p cat[ci, p + off(t)] * gO[co, p],            db = sum_p gO
//
// M = 16 c (ci) of a block, N = the y (grad_out) channels, K = positions.  A
// workgroup owns (split, block [, half of 64 N channels]); a step is 256
// positions, staged one step ahead into a second LDS buffer; 12 waves = 4
// position segments x 3 kernel rows, as in the plane-major kernels
// (gen_bwd_w.hip, conv_wgrad.hip), which at 256x256 spend 34 of 39 us on
// their compute (bf16 dW without the stage copies): 4-5 dword LDS reads and a
// realignment per shifted fragment.  Here every fragment is two transposing
// 8-byte reads of 32-byte position rows, whatever its shift.  MFMA slot 8q + 4h
// + e of a 32-position segment is position 16h + 4q + e for both operands.

#include "cl_wgrad.h"

#include <type_traits>

namespace ddpm {

constexpr int kClwSegs = 4;
constexpr int kClwMinSteps = 2;

template <int KS, int MB, bool PROD>
struct ClwLds {
  static constexpr int kX1 = kClUnits * 16;             // bytes of one kernel row's window
  static constexpr int kYOff = KS * kX1;
  static constexpr int kY1 = kFlatTile * 32;            // bytes of one 16-channel block of y
  static constexpr int kGOff = kYOff + MB * kY1;
  static constexpr int kBuf = kGOff + (PROD ? kY1 : 0);
  // the segments' sums [seg][tap][c][kRS]: 16-byte rows for the generator's
  // four-channel stores; an odd pitch for the convolution's, which run over taps
  static constexpr int kRS = MB * 16 + (PROD ? 4 : 1);
  static constexpr int kRed = (kClwSegs * KS * KS * 16 * kRS + KS * KS * kClwSegs * 16) * 4;
  static constexpr int kBytes = 2 * kBuf > kRed ? 2 * kBuf : kRed;
};

template <typename T, int KS, int MB, bool PROD>
__global__ __launch_bounds__(64 * kClwSegs * KS) void cl_wgrad_kernel(
    const T* __restrict__ x, const T* __restrict__ y, const T* __restrict__ gout,
    float* __restrict__ pw, float* __restrict__ pb, T* __restrict__ dw_out, T* __restrict__ db_out,
    ClWGeom g, BxFinish fin) {
  typedef Mma<T> M;
  typedef typename M::V V;
  typedef typename M::E ME;
  typedef ClwLds<KS, MB, PROD> L;
  constexpr int KK = KS * KS, r = KS / 2;
  constexpr int NW = kClwSegs * KS, NT = 64 * NW;
  extern __shared__ __attribute__((aligned(16))) char cwsm[];

  if constexpr (PROD) {
    if ((int)blockIdx.x >= g.dw_blocks) {
      // helper workgroup (uniform branch, before any barrier)
      const int64_t stride = (int64_t)(gridDim.x - g.dw_blocks) * NT;
      const int64_t first = (int64_t)(blockIdx.x - g.dw_blocks) * NT + threadIdx.x;
      const T* __restrict__ fgo = static_cast<const T*>(fin.gout);
      T* __restrict__ fgx = static_cast<T*>(fin.gx);
      for (int64_t it = first; it < fin.items; it += stride)
        bx_reduce_item<T, 4, true>(fin.part, fgo, fgx, fin.g, it);
      return;
    }
  }
  const int logical = xcd_remap(blockIdx.x, g.dw_blocks);
  const int ih = logical % g.halves;
  const int lg = logical / g.halves;
  const int split = lg / g.blocks;
  const int blk = lg - split * g.blocks;
  const int cblocks = PROD ? g.blocks / 3 : g.blocks;
  const int b = PROD ? blk / cblocks : 0;
  const int cb = blk - b * cblocks;
  const int d = PROD ? dil_of(b, g.d0, g.d1, g.d2) : 1;
  const int C = g.C;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int col16 = lane & 15, quad = lane >> 4;
  const int sg = wave % kClwSegs, ki = wave / kClwSegs;
  const int i0 = ih * MB * 16;  // first N channel of this workgroup
  const uint32_t S = g.f.S, lead = g.f.lead;

  const int step_beg = split * g.steps_per_split;
  int step_end = step_beg + g.steps_per_split;
  if (step_end > g.steps) step_end = g.steps;
  const int steps = step_end > step_beg ? step_end - step_beg : 0;

  // copies of a step: KS windows of the x block (8.5 KB each), then MB blocks
  // of y and the gradient block (8 KB each), 1 KB per copy
  constexpr int NX = (KS * kClUnits + 63) / 64, NY = MB * 8, NG = PROD ? 8 : 0;
  constexpr int NXJ = (NX + NW - 1) / NW, NYJ = (NY + NG + NW - 1) / NW;
  uint32_t xof[NXJ], yof[NYJ];
#pragma unroll
  for (int j = 0; j < NXJ; ++j) {
    const int u = 64 * (wave + NW * j) + lane;
    const int kr = u / kClUnits, rem = u - kr * kClUnits;
    xof[j] = kr < KS ? (uint32_t)((kr * d * g.f.P) * 32 + rem * 16) : kOob;
  }
  // (branch b's channels 16 cb .. +15 of the gradient: 8-channel groups j8, j8 + 1)
  const int j8 = b * (C / 8) + 2 * cb;
#pragma unroll
  for (int j = 0; j < NYJ; ++j) {
    const int cp = wave + NW * j;
    yof[j] = kOob;
    if (cp < NY) {
      const int u = 64 * cp + lane, yb = u / (2 * kFlatTile), rem = u - yb * 2 * kFlatTile;
      yof[j] = (uint32_t)yb * S * 32u + (uint32_t)rem * 16u;
    } else if (cp < NY + NG) {
      const int u = 64 * (cp - NY) + lane;
      const int k8 = j8 + (u & 1);
      if (16 * cb + 8 * (u & 1) < C)
        yof[j] = ((uint32_t)(k8 >> 1) * S + (uint32_t)(u >> 1)) * 32u + (uint32_t)(k8 & 1) * 16u;
    }
  }
  BufRes rx = make_buf(x, 0u), ry = make_buf(y, 0u), rg = make_buf(x, 0u);
  int rn = -1;
  auto image = [&](int n) {
    if (n != rn) {
      rn = n;
      rx = make_buf(x + (int64_t)n * g.x_img, (lead + (uint32_t)g.q * S) * 32u);
      ry = make_buf(y + (int64_t)n * g.y_img, (lead + (uint32_t)g.yq * S) * 32u);
      if constexpr (PROD)
        rg = make_buf(gout + (int64_t)n * g.g_img + (int64_t)C * S,
                      (lead + (uint32_t)((3 * C + 15) / 16) * S * 16u) * 2u);
    }
  };
  // step q: tile q % ft of image q / ft
  int sn, sp, spos;
  auto stage = [&](int buf) {
    image(sn);
    char* __restrict__ dst = cwsm + buf * L::kBuf;
    const uint32_t p0 = (uint32_t)spos;
    const uint32_t xs = ((uint32_t)cb * S + (uint32_t)((int)(lead + p0) - kClPad - r * d * g.f.P)) * 32u;
    const uint32_t ys = ((uint32_t)(ih * MB) * S + lead + p0) * 32u;
    const uint32_t gs = lead * 2u + p0 * 32u;
#pragma unroll
    for (int j = 0; j < NXJ; ++j) {
      const int cp = wave + NW * j;
      if (NX % NW != 0 && cp >= NX) break;
      const uint32_t vo = xof[j];
      if ((KS * kClUnits) % 64 == 0 || cp < NX - 1 || 64 * cp + lane < KS * kClUnits)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rx, (__attribute__((address_space(3))) void*)(dst + 1024 * cp), 16, vo, xs, 0, 0);
    }
#pragma unroll
    for (int j = 0; j < NYJ; ++j) {
      const int cp = wave + NW * j;
      if ((NY + NG) % NW != 0 && cp >= NY + NG) break;
      const uint32_t vo = yof[j];
      if (!PROD || cp < NY)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            ry, (__attribute__((address_space(3))) void*)(dst + L::kYOff + 1024 * cp), 16, vo, ys, 0, 0);
      else
        __builtin_amdgcn_raw_ptr_buffer_load_lds(
            rg, (__attribute__((address_space(3))) void*)(dst + L::kYOff + 1024 * cp), 16, vo, gs, 0, 0);
    }
    spos += kFlatTile;
    if (++sp == g.f.ft) {
      sp = spos = 0;
      ++sn;
    }
  };

  // generator: B fragment of the bias column (n == 0) against dK; convolution:
  // A fragment of ones against the grad_out block of the same index as cb
  const bool bias_wg = PROD ? ih == 0 : (cb < (C + 15) / 16 && cb / MB == ih);
  const bool do_bias = PROD || (bias_wg && ki == 0);
  const int bib = cb - ih * MB;
  V ones;
  {
    const ME one = !PROD || col16 == 0 ? (ME)1.0f : (ME)0.0f;
#pragma unroll
    for (int e = 0; e < 8; ++e) ones[e] = one;
  }
  f32x4 acc[KS][MB], accb[PROD ? KS : 1];
  // this lane's row of a transposing read: position 4 * quad + e of 16, bytes
  // 8a .. 8a + 7 of its 32
  const int trl = (4 * quad + ((lane >> 2) & 3)) * 32 + (lane & 3) * 8 + 32 * 32 * sg;
  // The sums over this split's steps.  MASK: positions outside the image left
  // out (flat_any).
  auto run = [&](auto maskc) {
    constexpr bool MASK = decltype(maskc)::value;
    int xl[KS];
#pragma unroll
    for (int kj = 0; kj < KS; ++kj) xl[kj] = ki * L::kX1 + trl + (kClPad + (kj - r) * d) * 32;
#pragma unroll
    for (int kj = 0; kj < KS; ++kj) {
      accb[PROD ? kj : 0] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int ib = 0; ib < MB; ++ib) acc[kj][ib] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    sn = step_beg / g.f.ft;
    sp = step_beg - sn * g.f.ft;
    spos = sp * kFlatTile;
    if (steps > 0) stage(0);
    __builtin_amdgcn_s_waitcnt(0);
    __syncthreads();
    for (int s = 0; s < steps; ++s) {
      const int buf = s & 1;
      const bool more = s + 1 < steps;
      if (more) stage(buf ^ 1);
      const char* __restrict__ bb = cwsm + buf * L::kBuf;
      auto read8 = [&](int off) {
        u32x4 v;
        uint32_t a0, a1, b0, b1;
        cl_read_tr(bb + off, a0, a1);
        cl_read_tr(bb + off + 512, b0, b1);
        v[0] = a0;
        v[1] = a1;
        v[2] = b0;
        v[3] = b1;
        return v;
      };
      // (the masked form stays rolled: unrolled, it cost the other one's
      // schedule, bf16 4x32x135x181 42.1 -> 46.8 us)
#pragma unroll(MASK ? 1 : 2)
      for (int j = 0; j < 2; ++j) {
        const int jo = 4096 * j;  // 128 positions of 32 bytes
        V bfr[MB];
#pragma unroll
        for (int ib = 0; ib < MB; ++ib)
          bfr[ib] = __builtin_bit_cast(V, read8(L::kYOff + ib * L::kY1 + trl + jo));
        ClProd<T> gp;
        if constexpr (PROD) gp.set(read8(L::kGOff + trl + jo));
        if (!PROD && do_bias) {
#pragma unroll
          for (int ib = 0; ib < MB; ++ib)
            if (ib == bib) accb[0] = M::mac1(ones, bfr[ib], accb[0]);
        }
        u32x4 xv[KS];
#pragma unroll
        for (int kj = 0; kj < KS; ++kj) xv[kj] = read8(xl[kj] + jo);
        int in0 = 8, in1 = 8;
        if constexpr (MASK) {
          const int pos = (step_beg + s) % g.f.ft * kFlatTile + 128 * j + 32 * sg + 4 * quad;
          in0 = flat_inside(g.f, pos);
          in1 = flat_inside(g.f, pos + 16);
        }
#pragma unroll
        for (int kj = 0; kj < KS; ++kj) {
          u32x4 av = xv[kj];
          if constexpr (PROD) av = gp.mul(av);
          if constexpr (MASK)
            av = (u32x4){flat_keep2(av[0], in0, 0), flat_keep2(av[1], in0, 2),
                         flat_keep2(av[2], in1, 0), flat_keep2(av[3], in1, 2)};
          const V afr = __builtin_bit_cast(V, av);
#pragma unroll
          for (int ib = 0; ib < MB; ++ib) acc[kj][ib] = M::mac1(afr, bfr[ib], acc[kj][ib]);
          if constexpr (PROD) accb[kj] = M::mac1(afr, ones, accb[kj]);
        }
      }
      __builtin_amdgcn_s_waitcnt(0);
      __syncthreads();
    }
  };
  run(std::false_type());
  {
    bool nan = false;
#pragma unroll
    for (int kj = 0; kj < KS; ++kj) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (PROD) nan = nan || accb[kj][e] != accb[kj][e];
#pragma unroll
        for (int ib = 0; ib < MB; ++ib) nan = nan || acc[kj][ib][e] != acc[kj][ib][e];
      }
    }
    if (__builtin_expect(flat_any<NW>(nan, reinterpret_cast<uint32_t*>(cwsm), wave), 0)) run(std::true_type());
  }

  // ---- fixed-order sum over the segments through LDS
  constexpr int NO = MB * 16, RS = L::kRS, SL = KK * 16 * RS;
  float* __restrict__ red = reinterpret_cast<float*>(cwsm);
  float* __restrict__ rb = red + kClwSegs * SL;
  if constexpr (PROD) {
    if (col16 == 0) {
#pragma unroll
      for (int kj = 0; kj < KS; ++kj)
#pragma unroll
        for (int e = 0; e < 4; ++e)
          rb[((ki * KS + kj) * kClwSegs + sg) * 16 + 4 * quad + e] = accb[kj][e];
    }
  } else if (do_bias && quad == 0) {
    rb[sg * 16 + col16] = accb[0][0];
  }
#pragma unroll
  for (int kj = 0; kj < KS; ++kj)
#pragma unroll
    for (int ib = 0; ib < MB; ++ib)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        red[sg * SL + ((ki * KS + kj) * 16 + 4 * quad + e) * RS + ib * 16 + col16] = acc[kj][ib][e];
  __syncthreads();
  if constexpr (PROD) {
    float* __restrict__ pwb = pw + ((int64_t)split * 3 + b) * KK * C * C;
    T* __restrict__ dwb = dw_out + (int64_t)b * C * KK * C;
    for (int idx = tid; idx < KK * 16 * NO / 4; idx += NT) {
      const int qd = 4 * idx;
      const int t = qd / (16 * NO), rem = qd - t * 16 * NO;
      const int c = rem / NO, il = rem - c * NO;
      const int ch = cb * 16 + c, i = i0 + il;
      if (ch >= C || i >= C) continue;  // C % 8 == 0: four channels i are all in or out
      const float* __restrict__ sp4 = red + (t * 16 + c) * RS + il;
      auto q4 = [&](int k) { return *reinterpret_cast<const f32x4*>(sp4 + k * SL); };
      const f32x4 v = ((q4(0) + q4(1)) + q4(2)) + q4(3);
      if (g.direct) {
        T* __restrict__ o = dwb + (uint32_t)((ch * KK + t) * C + i);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = from_f<T>(v[e]);
      } else {
        *reinterpret_cast<f32x4*>(pwb + (uint32_t)((t * C + ch) * C + i)) = v;
      }
    }
    for (int idx = tid; idx < (bias_wg ? KK * 16 : 0); idx += NT) {
      const int t = idx >> 4, c = idx & 15, ch = cb * 16 + c;
      if (ch >= C) continue;
      float v = 0.f;
      for (int j = 0; j < kClwSegs; ++j) v += rb[(t * kClwSegs + j) * 16 + c];
      if (g.direct)
        db_out[(int64_t)(b * C + ch) * KK + t] = from_f<T>(v);
      else
        pb[((int64_t)split * 3 * KK + b * KK + t) * C + ch] = v;
    }
  } else {
    const int CI = 4 * C;
    float* __restrict__ pwb = pw + (int64_t)split * 9 * CI * C;
    // four consecutive elements (c, t) of one co's run of 16 x 9 per task
    for (int idx = tid; idx < NO * 36; idx += NT) {
      const int i = idx / 36, r4 = 4 * (idx - i * 36);
      if (i0 + i >= C) continue;
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int c = (r4 + e) / 9, t = r4 + e - c * 9;
        const float* __restrict__ s1 = red + (t * 16 + c) * RS + i;
        v[e] = ((s1[0] + s1[SL]) + s1[2 * SL]) + s1[3 * SL];
      }
      const uint32_t o = (uint32_t)((i0 + i) * CI + cb * 16) * 9u + (uint32_t)r4;
      if (g.direct) {
#pragma unroll
        for (int e = 0; e < 4; ++e) dw_out[o + e] = from_f<T>(v[e]);
      } else {
        *reinterpret_cast<f32x4*>(pwb + o) = v;
      }
    }
    if (bias_wg && tid < 16) {
      const int co = cb * 16 + tid;
      if (co < C) {
        const float v = ((rb[tid] + rb[16 + tid]) + rb[32 + tid]) + rb[48 + tid];
        if (g.direct)
          db_out[co] = from_f<T>(v);
        else
          pb[(int64_t)split * C + co] = v;
      }
    }
  }
}

void clw_geom(ClWGeom& g, const FlatLay& f, int64_t n, int64_t c, bool generator) {
  g.N = (int)n;
  g.C = (int)c;
  g.f = f;
  g.d0 = g.d1 = g.d2 = 1;
  const int64_t cp = flat_planes(c);
  const int64_t xp = generator ? cp : 4 * c;
  g.q = (int)(xp / 16);
  g.x_img = xp * f.S;
  g.yq = (int)(cp / 16);
  g.y_img = cp * f.S;
  g.g_img = cl_cat_planes(c) * f.S;
  g.blocks = generator ? 3 * (int)((c + 15) / 16) : (int)(4 * c / 16);
  g.halves = c > 64 ? 2 : 1;
  const int64_t steps = n * f.ft;
  int64_t splits = 16;
  if (splits > (steps + kClwMinSteps - 1) / kClwMinSteps) splits = (steps + kClwMinSteps - 1) / kClwMinSteps;
  splits = wgrad_splits(splits, steps, (int64_t)g.blocks * g.halves);
  g.steps = (int)steps;
  g.steps_per_split = (int)((steps + splits - 1) / splits);
  g.splits = (int)((steps + g.steps_per_split - 1) / g.steps_per_split);
  g.direct = g.splits == 1;
  g.dw_blocks = g.splits * g.blocks * g.halves;
}

int64_t clw_partial_bytes(const ClWGeom& g, int kk, bool generator) {
  if (g.direct) return 0;
  const int64_t c = g.C;
  return (int64_t)g.splits * (generator ? 3 * kk * c * (c + 1) : 36 * c * c + c) * 4;
}

namespace {

template <typename F>
int clw_pick(int dtype, int64_t c, F&& f) {
  auto by_mb = [&](auto tag) {
    const int mb = c > 64 ? 4 : (int)((c + 15) / 16);
    if (mb == 1) return f(tag, std::integral_constant<int, 1>());
    if (mb == 2) return f(tag, std::integral_constant<int, 2>());
    if (mb == 3) return f(tag, std::integral_constant<int, 3>());
    return f(tag, std::integral_constant<int, 4>());
  };
  if (dtype == kBF16) return by_mb(bf16());
  if (dtype == kF16) return by_mb(f16());
  return kBadArgument;
}

}  // namespace

int clw_launch_gen(int dtype, int ksize, const ClWGeom& g, const void* x, const void* y,
                   const void* gout, float* pw, float* pb, void* dw, void* db, int helpers,
                   const BxFinish& fin, hipStream_t stream) {
  return clw_pick(dtype, g.C, [&](auto tag, auto mbc) {
    using T = decltype(tag);
    auto go = [&](auto ksc) {
      constexpr int KS = decltype(ksc)::value, MB = decltype(mbc)::value;
      typedef ClwLds<KS, MB, true> L;
      auto kern = cl_wgrad_kernel<T, KS, MB, true>;
      const int ae = allow_dynamic_lds(reinterpret_cast<const void*>(kern), L::kBytes);
      if (ae != 0) return ae;
      hipLaunchKernelGGL(kern, dim3((unsigned)(g.dw_blocks + helpers)), dim3(64 * kClwSegs * KS),
                         L::kBytes, stream, (const T*)x, (const T*)y, (const T*)gout, pw, pb, (T*)dw,
                         (T*)db, g, fin);
      return (int)hipGetLastError();
    };
    return ksize == 1 ? go(std::integral_constant<int, 1>()) : go(std::integral_constant<int, 3>());
  });
}

int clw_launch_conv(int dtype, const ClWGeom& g, const void* cat, const void* gout, float* pw,
                    float* pb, void* dw, void* db, hipStream_t stream) {
  return clw_pick(dtype, g.C, [&](auto tag, auto mbc) {
    using T = decltype(tag);
    constexpr int MB = decltype(mbc)::value;
    typedef ClwLds<3, MB, false> L;
    auto kern = cl_wgrad_kernel<T, 3, MB, false>;
    const int ae = allow_dynamic_lds(reinterpret_cast<const void*>(kern), L::kBytes);
    if (ae != 0) return ae;
    hipLaunchKernelGGL(kern, dim3((unsigned)g.dw_blocks), dim3(64 * kClwSegs * 3), L::kBytes, stream,
                       (const T*)cat, (const T*)gout, (const T*)nullptr, pw, pb, (T*)dw, (T*)db, g,
                       BxFinish{nullptr, nullptr, nullptr, TileGeom{}, 0, 1});
    return (int)hipGetLastError();
  });
}

}  // namespace ddpm
