// Fused kernel generator + dynamic dilated filter + concat, forward.
//
// Counterpart of the reference's _generator_dynamic_cat_fwd
// (_triton_kernels.py:268-420, launched at :873-908), redesigned for CDNA4:
//
//   gen[(b,c,tap), p] = sum_i W[(b,c,tap), i] * y[i, p] + bias[(b,c,tap)]
//   out_b[c, p]       = sum_tap q(gen[(b,c,tap), p]) * x[c, p + off(b,tap)]
//   cat               = [x, out_0, out_1, out_2]
//
// q() rounds the generated tap to the input dtype (bf16/f16), as the
// reference does before consuming it (_triton_kernels.py:332-335).  The
// workgroup body (gen_tile.h) keeps the x halo tile in LDS and the generated
// taps in the MFMA result registers; the identity part of the concat is
// written from the registers that stage the halo tile.

#include "gen_tile.h"
#include <type_traits>

namespace ddpm {

// CB = 4: 256 registers per lane (one 8-wave workgroup per CU, whose 133 KB
// halo tile fills the LDS anyway); CB = 2: 128 registers, two workgroups per
// CU, unless the y operand needs more (gt_waves_per_eu).
// PP: the concat as pair planes (kF32Pairs, fp32 only); CL: channels-last in
// a flat layout (2-byte types).
template <typename T, int KS, int NK, int CB, bool PP = false, bool CL = false>
__global__ __launch_bounds__(kGtThreads) __attribute__((amdgpu_waves_per_eu(gt_waves_per_eu<T, NK, CB>()))) void gen_fwd_kernel(
    const T* __restrict__ x, const T* __restrict__ y, const T* __restrict__ wt,
    const T* __restrict__ bias, T* __restrict__ out, TileGeom g, CvPack fpk, FlatZero zero) {
  gen_tile_body<T, KS, NK, CB, false, PP, CL>(x, y, wt, bias, out, nullptr, g, fpk, zero);
}

// a.lo * b.lo + a.hi * b.hi + c on packed T pairs (v_dot2_f32_bf16 / _f16).
template <typename T>
__device__ __forceinline__ float dot2(uint32_t a, uint32_t b, float c) {
  if constexpr (__is_same(T, bf16)) {
    typedef bf16 v2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b), c,
                                           false);
  } else {
    typedef f16 v2 __attribute__((ext_vector_type(2)));
    return __builtin_amdgcn_fdot2(__builtin_bit_cast(v2, a), __builtin_bit_cast(v2, b), c, false);
  }
}

// Exchanges between the wave's rows of 16 lanes: rows 2, 3 of a with rows 0, 1
// of b; rows 1, 3 of a with rows 0, 2 of b.
__device__ __forceinline__ void swap_rows32(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}
__device__ __forceinline__ void swap_rows16(uint32_t& a, uint32_t& b) {
  const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
  a = r[0];
  b = r[1];
}

// Forward for 2-byte types at K = 3 with the taps paired in the MFMA rows.
// The generator rows of a step are 8 channels x 2 taps (row m: channel
// c0 + 8*mb + m/2, tap 2j + m%2; the fifth step of a branch holds tap 8 and a
// zero row, a step of its own without the partner's reads: 8x64x256x256 bf16
// 280 -> 262 us, 4x96x150x211 159 -> 140 us), so a lane's 4 results are (ca, t0), (ca, t1), (cb, t0), (cb, t1)
// for two channels ca, cb: one cvt_pk rounds a channel's two taps to T
// together and one v_dot2_f32 multiplies them by x at the two shifted pixels
// and accumulates -- 1.5 VALU instructions per (channel, tap, pixel) where the
// one-tap rows need 4 (round, widen, widen x, fma).  Every pair step's weight
// slice (15 x 2 row blocks x C input channels, 16-byte fragment units copied
// straight from the weight rows; C % 8 == 0) stays in LDS, so the loop has no
// barrier.  The x halo tile, the identity channels and the y operand are
// the tile kernels' (gen_tile.h).
template <typename T, int NK, int CB, bool CL>
__global__ __launch_bounds__(kGtThreads) __attribute__((amdgpu_waves_per_eu(gt_waves_per_eu<T, NK, CB>()))) void gen_fwd_pair_kernel(
    const T* __restrict__ x, const T* __restrict__ y, const T* __restrict__ wt,
    const T* __restrict__ bias, T* __restrict__ out, TileGeom g, CvPack fpk, FlatZero zero) {
  static_assert(sizeof(T) == 2, "2-byte types");
  typedef Mma<T> M;
  typedef typename M::V V;
  constexpr int KK = 9;
  constexpr int NPB = 5;        // tap pairs per branch
  constexpr int NPS = 3 * NPB;  // pair steps
  constexpr int E = 2;
  constexpr int XB = 4 * E;     // bytes of one 4-channel x entry
  constexpr int SU = 2 * NK;    // fragment units (x 64 lanes x 16 B) of one pair step: [mb][kk]
  constexpr int TW = 16 * CB;
  constexpr int NBW = 2 * CB;

  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  unsigned char* __restrict__ xs = smem;                                         // [4][plane]
  unsigned char* __restrict__ abuf = smem + 4 * g.plane;                         // [NPS][SU][64] x 16 B
  float* __restrict__ bs = reinterpret_cast<float*>(abuf + NPS * SU * 64 * 16);  // [NPS][32]

  const int bid = xcd_remap(blockIdx.x, gridDim.x);
  const int cb = bid % g.cblocks;
  const int nt = bid / g.cblocks;
  const int tile = nt % g.tiles;
  const int n = nt / g.tiles;
  const int ty = tile / g.tiles_w, tx = tile - ty * g.tiles_w;
  const int h0 = ty * kGtTH, w0 = tx * TW;
  const int C = g.C, H = g.H, W = g.W, R = g.R, LW = g.LW;
  const int64_t OS = g.OS;
  const uint32_t OSE = g.OS * (uint32_t)E;  // bytes of one concat plane
  const int OP = g.OP;
  out += g.olead;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int col16 = lane & 15, quad = lane >> 4;
  const int c0 = cb * 16;
  const int nch = C - c0 < 16 ? C - c0 : 16;

  // x halo tile first (its loads are consumed here); then the bias rows, the
  // weight slices and the y operand, all in flight together
  gt_stage_x<T, XB, CB, false, CL>(x, out, xs, g, n, c0, nch, h0, w0, TW, tid);
  // ---- bias rows [ps][mb*16 + m], written to LDS at the end of the prologue
  static_assert(NPS * 32 <= kGtThreads, "one bias value per thread");
  uint32_t bv;
  {
    const int ps = tid >> 5, rr = tid & 31;
    const int mb = rr >> 4, m = rr & 15;
    const int b = ps / NPB, j = ps - b * NPB;
    const int c = c0 + 8 * mb + (m >> 1), t = 2 * j + (m & 1);
    const BufRes bres = make_buf(bias, (uint32_t)(3 * C * KK * E));
    bv = gf_load_raw<E>(bres, (tid < NPS * 32 && c < C && t < KK)
                                  ? (uint32_t)((b * C + c) * KK + t) * (uint32_t)E
                                  : kOob);
  }
  // ---- every pair step's weight slice -> LDS: unit (ps, mb, kk, lane) holds
  //      the 16 bytes W[(b, c0 + 8mb + m/2, 2j + m%2)][kk*32 + 8q .. +7],
  //      m = lane & 15, q = lane >> 4 (zero for tap 9 and channels >= C)
  {
    const BufRes wres = make_buf(wt, (uint32_t)(3 * C * KK * C * E));
    const int m = lane & 15;
    for (int u = wave; u < NPS * SU; u += kGtWaves) {
      const int ps = u / SU, rem = u - ps * SU;
      const int mb = rem / NK, kk = rem - mb * NK;
      const int b = ps / NPB, j = ps - b * NPB;
      const int c = c0 + 8 * mb + (m >> 1), t = 2 * j + (m & 1), i0 = kk * 32 + 8 * quad;
      const uint32_t off =
          (c < C && t < KK && i0 < C) ? (uint32_t)((((b * C + c) * KK + t) * C + i0) * E) : kOob;
      __builtin_amdgcn_raw_ptr_buffer_load_lds(
          wres, (__attribute__((address_space(3))) void*)(abuf + (size_t)u * 64 * 16), 16, off, 0, 0,
          0);
    }
  }
  V bfr[NBW][NK][1];
  gt_load_y<T, NK, CB>(y, bfr, g, n, h0, w0, wave, col16, quad);
  if (tid < NPS * 32) bs[tid] = gf_raw_to_f<T>(bv);
  // ddpm_gen_fwd_pack: this workgroup's share of the fuse convolution's
  // weight packing
  if (fpk.total > 0) cv_pack_share<T>(fpk, (int)blockIdx.x, (int)gridDim.x, tid, kGtThreads);
  if constexpr (CL) flat_zero_share<T>(zero, (int)blockIdx.x, (int)gridDim.x, tid, kGtThreads);
  __builtin_amdgcn_s_waitcnt(0);  // the LDS-direct weight copies
  __syncthreads();
  if constexpr (CL) gt_store_identity<T, CB>(out, xs, g, n, c0, nch, h0, w0, tid);

  // x entry of this lane's two channels (8mb + 2q, +1) at its block-0 pixel:
  // plane 2mb + q/2, bytes 4*(q%2) .. +3 of the 4-channel entry
  const uint32_t lb = (uint32_t)((quad >> 1) * g.plane + col16 * XB + 4 * (quad & 1));
  // byte offset of row rr (0, 1) of this wave's blocks at zero shift in row
  // block mb's planes; block blk sits at row blk / CB, 16 * (blk % CB) entries
  // to the right
  auto rbase = [&](int rr, int mb) {
    return (uint32_t)(((2 * wave + rr + R) * LW + R) * XB + 2 * mb * g.plane);
  };
  // global byte offset of channel c0 + 8mb + 2q + e at pixel column `col` of
  // block blk (kOob outside the image or the channel block)
  auto goff = [&](int col, int blk, int mb, int e) {
    const int gh = h0 + 2 * wave + blk / CB, gw = w0 + 16 * (blk % CB) + col;
    const int cl = 8 * mb + 2 * quad + e;
    return (gh < H && gw < W && cl < nch) ? (uint32_t)cl * OSE + (uint32_t)(gh * OP + gw) * E : kOob;
  };

  float acc[NBW][2][2];  // branch output of channels (ca, cb) of each row block, per pixel block
  // Pair step j of branch b.  TWO: taps 2j and 2j + 1; else the lone tap 8,
  // whose partner -- a zero row, NaN where y is infinite -- is left out on
  // both sides.
  auto step = [&](int b, int j, auto twoc) {
    constexpr bool TWO = decltype(twoc)::value;
    const int ps = b * NPB + j;
    const int d = dil_of(b, g.d0, g.d1, g.d2);
    const int t0 = 2 * j, t1 = t0 + 1;
    const int sh0 = ((t0 / 3 - 1) * d * LW + (t0 % 3 - 1) * d) * XB;
    const int sh1 = TWO ? ((t1 / 3 - 1) * d * LW + (t1 % 3 - 1) * d) * XB : sh0;
    // x pairs (channel a: t0, t1) and (channel b: t0, t1) from the two reads
    constexpr uint32_t sela = TWO ? 0x05040100u : 0x0c0c0100u;
    constexpr uint32_t selb = TWO ? 0x07060302u : 0x0c0c0302u;
    const unsigned char* __restrict__ ab = abuf + ps * SU * 64 * 16;
    // both row blocks' MFMAs first, then both epilogues: the second block's
    // MFMAs run while the first block's epilogue issues
    f32x4 dacc[2][NBW];
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
      V afr[NK];
#pragma unroll
      for (int kk = 0; kk < NK; ++kk)
        afr[kk] = __builtin_bit_cast(V, *reinterpret_cast<const u32x4*>(ab + ((mb * NK + kk) * 64 + lane) * 16));
      const f32x4 binit = *reinterpret_cast<const f32x4*>(bs + ps * 32 + mb * 16 + 4 * quad);
#pragma unroll
      for (int blk = 0; blk < NBW; ++blk) {
        dacc[mb][blk] = binit;
#pragma unroll
        for (int kk = 0; kk < NK; ++kk) dacc[mb][blk] = M::mac1(afr[kk], bfr[blk][kk][0], dacc[mb][blk]);
      }
    }
#pragma unroll
    for (int mb = 0; mb < 2; ++mb) {
      uint32_t l = lb;
      asm volatile("" : "+v"(l));
      // one base per (row, shift); the block's column is the reads' immediate offset
      const unsigned char* __restrict__ p0[2] = {xs + l + (rbase(0, mb) + sh0), xs + l + (rbase(1, mb) + sh0)};
      const unsigned char* __restrict__ p1[2] = {xs + l + (rbase(0, mb) + sh1), xs + l + (rbase(1, mb) + sh1)};
#pragma unroll
      for (int blk = 0; blk < NBW; ++blk) {
        const int co = 16 * (blk % CB) * XB;
        const uint32_t x0 = *reinterpret_cast<const uint32_t*>(p0[blk / CB] + co);
        const uint32_t x1 = TWO ? *reinterpret_cast<const uint32_t*>(p1[blk / CB] + co) : x0;
        const uint32_t qa = pack2<T>(dacc[mb][blk][0], TWO ? dacc[mb][blk][1] : 0.f);
        const uint32_t qb = pack2<T>(dacc[mb][blk][2], TWO ? dacc[mb][blk][3] : 0.f);
        acc[blk][mb][0] = dot2<T>(qa, __builtin_amdgcn_perm(x1, x0, sela), acc[blk][mb][0]);
        acc[blk][mb][1] = dot2<T>(qb, __builtin_amdgcn_perm(x1, x0, selb), acc[blk][mb][1]);
      }
    }
  };
#pragma unroll 1
  for (int b = 0; b < 3; ++b) {
#pragma unroll
    for (int blk = 0; blk < NBW; ++blk)
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) acc[blk][mb][0] = acc[blk][mb][1] = 0.f;
#pragma unroll 1
    for (int j = 0; j < NPB - 1; ++j) step(b, j, std::true_type());
    step(b, NPB - 1, std::false_type());
    // ---- branch b: channels c0 + 8mb + 2q + e of output block b+1
    if constexpr (CL) {
      // channels-last.  A lane holds 2 of a pixel's 8 channels per row block;
      // swapping rows of 16 lanes between four pixel blocks gives lane row
      // q the 8 channels of block q's pixels, one 16-byte store (two blocks:
      // lane rows q and q + 2 hold 4 channels each of block q % 2, 8 bytes)
      const BufRes cres = make_buf(out + n * g.oimg, (uint32_t)(4 * C) * OSE);
#pragma unroll
      for (int mb = 0; mb < 2; ++mb) {
        const int cl = 8 * mb, pl = (b + 1) * C + c0 + cl;
        const uint32_t base = (uint32_t)(pl >> 4) * g.OS * 32u + (uint32_t)(pl & 15) * 2u;
        constexpr int Q = NBW < 4 ? 2 : 4;  // pixel blocks per exchange
#pragma unroll
        for (int b0 = 0; b0 < NBW; b0 += Q) {
          const int blk = b0 + (quad & (Q - 1));
          const int gh = h0 + 2 * wave + blk / CB, gw = w0 + 16 * (blk % CB) + col16;
          const uint32_t o = gh < H && gw < W && cl < nch
                                 ? base + (uint32_t)(gh * OP + gw) * 32u + (Q == 4 ? 0u : 8u * (quad >> 1))
                                 : kOob;
          uint32_t d[Q];
#pragma unroll
          for (int i = 0; i < Q; ++i) d[i] = pack2<T>(acc[b0 + i][mb][0], acc[b0 + i][mb][1]);
          if constexpr (Q == 4) {
            swap_rows32(d[0], d[2]);
            swap_rows32(d[1], d[3]);
            swap_rows16(d[0], d[1]);
            swap_rows16(d[2], d[3]);
            __builtin_amdgcn_raw_buffer_store_b128((u32x4){d[0], d[1], d[2], d[3]}, cres, o, 0, 0);
          } else {
            swap_rows16(d[0], d[1]);
            typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
            __builtin_amdgcn_raw_buffer_store_b64((u32x2){d[0], d[1]}, cres, o, 0, 0);
          }
        }
      }
    } else {
      const BufRes bres = make_buf(out + n * g.oimg + ((int64_t)(b + 1) * C + c0) * OS,
                                   (uint32_t)nch * OSE);
      int col = col16;  // (opaque: the offsets stay out of the steps' registers)
      asm volatile("" : "+v"(col));
#pragma unroll
      for (int blk = 0; blk < NBW; ++blk)
#pragma unroll
        for (int mb = 0; mb < 2; ++mb)
#pragma unroll
          for (int e = 0; e < 2; ++e) buf_store1<T>(bres, goff(col, blk, mb, e), acc[blk][mb][e]);
    }
  }
}

namespace {

template <typename F>
int with_type(int dt, F&& f) {
  switch (dt) {
    case kF32:
      return f(float());
    case kBF16:
      return f(bf16());
    case kF16:
      return f(f16());
    default:
      return kBadArgument;
  }
}

}  // namespace

// Shared with the backward entry points.
int gen_make_geom(GenGeom& g, int64_t n, int64_t c, int64_t h, int64_t w, int k, int d0, int d1,
                  int d2, int kmax) {
  if (n < 0 || c < 0 || h < 0 || w < 0) return kBadArgument;
  if (k < 1 || (k % 2) == 0 || d0 < 1 || d1 < 1 || d2 < 1) return kBadArgument;
  if (k > kmax || c > 128) return kUnsupported;
  if (h > (1 << 20) || w > (1 << 20) || h * w > ((int64_t)1 << 31)) return kUnsupported;
  if (k == 1) d0 = d1 = d2 = 1;  // a 1x1 tap has no neighbour to dilate
  g.N = (int)n;
  g.C = (int)c;
  g.H = (int)h;
  g.W = (int)w;
  g.K = k;
  g.d0 = d0;
  g.d1 = d1;
  g.d2 = d2;
  int dmax = d0 > d1 ? d0 : d1;
  dmax = dmax > d2 ? dmax : d2;
  g.R = (k / 2) * dmax;
  g.cblocks = (int)((c + 15) / 16);
  return kOk;
}

}  // namespace ddpm

using namespace ddpm;

extern "C" int64_t ddpm_flat_cat_elems(int64_t n, int64_t c, int64_t h, int64_t w, int guard,
                                       int dtype);

namespace {

// ddpm_gen_fwd's work; fpk (optional): a fuse-convolution weight packing for
// the kernel's workgroups to run.  check_only: validate and return before
// launching.  f (optional): the concat is a flat tensor of that layout; the
// kernel's workgroups zero its elements outside the images.
int gf_run(const void* x, const void* y, const void* weight, const void* bias, void* out,
           int64_t n, int64_t c, int64_t h, int64_t w, int kernel_size, int d0, int d1, int d2,
           int dtype, hipStream_t stream, const CvPack* fpk, bool check_only,
           const FlatLay* f = nullptr) {
  // kF32Pairs: fp32 inputs, the concat written as pair planes (C % 16 == 0)
  const bool pp = dtype == kF32Pairs;
  if (pp) {
    if (c % 16 != 0 || 32 * h * w * 4 > 0x7fffffffLL) return kUnsupported;
    dtype = kF32;
  }
  if (dtype < kF32 || dtype > kF16) return kBadArgument;
  GenGeom gg;
  int st = gen_make_geom(gg, n, c, h, w, kernel_size, d0, d1, d2, kGenFwdMaxK);
  if (st != kOk) return st;
  if (n == 0 || c == 0 || h == 0 || w == 0) return kOk;
  if (!x || !y || !weight || !bias || !out) return kBadArgument;
  if (check_only) return kOk;
  const int esz = dtype == kF32 ? 4 : 2;
  const CvPack pk = fpk ? *fpk : CvPack{nullptr, nullptr, ConvGeom{}, 0, 0, 0, 0};
  // 32-bit buffer offsets inside one image's [C][H][W] planes (and 16 planes
  // past a channel block's first one)
  if (c * h * w * esz > 0x7fffffffLL || 16 * h * w * esz > 0x7fffffffLL) return kUnsupported;
  TileGeom g;
  size_t lds = 0;
  const int parts = esz == 4 ? 2 : 1;
  const int nk = gt_nk((int)c);
  int cb = 4;
  st = tile_geom_for(g, gg, 4 * esz, parts, cb, lds);
  if (st != kOk) return st;
  FlatZero zero{nullptr, FlatLay{}, 0};
  if (f) {
    g.OP = f->P;
    g.OS = f->S;
    g.olead = (esz == 2 ? 16 : 1) * f->lead;
    g.oimg = 4 * c * (int64_t)f->S;
    zero = FlatZero{out, *f, (int)(n * 4 * c)};
  }
  // 2-byte types at K = 3 (C % 8 == 0, aligned weight): taps paired in the
  // MFMA rows, every weight slice resident in LDS, where that leaves room for
  // the halo tile
  auto pair_lds = [&](const TileGeom& t) {
    return (size_t)4 * t.plane + (size_t)15 * 2 * nk * 64 * 16 + (size_t)15 * 32 * 4;
  };
  size_t lds_pair = pair_lds(g);
  bool pair = esz == 2 && kernel_size == 3 && c % 8 == 0 && (uintptr_t)weight % 16 == 0;
  if (pair && nk > 2) {
    // one workgroup per CU (the weights take 92 or 123 KB): the tile width
    // with the shortest run of rounds, a workgroup taking about 1 + cb.  f16
    // at three chunks and 64 columns spills (184 us against 32 columns' 152 us
    // at 4x96x150x211 when it was built, 149 us now; bf16's 256 registers just
    // hold it in its loops, 144 us).  The kernel with one tap per step and 128
    // channels' padding took 219 us there (bf16), and 158 us against 115 us at
    // 1x128x256x256.  At four chunks 64
    // columns fit the LDS with dilations (1, 1, 1) only: no kernel is built
    // for them.
    pair = false;
    int64_t best = 0;
    for (int tcb = nk == 4 || dtype == kF16 ? 2 : 4; tcb >= 1; tcb /= 2) {
      TileGeom t;
      size_t tl;
      if (tile_geom(t, gg, 4 * esz, parts, tcb, tl) != kOk || pair_lds(t) > (size_t)kGtMaxLds) continue;
      const int64_t cost =
          ((int64_t)t.N * t.tiles * t.cblocks + kGtFillWGs - 1) / kGtFillWGs * (1 + tcb);
      if (pair && cost >= best) continue;
      pair = true;
      best = cost;
      cb = tcb;
      t.OP = g.OP;
      t.OS = g.OS;
      t.olead = g.olead;
      t.oimg = g.oimg;
      lds_pair = pair_lds(t);
      g = t;
    }
  }
  pair = pair && lds_pair <= (size_t)kGtMaxLds;
  if (pair) {
    return with_type(dtype, [&](auto tag) {
      using T = decltype(tag);
      if constexpr (sizeof(T) == 2) {
        auto launch = [&](auto kern) {
          const int ae = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds_pair);
          if (ae != 0) return ae;
          hipLaunchKernelGGL(kern, dim3((unsigned)((int64_t)g.N * g.tiles * g.cblocks)),
                             dim3(kGtThreads), lds_pair, stream, (const T*)x, (const T*)y,
                             (const T*)weight, (const T*)bias, (T*)out, g, pk, zero);
          return (int)hipGetLastError();
        };
        auto pick = [&](auto clc) {
          constexpr bool CL = decltype(clc)::value;
          auto by_nk = [&](auto cbc) {
            constexpr int CB = decltype(cbc)::value;
            if (nk == 1) return launch(gen_fwd_pair_kernel<T, 1, CB, CL>);
            if (nk == 2) return launch(gen_fwd_pair_kernel<T, 2, CB, CL>);
            // (the tile is the geometry's: one that has no kernel is refused)
            if constexpr (CB < 4 || !__is_same(T, f16)) {
              if (nk == 3) return launch(gen_fwd_pair_kernel<T, 3, CB, CL>);
            }
            if constexpr (CB < 4) {
              if (nk == 4) return launch(gen_fwd_pair_kernel<T, 4, CB, CL>);
            }
            return (int)kUnsupported;
          };
          if (cb == 4) return by_nk(std::integral_constant<int, 4>());
          if (cb == 2) return by_nk(std::integral_constant<int, 2>());
          return by_nk(std::integral_constant<int, 1>());
        };
        return f ? pick(std::true_type()) : pick(std::false_type());
      } else {
        return (int)kBadArgument;
      }
    });
  }
  return with_type(dtype, [&](auto tag) {
    using T = decltype(tag);
    auto launch = [&](auto kern) {
      const int ae = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds);
      if (ae != 0) return ae;
      hipLaunchKernelGGL(kern, dim3((unsigned)((int64_t)g.N * g.tiles * g.cblocks)),
                         dim3(kGtThreads), lds, stream, (const T*)x, (const T*)y,
                         (const T*)weight, (const T*)bias, (T*)out, g, pk, zero);
      return (int)hipGetLastError();
    };
    // 1 to 4 chunks of 32 input channels
    auto pick = [&](auto ks, auto ppc, auto clc) {
      constexpr int KS = decltype(ks)::value;
      constexpr bool PP = decltype(ppc)::value && sizeof(T) == 4;
      constexpr bool CL = decltype(clc)::value && sizeof(T) == 2;
      if (nk > 2)  // 32-column tiles
        return nk == 3 ? launch(gen_fwd_kernel<T, KS, 3, 2, PP, CL>) : launch(gen_fwd_kernel<T, KS, 4, 2, PP, CL>);
      if (cb == 4)
        return nk == 1 ? launch(gen_fwd_kernel<T, KS, 1, 4, PP, CL>) : launch(gen_fwd_kernel<T, KS, 2, 4, PP, CL>);
      if (cb == 1)
        return nk == 1 ? launch(gen_fwd_kernel<T, KS, 1, 1, PP, CL>) : launch(gen_fwd_kernel<T, KS, 2, 1, PP, CL>);
      return nk == 1 ? launch(gen_fwd_kernel<T, KS, 1, 2, PP, CL>) : launch(gen_fwd_kernel<T, KS, 2, 2, PP, CL>);
    };
    auto by_k = [&](auto ppc, auto clc) {
      if (kernel_size == 1) return pick(std::integral_constant<int, 1>(), ppc, clc);
      if (kernel_size == 3) return pick(std::integral_constant<int, 3>(), ppc, clc);
      return pick(std::integral_constant<int, 5>(), ppc, clc);
    };
    if (pp) return by_k(std::true_type(), std::false_type());
    return f ? by_k(std::false_type(), std::true_type()) : by_k(std::false_type(), std::false_type());
  });
}

}  // namespace

extern "C" int ddpm_gen_fwd(const void* x, const void* y, const void* weight, const void* bias,
                            void* out, int64_t n, int64_t c, int64_t h, int64_t w, int kernel_size,
                            int d0, int d1, int d2, int dtype, hipStream_t stream) {
  return gf_run(x, y, weight, bias, out, n, c, h, w, kernel_size, d0, d1, d2, dtype, stream,
                nullptr, false);
}

extern "C" int ddpm_gen_fwd_pack(const void* x, const void* y, const void* weight,
                                 const void* bias, void* out, const void* fuse_weight,
                                 void* fuse_workspace, int64_t fuse_workspace_bytes, int64_t n,
                                 int64_t c, int64_t h, int64_t w, int kernel_size, int d0, int d1,
                                 int d2, int dtype, hipStream_t stream) {
  // both parts validated before anything is launched
  int st = gf_run(x, y, weight, bias, out, n, c, h, w, kernel_size, d0, d1, d2, dtype, stream,
                  nullptr, true);
  if (st != kOk) return st;
  CvPack pk;
  st = cv_fwd_pack(pk, out, fuse_weight, fuse_workspace, fuse_workspace_bytes, n, c, h, w, dtype);
  if (st != kOk) return st;
  return gf_run(x, y, weight, bias, out, n, c, h, w, kernel_size, d0, d1, d2, dtype, stream, &pk,
                false);
}

extern "C" int ddpm_flat_gen_fwd_pack(const void* x, const void* y, const void* weight,
                                      const void* bias, void* cat, const void* fuse_weight,
                                      void* fuse_workspace, int64_t fuse_workspace_bytes, int64_t n,
                                      int64_t c, int64_t h, int64_t w, int kernel_size, int d0,
                                      int d1, int d2, int guard, int dtype, hipStream_t stream) {
  int st = gf_run(x, y, weight, bias, cat, n, c, h, w, kernel_size, d0, d1, d2, dtype, stream,
                  nullptr, true);
  if (st != kOk) return st;
  if (n == 0 || c == 0 || h == 0 || w == 0) return kOk;
  FlatLay f;
  if (ddpm_flat_cat_elems(n, c, h, w, guard, dtype) == 0 ||
      !flat_lay(f, h, w, guard, 4 * c, dtype == kBF16 || dtype == kF16 ? 2 : 4))
    return kUnsupported;
  if ((uintptr_t)cat % 16 != 0) return kBadArgument;
  CvPack pk;
  st = cv_fwd_pack(pk, cat, fuse_weight, fuse_workspace, fuse_workspace_bytes, n, c, h, w, dtype, &f);
  if (st != kOk) return st;
  return gf_run(x, y, weight, bias, cat, n, c, h, w, kernel_size, d0, d1, d2, dtype, stream, &pk,
                false, &f);
}
