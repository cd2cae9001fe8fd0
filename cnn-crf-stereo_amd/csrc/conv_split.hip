// float32 feature layers (fused valid convolution + bias + tanh) on the 16-bit
// matrix cores.
//
// gfx950 runs v_mfma_f32_16x16x32_f16 (and _bf16) at 16 times the rate of
// v_mfma_f32_16x16x4_f32.  Both operands are split into two float16 terms,
// x s = xh + xl / 4096 and w t = wh + wl / 4096 (split_pair), with a power of two s
// for each pixel's 32 channels of a stage and t for each output channel, and a
// product is formed from
//   (wl xh + wh xl) / 4096 + wh xh,
// each exact in the matrix core and accumulated in float32; wl xl, the one left
// out, is at most 2^-22 |x w| (2^-25 root mean square).  Where that does not do
// (BlockRange) a tile is computed on v_mfma_f32_16x16x4_f32 from memory instead: with
// huge or infinite inputs, or channels of a pixel more than 2^29 apart that meet
// uneven weights; and all tiles where the weights of a row are so far apart (their pack
// then holds them in float32).  Every output keeps float32's precision for any inputs.
// Channels past the last multiple of 32 take an exact
// three-way bfloat16 split (split3) and six of its nine products instead: their
// reduction steps hold several taps, hence several pixels, in one instruction, so
// no scale fits.  A 32-deep step is summed from zero and added to the accumulator
// once (by the fma that takes the pixel's scale back), so an output takes 30
// roundings at its own size (the float32 instruction took 225): the relative
// error of a layer against 64 bits is 1.3e-7 (3x3) and 1.1e-7 (2x2), where
// v_mfma_f32_16x16x4_f32 left 5.4e-7 and 3.6e-7 (tanh off, 200 x 300 maps).
//
// k_conv_split: a workgroup of 4 waves computes a tile of 8 x 16 pixels for all
// output channels; a wave owns MT = 2 rows of 16 pixels times NT 16-channel tiles
// of accumulators.  The (8+KH-1) x (16+KW-1) input halo tile is staged in LDS one
// stage of four 8-channel groups at a time, split into its planes on the way (180
// pixels x 64 bytes x 2 = 23 KB for 3x3); a step's weights (14 KB for 100
// channels) are copied to LDS once per workgroup while the step before runs.
// Three workgroups share a CU, and one's staging and epilogue run under the
// others' MFMAs.  A step issues 3 * MT * NT MFMAs (42, 700 cycles); its additions
// are spread between the next tile's MFMAs.
//
// Measured (100 channels, us; the float32-MFMA kernel -> six bfloat16 products
// with the weights read from L2 by every wave -> both terms in one unit, which lost
// the small channels of uneven pixels -> this): 3x3 at 1256 x 389 1456 -> 565 -> 411
// -> 431, at 524 x 268 - -> 175 -> 109 -> 115, 2x2 at 749 x 501 530 -> 205 -> 151 ->
// 157, at 325 x 245 140 -> 65 -> 41 -> 43, at 200 x 100 - -> 37 -> 18 -> 19.  (The
// second unit takes one more addition per value and step.)  At 1256 x 389 the matrix
// cores are busy half of the time; the rest is staging, the epilogue's tanh, and waits.
// Tiles of 16 x 16 (MT = 4, two workgroups per CU; with one unit) took 412, 128, 163,
// 52 and 30 us.
#include <type_traits>

#include "conv_split.hpp"

namespace ccs {

template <int KH_, int KW_, int CG_, int NT_, int MT_ = 2>
struct SplitCfg {
  static constexpr int KH = KH_, KW = KW_, CG = CG_, NT = NT_;
  static constexpr int Cs = CG * 8, MT = MT_, threads = 256;
  static constexpr int TH = 4 * MT, TW = 16;  // output tile: MT rows of 16 pixels per wave
  static constexpr int taps = KH * KW;
  static constexpr int FULL = CG / 4, REM = CG % 4;  // stages of four groups, groups of the last stage
  static constexpr int REM_NQ = (taps * REM + 3) / 4;
  static constexpr int NQ = FULL * taps + REM_NQ;  // 32-deep reduction steps
  static constexpr int AR = TH + KH - 1, AC = TW + KW - 1, NPX = AR * AC;
  static constexpr int plane = NPX * 64;  // bytes of one plane of a four-group stage
  static constexpr int rplane = NPX * REM * 16;  // and of the last stage
  static constexpr int scale_off = 2 * plane > 3 * rplane ? 2 * plane : 3 * rplane;
  // two steps' weights (two planes; in the last stage three, behind its smaller planes)
  static constexpr int w2 = NT * 2048, w3 = NT * 3072;
  static constexpr int w2_off = (scale_off + NPX * 4 + 1023) & ~1023;
  static constexpr int w3_off = (3 * rplane + 1023) & ~1023;
  static constexpr int zero_off = w2_off + 2 * w2 > w3_off + 2 * w3 ? w2_off + 2 * w2 : w3_off + 2 * w3;
  static constexpr int fail_off = zero_off + 16;  // per wave: its share of the inputs fails
  static constexpr int lds_bytes = fail_off + 16;
  // packed weights: two-plane fragments, three-plane fragments, row scales, and per
  // tile of 16 rows kWide (its two-plane fragments are float32 values instead) and kUneven
  static constexpr size_t frag_bytes = (size_t)NT * 1024 * (2 * FULL * taps + 3 * REM_NQ);
  static constexpr size_t flag_off = frag_bytes + NT * 16 * sizeof(float);
  static constexpr size_t packed_bytes = flag_off + (NT + 3) / 4 * 16;
};
enum RowFlag { kWide = 1, kUneven = 2 };

// Reduction step q of the packed weights, lane group lgrp: the tap and the
// first channel of its eight (c0 < 0: padding).  The first FULL * taps steps
// take one tap and four channel groups each; the steps of the last stage take
// its taps * REM (tap, group) pairs in tap-major order.
template <class Cfg>
__host__ __device__ inline void split_step(int q, int lgrp, int* tap, int* c0) {
  if (q < Cfg::FULL * Cfg::taps) {
    *tap = q % Cfg::taps;
    *c0 = (4 * (q / Cfg::taps) + lgrp) * 8;
  } else {
    constexpr int R = Cfg::REM > 0 ? Cfg::REM : 1;
    const int kg = 4 * (q - Cfg::FULL * Cfg::taps) + lgrp;
    *tap = kg / R;
    *c0 = kg < Cfg::taps * R ? (4 * Cfg::FULL + kg % R) * 8 : -1;
  }
}

// Packed layout: step q < FULL * taps as [q][t][2][lane][8] float16, the others
// as [q][t][3][lane][8] bfloat16, the fragment of channel tile t with lane
// (lrow, lgrp) holding output channel 16 t + lrow; then the row scales.  All
// weights of a row are divided by its scale.  A tile with a row that pairs do not
// hold has scales of 1 and its first fragments as [q][t][2][lane][4] float32.
// Block (t, y) packs row y of tile t and a share of its last steps; its 16 groups of
// 16 lanes each look at one row first.
//
// A pair holds 23 of a float's 24 bits, so that every fourth weight would be off by
// 2^-24 or 2^-23 of itself, the same for all pixels: maps whose channels have a mean were
// off by that mean times the sum of a channel's roundings, everywhere alike (the mean of
// an output channel by 4e-9 in a tower of values around 0.3, where float32 products leave
// 0.7e-9, and by up to 1e-7 of its size with positive inputs).  So what the low term of a
// tap leaves out is added to the next one's, what the last leaves to the tap whose low
// term is finest, and what that leaves to the next of 16 channels.  Only weights of at least half
// of the channel's largest take part, and from another channel only what is 2^-23 of this
// channel's largest at most: every weight stays within 2^-22 of itself, and a zero stays 0.
template <int N>
__device__ __forceinline__ void split_taps(const float (&v)[N], float s, _Float16 (&h)[N], _Float16 (&l)[N]) {
  float m = 0.f, carry = 0.f, finest = __builtin_huge_valf();
#pragma unroll
  for (int i = 0; i < N; ++i) m = fmaxf(m, fabsf(v[i]));
  int best = -1;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const float x = v[i] * s;
    h[i] = (_Float16)x;
    const float r = fmaf((float)h[i], -kLowUnit, x * kLowUnit);
    const bool large = m > 0.f && 2.f * fabsf(v[i]) >= m;
    const float want = large ? r + carry : r;
    l[i] = (_Float16)want;
    carry = large ? want - (float)l[i] : carry + (want - (float)l[i]);
    if (large && fabsf(r) < finest) {
      finest = fabsf(r);
      best = i;
    }
  }
  float fine = 0.f;
#pragma unroll
  for (int i = 0; i < N; ++i) fine = i == best ? (float)l[i] : fine;
  const float limit = m * s * kLowUnit * 0x1p-23f;
  float rest = 0.f;  // what the channels of this row of 16 lanes up to here leave out
#pragma unroll
  for (int i = 0; i < 16; ++i) {
    const float before = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(rest), 0x111, 0xf, 0xf, true));  // row_shr:1
    const float want = fine + (carry + before), got = (float)(_Float16)want;
    const bool take = best >= 0 && fabsf(before) <= limit;
    if ((int)(threadIdx.x & 15) == i) {
      rest = take ? want - got : before;
      fine = take ? got : fine;
    }
  }
#pragma unroll
  for (int i = 0; i < N; ++i) l[i] = i == best ? (_Float16)fine : l[i];
}

constexpr int kPackShares = 16;
template <class Cfg>
__global__ __launch_bounds__(256) void k_pack_split(const float* __restrict__ w, int K, int C, int adj,
                                                    unsigned char* __restrict__ out) {
  __shared__ int exps[16];
  const int tid = threadIdx.x, t = blockIdx.x;
  // adj: Wt[n][c] flipped, Wt[n][c][a][b] = w[c][n][KH-1-a][KW-1-b]
  auto at = [&](int n, int c, int tap) {
    return w[adj ? ((long)c * K + n) * Cfg::taps + tap : ((long)n * C + c) * Cfg::taps + (Cfg::taps - 1 - tap)];
  };
  const int row = 16 * t + (tid >> 4);
  BlockRange r;
  if (row < K) {  // (eight loads in flight)
#pragma unroll 8
    for (int i = tid & 15; i < C * Cfg::taps; i += 16) {
      const float v = at(row, i / Cfg::taps, i % Cfg::taps);
      r.above = fmaxf(r.above, fabsf(v));  // (the class's asm keeps the loop from being unrolled)
      r.least = fminf(r.least, fabsf(v));
      r.add_nonzero(v, v);
    }
  }
  unsigned mx = r.largest();
  for (int o = 1; o < 16; o <<= 1) mx = max(mx, (unsigned)__shfl_xor((int)mx, o, 16));
  const bool wide = __syncthreads_or(mx >= 242u << 23 || r.apart(split_exp(mx)));
  const bool uneven = __syncthreads_or(r.uneven(mx));
  if ((tid & 15) == 0) {
    exps[tid >> 4] = wide ? 127 : split_exp(mx);
    if (blockIdx.y == 0)
      reinterpret_cast<float*>(out + Cfg::frag_bytes)[row] = wide ? 1.f : __uint_as_float((unsigned)split_exp(mx) << 23);
  }
  if (blockIdx.y == 0 && tid == 0) reinterpret_cast<int*>(out + Cfg::flag_off)[t] = wide ? kWide : uneven ? kUneven : 0;
  __syncthreads();
  constexpr int NQ2 = Cfg::FULL * Cfg::taps, kLast = Cfg::REM_NQ * 64 / kPackShares;
  static_assert(Cfg::FULL * 32 <= 128 && kLast <= 128, "a thread per channel, then one per lane's share of a last step");
  if (tid < 128) {  // (whole waves)
    const int n = 16 * t + blockIdx.y, c = tid, e = c & 7, lane = ((c >> 3) & 3) * 16 + blockIdx.y, stage = c >> 5;
    float v[Cfg::taps];
#pragma unroll
    for (int j = 0; j < Cfg::taps; ++j) v[j] = stage < Cfg::FULL && n < K && c < C ? at(n, c, j) : 0.f;
    _Float16 h[Cfg::taps], l[Cfg::taps];
    split_taps(v, split_scale(exps[blockIdx.y]), h, l);
    if (stage < Cfg::FULL) {
#pragma unroll
      for (int j = 0; j < Cfg::taps; ++j) {
        unsigned char* frag = out + ((long)((stage * Cfg::taps + j) * Cfg::NT + t) * 128 + lane) * 16;
        if (wide) {
          reinterpret_cast<float*>(frag + (e >> 2) * 1024)[e & 3] = v[j];
        } else {
          reinterpret_cast<_Float16*>(frag)[e] = h[j];
          reinterpret_cast<_Float16*>(frag + 1024)[e] = l[j];
        }
      }
    }
  } else {
    const int u = blockIdx.y * kLast + tid - 128;
    if (tid - 128 < kLast) {
      const int lane = u & 63, n = 16 * t + (lane & 15), eb = exps[lane & 15], q = NQ2 + (u >> 6);
      int tap, c0;
      split_step<Cfg>(q, lane >> 4, &tap, &c0);
      const float unit = __uint_as_float(eb < 254 ? (unsigned)(254 - eb) << 23 : 0x400000u);  // 1 / the row's scale
      float v[8];
      bf16 p[3][8];
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = (n < K && c0 >= 0 && c0 + e < C ? at(n, c0 + e, tap) : 0.f) * unit;
      split3(v, p[0], p[1], p[2]);
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        bf16x8 o;
#pragma unroll
        for (int e = 0; e < 8; ++e) o[e] = p[k][e];
        *reinterpret_cast<bf16x8*>(out + (size_t)NQ2 * Cfg::NT * 2048 +
                                   ((long)(((q - NQ2) * Cfg::NT + t) * 3 + k) * 64 + lane) * 16) = o;
      }
    }
  }
}

// The four 16-byte groups of an LDS pixel are XOR-swizzled so that the reads of
// eight consecutive pixels land in eight distinct bank groups.
__device__ __forceinline__ int split_swz(int px, int g) { return g ^ ((px >> 1) & 3); }

// Each lane's 16 bytes from src go to dst + 16 lane (dst is uniform), counted by vmcnt.
__device__ __forceinline__ void load_lds16(const void* src, void* dst) {
  __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)dst, 16, 0, 0);
}

template <class Cfg>
__global__ __launch_bounds__(256, 2) void k_conv_split(const float* __restrict__ x, int Hin, int Win,
                                                       const unsigned char* __restrict__ wpk, const float* __restrict__ bias,
                                                       int K, int act, float* __restrict__ y, int Ho, int Wo,
                                                       int tiles_x, int tiles) {
  constexpr int MT = Cfg::MT, NT = Cfg::NT, AC = Cfg::AC, NPX = Cfg::NPX, Cs = Cfg::Cs;
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lrow = lane & 15, lgrp = lane >> 4;
  // Blocks b and b + 8 share an XCD: each XCD takes a contiguous run of tiles,
  // whose halos then meet in its L2.
  const int per = (tiles + 7) / 8;
  const int tile = (blockIdx.x & 7) * per + (blockIdx.x >> 3);
  if (tile >= tiles) return;  // (uniform) the grid is rounded up to 8 runs
  const int h0 = (tile / tiles_x) * Cfg::TH, w0 = (tile % tiles_x) * Cfg::TW;
  if (tid == 0) *reinterpret_cast<u32x4*>(lds + Cfg::zero_off) = u32x4{0u, 0u, 0u, 0u};
  bool fails = false;  // an input of this lane needs float32 products
  int flags = 0;
#pragma unroll
  for (int t = 0; t < NT; ++t) flags |= reinterpret_cast<const int*>(wpk + Cfg::flag_off)[t];
  bool again = flags & kWide;  // (uniform) the tile takes float32 products

  // Stage of G groups from channel group cg0: unit (pixel, group) of eight
  // channels, all loads issued before the first is split and stored.
  // Coordinates are clamped to the map (those values feed only output pixels
  // past Ho x Wo).
  auto stage = [&](auto gc, int cg0) {
    constexpr int G = decltype(gc)::value;
    constexpr int NU = NPX * G, PER = (NU + Cfg::threads - 1) / Cfg::threads;
    f32x4 in[PER][2];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int v = min(tid + Cfg::threads * i, NU - 1);
      const int px = v / G, g = v % G;
      const int hi = min(h0 + px / AC, Hin - 1), wi = min(w0 + px % AC, Win - 1);
      const f32x4* src = reinterpret_cast<const f32x4*>(x + ((long)hi * Win + wi) * Cs + (cg0 + g) * 8);
      in[i][0] = src[0];
      in[i][1] = src[1];
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int v = tid + Cfg::threads * i;
      const int px = v / G, g = v % G;
      float f[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = in[i][e >> 2][e & 3];
      if constexpr (G == 4) {
        // A pixel's four units lie in a quad of lanes: one scale for its 32 channels.
        auto quad_max = [](unsigned m) {
          m = max(m, (unsigned)__builtin_amdgcn_mov_dpp((int)m, 0xb1, 0xf, 0xf, true));
          return max(m, (unsigned)__builtin_amdgcn_mov_dpp((int)m, 0x4e, 0xf, 0xf, true));
        };
        BlockRange r;
#pragma unroll
        for (int e = 0; e < 8; e += 2) r.add_largest(f[e], f[e + 1]);
        const unsigned mx = quad_max(r.largest());
        const int eb = split_exp(mx);
        fails |= r.huge();
        if (flags & kUneven) {  // (uniform)
#pragma unroll
          for (int e = 0; e < 8; e += 2) r.add_nonzero(f[e], f[e + 1]);
          fails |= r.apart(eb);
        }
        const unsigned neg = parity_sign(mx);  // (see kNegate)
        f16x8 p[2];
        split_pair(f, with_sign(split_scale(eb), neg), p[0], p[1]);
        if (v < NU) {
          const int off = px * 64 + split_swz(px, g) * 16;
#pragma unroll
          for (int k = 0; k < 2; ++k) *reinterpret_cast<f16x8*>(lds + k * Cfg::plane + off) = p[k];
          if (g == 0) *reinterpret_cast<float*>(lds + Cfg::scale_off + px * 4) = with_sign(split_unscale(eb), neg);
        }
      } else {
        bf16 p[3][8];
        BlockRange r;
#pragma unroll
        for (int e = 0; e < 8; e += 2) r.add_largest(f[e], f[e + 1]);
        fails |= r.huge();
        split3(f, p[0], p[1], p[2]);
        if (v < NU) {
#pragma unroll
          for (int k = 0; k < 3; ++k) {
            bf16x8 o;
#pragma unroll
            for (int e = 0; e < 8; ++e) o[e] = p[k][e];
            *reinterpret_cast<bf16x8*>(lds + k * Cfg::rplane + (px * G + g) * 16) = o;
          }
        }
      }
    }
    const bool any = __any(fails);  // (read behind the barrier that follows)
    if (lane == 0) *reinterpret_cast<int*>(lds + Cfg::fail_off + 4 * wave) = any;
  };

  // Lane (lrow, lgrp) holds pixel lrow of row MT wave + m and channels
  // 16 t + 4 lgrp .. +3 (the weights are the A operand), over the rows' scales.
  f32x4 acc[MT][NT];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  // A step's weight fragments (1 KB each: one load of a wave, straight to LDS)
  // are copied once per workgroup, a step ahead, to the buffer the step before
  // has left.
  auto copy_w = [&](const unsigned char* src, int off, int frags) {
#pragma unroll 1
    for (int f = wave; f < frags; f += 4) load_lds16(src + (long)f * 1024 + lane * 16, lds + off + f * 1024);
  };
  auto copy2 = [&](int q) { copy_w(wpk + (long)q * Cfg::w2, Cfg::w2_off + (q & 1) * Cfg::w2, 2 * NT); };
  auto copy3 = [&](int ql) {
    copy_w(wpk + (long)Cfg::FULL * Cfg::taps * Cfg::w2 + (long)ql * Cfg::w3, Cfg::w3_off + (ql & 1) * Cfg::w3, 3 * NT);
  };
  // The scales of the output pixels' first inputs, whose signs the last stage's products
  // take (its reduction steps hold several inputs).
  float corner[MT];
  // The copies of this wave have arrived, and so have everyone's.
  auto step_barrier = [&]() {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
  };

  // The step's products are summed from zero and added to the accumulators
  // once, in the vector unit: the matrix core's roundings then happen at the
  // size of 32 products, and only the additions at that of the whole sum.
  auto step2 = [&](int q, int ti, int tj) {
    f16x8 a[2][MT];
    float sc[MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int px = (MT * wave + m + ti) * AC + tj + lrow;
      const int o = px * 64 + split_swz(px, lgrp) * 16;
#pragma unroll
      for (int k = 0; k < 2; ++k) a[k][m] = *reinterpret_cast<const f16x8*>(lds + o + k * Cfg::plane);
      sc[m] = *reinterpret_cast<const float*>(lds + Cfg::scale_off + px * 4);
    }
    const f16x8* wb = reinterpret_cast<const f16x8*>(lds + Cfg::w2_off + (q & 1) * Cfg::w2) + lane;
    f16x8 b0[2] = {wb[0], wb[64]}, b1[2];
    f32x4 low[2][MT], high[2][MT];  // the products with a low term, and the others
    auto add = [&](int t, int m) {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        acc[m][t][e] = fmaf(fmaf(low[t & 1][m][e], 1.f / kLowUnit, high[t & 1][m][e]), sc[m], acc[m][t][e]);
    };
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x4(&c)[MT] = low[t & 1];
#pragma unroll
      for (int m = 0; m < MT; ++m)
        c[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b0[1], a[0][m], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      // (the next tile's fragments are read behind these: the wait before a
      // tile's first product is for every LDS read issued so far)
      __builtin_amdgcn_sched_barrier(0);
      b1[0] = wb[128 * min(t + 1, NT - 1)];
      b1[1] = wb[128 * min(t + 1, NT - 1) + 64];
      if (t > 0) add(t - 1, 0);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        __builtin_amdgcn_sched_barrier(0);
        c[m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b0[0], a[1][m], c[m], 0, 0, 0);
        if (t > 0 && m > 0) add(t - 1, m);
      }
#pragma unroll
      for (int m = 0; m < MT; ++m)
        high[t & 1][m] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b0[0], a[0][m], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      b0[0] = b1[0];
      b0[1] = b1[1];
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) add(NT - 1, m);
  };
  // A step of the last stage (ql of REM_NQ): its lane groups hold different taps,
  // hence different pixels, so it takes the exact three-way split without scales.
  auto step3 = [&](int ql) {
    constexpr int R = Cfg::REM > 0 ? Cfg::REM : 1;
    const int kg = 4 * ql + lgrp;
    const bool ok = kg < Cfg::taps * R;
    const int tap = ok ? kg / R : 0, g = ok ? kg % R : 0;
    const int ti = tap / Cfg::KW, tj = tap % Cfg::KW;
    bf16x8 a[3][MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int px = (MT * wave + m + ti) * AC + tj + lrow;
      const int o = ok ? (px * R + g) * 16 : Cfg::zero_off;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        u32x4 v = *reinterpret_cast<const u32x4*>(lds + o + (ok ? k * Cfg::rplane : 0));
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] ^= corner[m] < 0.f ? 0x80008000u : 0u;
        a[k][m] = __builtin_bit_cast(bf16x8, v);
      }
    }
    const bf16x8* p = reinterpret_cast<const bf16x8*>(lds + Cfg::w3_off + (ql & 1) * Cfg::w3) + lane;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      bf16x8 b[3];
#pragma unroll
      for (int k = 0; k < 3; ++k) b[k] = p[t * 192 + 64 * k];
      f32x4 cur[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m)
        cur[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[0], a[2][m], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      auto mm = [&](int kw, int kx) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
          cur[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b[kw], a[kx][m], cur[m], 0, 0, 0);
      };
      mm(2, 0);
      mm(1, 1);
      mm(0, 1);
      mm(1, 0);
      mm(0, 0);
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const float sg = corner[m] < 0.f ? -1.f : 1.f;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[m][t][e] = fmaf(cur[m][e], sg, acc[m][t][e]);
        asm volatile("" : "+v"(acc[m][t]));  // added here, not behind the step (the sums of all tiles would spill)
      }
    }
  };

  // Whether the staged inputs fail in one of the waves (behind the barrier).
  auto failed = [&]() {
    const u32x4 f = *reinterpret_cast<const u32x4*>(lds + Cfg::fail_off);
    return __builtin_amdgcn_readfirstlane(f[0] | f[1] | f[2] | f[3]) != 0;
  };
  // (from the first failure on, without steps: leaving the loops instead takes 50 registers more)
  copy2(0);
#pragma unroll 1
  for (int s = 0; s < Cfg::FULL; ++s) {
    stage(std::integral_constant<int, 4>{}, 4 * s);
    step_barrier();
    again |= failed();
    if constexpr (Cfg::REM > 0) {
#pragma unroll
      for (int m = 0; m < MT; ++m)
        corner[m] = *reinterpret_cast<const float*>(lds + Cfg::scale_off + ((MT * wave + m) * AC + lrow) * 4);
    }
    const int taps = again ? 0 : Cfg::taps;
#pragma unroll 1
    for (int tap = 0; tap < taps; ++tap) {
      const int q = s * Cfg::taps + tap;
      if (q + 1 < Cfg::FULL * Cfg::taps) copy2(q + 1);
      step2(q, tap / Cfg::KW, tap % Cfg::KW);
      step_barrier();
    }
  }
  if constexpr (Cfg::REM > 0) {
    copy3(0);
    stage(std::integral_constant<int, Cfg::REM>{}, 4 * Cfg::FULL);
    step_barrier();
    again |= failed();
    const int steps = again ? 0 : Cfg::REM_NQ;
#pragma unroll 1
    for (int ql = 0; ql < steps; ++ql) {
      if (ql + 1 < Cfg::REM_NQ) copy3(ql + 1);
      step3(ql);
      if (ql + 1 < Cfg::REM_NQ) step_barrier();
    }
  }

  // The tile on v_mfma_f32_16x16x4_f32, for what the pairs do not hold.  Inputs and
  // weights come from memory: as slow as a layer in float32 products (3x3 at 1256 x
  // 389 with every tile out of range 1.5 to 1.6 ms, 1.46 ms by the kernel that this one
  // replaced), and rare.
  const f32x4* rows = reinterpret_cast<const f32x4*>(wpk + Cfg::frag_bytes);
  auto float_tile = [&]() {
    const int* flag = reinterpret_cast<const int*>(wpk + Cfg::flag_off);
    const float* scale = reinterpret_cast<const float*>(rows) + lrow;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[m][t] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
    for (int q = 0; q < Cfg::NQ; ++q) {
      int tap, c0;
      split_step<Cfg>(q, lgrp, &tap, &c0);
      const bool ok = c0 >= 0;
      f32x4 xv[MT][2];
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int hi = min(h0 + MT * wave + m + (ok ? tap / Cfg::KW : 0), Hin - 1);
        const int wi = min(w0 + lrow + (ok ? tap % Cfg::KW : 0), Win - 1);
        const f32x4* src = reinterpret_cast<const f32x4*>(x + ((long)hi * Win + wi) * Cs + (ok ? c0 : 0));
        xv[m][0] = src[0];
        xv[m][1] = src[1];
        if (!ok) xv[m][0] = xv[m][1] = f32x4{0.f, 0.f, 0.f, 0.f};
      }
      const int ql = q - Cfg::FULL * Cfg::taps;
#pragma unroll 1
      for (int t = 0; t < NT; ++t) {
        float v[8];
        if (ql < 0) {
          const u32x4* p = reinterpret_cast<const u32x4*>(wpk + (long)(q * NT + t) * 2048) + lane;
          const u32x4 p0 = p[0], p1 = p[64];
          if (flag[t] & kWide) {  // (uniform)
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = __uint_as_float(e < 4 ? p0[e & 3] : p1[e & 3]);
          } else {
            const f16x8 h = __builtin_bit_cast(f16x8, p0), l = __builtin_bit_cast(f16x8, p1);
            const float s = scale[16 * t] * 0x1p-14f;
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = fmaf((float)l[e], 1.f / kLowUnit, (float)h[e]) * s;
          }
        } else {
          const bf16x8* p =
              reinterpret_cast<const bf16x8*>(wpk + (long)Cfg::FULL * Cfg::taps * Cfg::w2 + (long)(ql * NT + t) * 3072) + lane;
          const bf16x8 h = p[0], mid = p[64], l = p[128];
          const float s = scale[16 * t];
#pragma unroll
          for (int e = 0; e < 8; ++e) v[e] = ((float)h[e] + (float)mid[e] + (float)l[e]) * s;
        }
#pragma unroll
        for (int tt = 0; tt < NT; ++tt)  // (the accumulators' index is a constant)
          if (tt == t) {
#pragma unroll
            for (int m = 0; m < MT; ++m)
#pragma unroll
              for (int e = 0; e < 8; ++e)
                acc[m][tt] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[e], xv[m][e >> 2][e & 3], acc[m][tt], 0, 0, 0);
          }
      }
    }
  };
  if (again) float_tile();

  // Epilogue: row scale, bias, tanh, four channels of one pixel per lane and
  // store (16 bytes).  Padding channels are stored as zeros (an infinite input
  // times their zero weights is NaN).
  __builtin_amdgcn_sched_barrier(0);  // (its loads stay behind the last step: registers)
  f32x4 rs[NT], bn[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    rs[t] = rows[4 * t + lgrp];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int n = 16 * t + 4 * lgrp + e;
      bn[t][e] = (n < K && bias) ? bias[n] : 0.f;
    }
  }
  if (again) {  // (in float32 products the scales are taken with the weights)
#pragma unroll
    for (int t = 0; t < NT; ++t) rs[t] = f32x4{1.f, 1.f, 1.f, 1.f};
  }
  auto epilogue = [&](auto f) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int ho = h0 + MT * wave + m, wo = w0 + lrow;
      if (ho >= Ho || wo >= Wo) continue;
      float* row = y + ((long)ho * Wo + wo) * Cs;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int n0 = 16 * t + 4 * lgrp;
        f32x4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = f(fmaf(acc[m][t][e], rs[t][e], bn[t][e]));
        if (16 * t + 16 > K) {  // (uniform) the tile that holds padding channels
#pragma unroll
          for (int e = 0; e < 4; ++e) v[e] = n0 + e < K ? v[e] : 0.f;
        }
        if (n0 < Cs) *reinterpret_cast<f32x4*>(row + n0) = v;
      }
    }
  };
  if (act)
    epilogue([](float v) { return tanh_fast(v); });
  else
    epilogue([](float v) { return v; });
}

// Calls f with the configuration of a supported layer; false if there is none.
template <typename F>
static bool with_split_cfg(int K, int C, int KH, int KW, F&& f) {
  const int cs = feature_stride(C), nt = (K + 15) / 16;
  if (feature_stride(K) != cs) return false;
  if (cs == 104 && nt == 7 && KH == 3 && KW == 3) f(SplitCfg<3, 3, 13, 7>{});
  else if (cs == 104 && nt == 7 && KH == 2 && KW == 2) f(SplitCfg<2, 2, 13, 7>{});
  else if (cs == 64 && nt == 4 && KH == 3 && KW == 3) f(SplitCfg<3, 3, 8, 4>{});
  else return false;
  return true;
}

bool split_supported(int K, int C, int KH, int KW) {
  return with_split_cfg(K, C, KH, KW, [](auto) {});
}

size_t split_packed_bytes(int K, int C, int KH, int KW) {
  size_t n = 0;
  with_split_cfg(K, C, KH, KW, [&](auto cfg) {
    using Cfg = decltype(cfg);
    n = Cfg::packed_bytes;
  });
  return n;
}

void split_pack(const float* w, int K, int C, int KH, int KW, int adj, void* packed, hipStream_t st) {
  with_split_cfg(K, C, KH, KW, [&](auto cfg) {
    using Cfg = decltype(cfg);
    k_pack_split<Cfg><<<dim3(Cfg::NT, kPackShares), 256, 0, st>>>(w, K, C, adj, (unsigned char*)packed);
  });
}

void split_launch(const float* x, int H, int W, int C, const void* packed, const float* b, int K, int KH, int KW,
                  int act, float* y, hipStream_t st) {
  const int Ho = H - KH + 1, Wo = W - KW + 1;
  auto launch = [&](auto cfg) {
    using Cfg = decltype(cfg);
    const auto kern = k_conv_split<Cfg>;
    const int tx = (int)ceil_div(Wo, Cfg::TW), tiles = tx * (int)ceil_div(Ho, Cfg::TH);
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::lds_bytes);
    kern<<<8 * ((tiles + 7) / 8), Cfg::threads, Cfg::lds_bytes, st>>>(x, H, W, (const unsigned char*)packed, b, K, act,
                                                                     y, Ho, Wo, tx, tiles);
  };
  with_split_cfg(K, C, KH, KW, [&](auto cfg) {
    using Cfg = decltype(cfg);
    using Small = SplitCfg<Cfg::KH, Cfg::KW, Cfg::CG, Cfg::NT, 1>;
    // Tiles of four rows while they do not fill two workgroups per CU: the layer
    // then takes as long as one tile does (us, four rows / eight: 64 x 64 3x3
    // 24 / 33, 200 x 100 2x2 (325 tiles of four rows) 18 / 22; past that 325 x 245 2x2,
    // 1281 tiles of four rows or 651 of eight, 48 / 42).
    if ((long)ceil_div(Wo, Small::TW) * ceil_div(Ho, Small::TH) <= 2 * cu_count())
      launch(Small{});
    else
      launch(cfg);
  });
}

}  // namespace ccs
