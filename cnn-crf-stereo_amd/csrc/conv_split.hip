// float32 feature layers (fused valid convolution + bias + tanh) on the bf16
// matrix cores.
//
// gfx950 runs v_mfma_f32_16x16x32_bf16 at 16 times the rate of
// v_mfma_f32_16x16x4_f32.  Both operands are split exactly into three bfloat16
// terms, x = xh + xm + xl and w = wh + wm + wl (split3), and a product is formed
// from six of the nine partial products,
//   xh wh + (xh wm + xm wh) + (xm wm + xh wl + xl wh),
// each exact in the matrix core and accumulated in float32.  The three products
// left out (xm wl, xl wm, xl wl) are below 2^-26 |x w| together, under
// float32's own rounding of a single product.  A 32-deep reduction step is
// summed from zero and added to the accumulator once, so an output takes 30
// roundings at its own size (the float32 instruction took 225): the relative
// error of a layer against 64 bits is 1.2e-7 (3x3) and 0.8e-7 (2x2), where
// v_mfma_f32_16x16x4_f32 left 5.4e-7 and 3.6e-7 (tanh off, 200 x 300 maps).
//
// k_conv_split: a workgroup of 4 waves computes a 16 x 16-pixel output tile for
// all output channels; a wave owns four rows of 16 pixels (MT = 4) times NT
// 16-channel tiles of accumulators.  The (16+KH-1) x (16+KW-1) input halo tile
// is staged in LDS one stage of four 8-channel groups at a time, split into its
// three planes on the way (324 pixels x 64 bytes x 3 = 61 KB for 3x3, so two
// workgroups share a CU and one's staging runs under the other's MFMAs).  A
// square tile has the least halo and wastes least at the edges of odd frames.
// The weights are packed in fragment order and read straight from L2 into
// registers, one channel tile ahead: per reduction step a wave issues
// 6 * 4 * NT MFMAs (168 for 100 channels, 2688 cycles) on 12 LDS fragments and
// 3 NT weight fragments, so the loop has no barrier and is bound by the matrix
// cores.  Measured (100 channels, against the float32-MFMA kernel it replaces):
// 3x3 at 1256 x 389 1456 -> 482 us (181 TFLOP/s of the layer, 1.09 PFLOP/s of
// bf16 products, the rate a large bf16 matrix product reaches on this card),
// 2x2 at 749 x 501 530 -> 217 us, 2x2 at 325 x 245 140 -> 65 us.  Reading the
// weights two tiles ahead, or adding a step's sums one tile later, changed
// nothing (476-485 us).
#include <type_traits>

#include "conv_split.hpp"

namespace ccs {

template <int KH_, int KW_, int CG_, int NT_>
struct SplitCfg {
  static constexpr int KH = KH_, KW = KW_, CG = CG_, NT = NT_;
  static constexpr int Cs = CG * 8, MT = 4, TS = 16;
  static constexpr int taps = KH * KW;
  static constexpr int FULL = CG / 4, REM = CG % 4;  // stages of four groups, groups of the last stage
  static constexpr int REM_NQ = (taps * REM + 3) / 4;
  static constexpr int NQ = FULL * taps + REM_NQ;  // 32-deep reduction steps
  static constexpr int AR = TS + KH - 1, AC = TS + KW - 1, NPX = AR * AC;
  static constexpr int plane = NPX * 64;  // bytes of one plane of a stage
  static constexpr int zero_off = 3 * plane;
  static constexpr int lds_bytes = zero_off + 16;
};

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

// Packed layout: [q][t][plane][lane][8], the fragment of channel tile t, with
// lane (lrow, lgrp) holding output channel 16 t + lrow.  One thread per lane.
template <class Cfg>
__global__ void k_pack_split(const float* __restrict__ w, int K, int C, int adj, bf16* __restrict__ out) {
  const int idx = blockIdx.x * blockDim.x + threadIdx.x;
  if (idx >= Cfg::NQ * Cfg::NT * 64) return;
  const int lane = idx & 63, t = (idx >> 6) % Cfg::NT, q = (idx >> 6) / Cfg::NT;
  const int n = 16 * t + (lane & 15);
  int tap, c0;
  split_step<Cfg>(q, lane >> 4, &tap, &c0);
  float v[8];
  bf16 p[3][8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int c = c0 + e;
    const int i = tap / Cfg::KW, j = tap % Cfg::KW;
    // adj: Wt[n][c] flipped, Wt[n][c][a][b] = w[c][n][KH-1-a][KW-1-b]
    v[e] = n < K && c0 >= 0 && c < C
               ? w[adj ? (((long)c * K + n) * Cfg::KH + i) * Cfg::KW + j
                       : (((long)n * C + c) * Cfg::KH + (Cfg::KH - 1 - i)) * Cfg::KW + (Cfg::KW - 1 - j)]
               : 0.f;
  }
  split3(v, p[0], p[1], p[2]);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    bf16x8 o;
#pragma unroll
    for (int e = 0; e < 8; ++e) o[e] = p[k][e];
    *reinterpret_cast<bf16x8*>(out + (((long)(q * Cfg::NT + t) * 3 + k) * 64 + lane) * 8) = o;
  }
}

// The four 16-byte groups of an LDS pixel are XOR-swizzled so that the reads of
// eight consecutive pixels land in eight distinct bank groups.
__device__ __forceinline__ int split_swz(int px, int g) { return g ^ ((px >> 1) & 3); }

template <class Cfg>
__global__ __launch_bounds__(256, 2) void k_conv_split(const float* __restrict__ x, int Hin, int Win,
                                                       const bf16* __restrict__ wpk, const float* __restrict__ bias,
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
  const int h0 = (tile / tiles_x) * Cfg::TS, w0 = (tile % tiles_x) * Cfg::TS;
  if (tid == 0) *reinterpret_cast<u32x4*>(lds + Cfg::zero_off) = u32x4{0u, 0u, 0u, 0u};

  // Stage of G groups from channel group cg0: unit (pixel, group) of eight
  // channels, all loads issued before the first is split and stored.
  // Coordinates are clamped to the map (those values feed only output pixels
  // past Ho x Wo).
  auto stage = [&](auto gc, int cg0) {
    constexpr int G = decltype(gc)::value;
    constexpr int NU = NPX * G, PER = (NU + 255) / 256;
    u32x4 r[PER][2];
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int v = min(tid + 256 * i, NU - 1);
      const int px = v / G, g = v % G;
      const int hi = min(h0 + px / AC, Hin - 1), wi = min(w0 + px % AC, Win - 1);
      const u32x4* src = reinterpret_cast<const u32x4*>(x + ((long)hi * Win + wi) * Cs + (cg0 + g) * 8);
      r[i][0] = src[0];
      r[i][1] = src[1];
    }
#pragma unroll
    for (int i = 0; i < PER; ++i) {
      const int v = tid + 256 * i;
      const int px = v / G, g = v % G;
      float f[8];
      bf16 p[3][8];
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] = __uint_as_float(r[i][e >> 2][e & 3]);
      split3(f, p[0], p[1], p[2]);
      const int off = G == 4 ? px * 64 + split_swz(px, g) * 16 : (px * G + g) * 16;
      if (v < NU) {
#pragma unroll
        for (int k = 0; k < 3; ++k) {
          bf16x8 o;
#pragma unroll
          for (int e = 0; e < 8; ++e) o[e] = p[k][e];
          *reinterpret_cast<bf16x8*>(lds + k * Cfg::plane + off) = o;
        }
      }
    }
  };

  // Accumulators start at the bias: lane (lrow, lgrp) holds pixel lrow of row
  // 4 wave + m and channels 16 t + 4 lgrp .. +3 (the weights are the A operand).
  f32x4 acc[MT][NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    f32x4 bn;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int n = 16 * t + 4 * lgrp + e;
      bn[e] = (n < K && bias) ? bias[n] : 0.f;
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[m][t] = bn;
  }

  // Weight fragments: three planes of a channel tile, 1 KB apart.  Fragment
  // f = q * NT + t; a read past the last one is clamped to it.
  const bf16x8* wl = reinterpret_cast<const bf16x8*>(wpk) + lane;
  auto load_w = [&](int f, bf16x8 (&b)[3]) {
    const bf16x8* p = wl + (long)min(f, Cfg::NQ * NT - 1) * 3 * 64;
#pragma unroll
    for (int k = 0; k < 3; ++k) b[k] = p[64 * k];
  };
  bf16x8 b0[3], b1[3];
  load_w(0, b0);

  // One reduction step: offs(m) is the LDS byte offset of row tile m's fragment
  // in plane 0, poff the plane distance (0 for the zero vector).
  auto step = [&](int q, auto&& offs, int poff) {
    bf16x8 a[3][MT];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int o = offs(m);
#pragma unroll
      for (int k = 0; k < 3; ++k) a[k][m] = *reinterpret_cast<const bf16x8*>(lds + o + k * poff);
    }
    // The step's products are summed from zero and added to the accumulators
    // once, in the vector unit: the matrix core's roundings then happen at the
    // size of 32 products, and only the additions at that of the whole sum.
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      load_w(q * NT + t + 1, b1);
      __builtin_amdgcn_sched_barrier(0);
      f32x4 cur[MT];
#pragma unroll
      for (int m = 0; m < MT; ++m)
        cur[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0[0], a[2][m], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      auto mm = [&](int kw, int kx) {
#pragma unroll
        for (int m = 0; m < MT; ++m)
          cur[m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(b0[kw], a[kx][m], cur[m], 0, 0, 0);
      };
      mm(2, 0);
      mm(1, 1);
      mm(0, 1);
      mm(1, 0);
      mm(0, 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < MT; ++m) acc[m][t] += cur[m];
#pragma unroll
      for (int k = 0; k < 3; ++k) b0[k] = b1[k];
    }
  };

#pragma unroll 1
  for (int s = 0; s < Cfg::FULL; ++s) {
    if (s > 0) __syncthreads();  // every wave has read the previous stage
    stage(std::integral_constant<int, 4>{}, 4 * s);
    __syncthreads();
#pragma unroll 1
    for (int tap = 0; tap < Cfg::taps; ++tap) {
      const int ti = tap / Cfg::KW, tj = tap % Cfg::KW;
      step(
          s * Cfg::taps + tap,
          [&](int m) {
            const int px = (4 * wave + m + ti) * AC + tj + lrow;
            return px * 64 + split_swz(px, lgrp) * 16;
          },
          Cfg::plane);
    }
  }
  if constexpr (Cfg::REM > 0) {
    __syncthreads();
    stage(std::integral_constant<int, Cfg::REM>{}, 4 * Cfg::FULL);
    __syncthreads();
#pragma unroll 1
    for (int ql = 0; ql < Cfg::REM_NQ; ++ql) {
      const int kg = 4 * ql + lgrp;
      const bool ok = kg < Cfg::taps * Cfg::REM;
      const int tap = ok ? kg / Cfg::REM : 0, g = ok ? kg % Cfg::REM : 0;
      const int ti = tap / Cfg::KW, tj = tap % Cfg::KW;
      step(
          Cfg::FULL * Cfg::taps + ql,
          [&](int m) {
            const int px = (4 * wave + m + ti) * AC + tj + lrow;
            return ok ? (px * Cfg::REM + g) * 16 : Cfg::zero_off;
          },
          ok ? Cfg::plane : 0);
    }
  }

  // Epilogue: tanh, four channels of one pixel per lane and store (16 bytes).
  // Padding channels are stored as zeros (an infinite input times their zero
  // weights is NaN).
  auto epilogue = [&](auto f) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int ho = h0 + 4 * wave + m, wo = w0 + lrow;
      if (ho >= Ho || wo >= Wo) continue;
      float* row = y + ((long)ho * Wo + wo) * Cs;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int n0 = 16 * t + 4 * lgrp;
        f32x4 v = {f(acc[m][t][0]), f(acc[m][t][1]), f(acc[m][t][2]), f(acc[m][t][3])};
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
    n = (size_t)Cfg::NQ * Cfg::NT * 3 * 1024;
  });
  return n;
}

void split_pack(const float* w, int K, int C, int KH, int KW, int adj, void* packed, hipStream_t st) {
  with_split_cfg(K, C, KH, KW, [&](auto cfg) {
    using Cfg = decltype(cfg);
    k_pack_split<Cfg><<<ceil_div((long)Cfg::NQ * Cfg::NT * 64, 256), 256, 0, st>>>(w, K, C, adj, (bf16*)packed);
  });
}

void split_launch(const float* x, int H, int W, int C, const void* packed, const float* b, int K, int KH, int KW,
                  int act, float* y, hipStream_t st) {
  with_split_cfg(K, C, KH, KW, [&](auto cfg) {
    using Cfg = decltype(cfg);
    const auto kern = k_conv_split<Cfg>;
    const int Ho = H - KH + 1, Wo = W - KW + 1;
    const int tx = (int)ceil_div(Wo, Cfg::TS), tiles = tx * (int)ceil_div(Ho, Cfg::TS);
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::lds_bytes);
    kern<<<8 * ((tiles + 7) / 8), 256, Cfg::lds_bytes, st>>>(x, H, W, (const bf16*)packed, b, K, act, y, Ho, Wo, tx,
                                                             tiles);
  });
}

}  // namespace ccs
