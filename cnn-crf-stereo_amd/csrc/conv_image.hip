// The image layer (1 to 3 planes, 3x3, valid convolution + bias + tanh) on the
// bf16 matrix cores.
//
// A pixel's C * 9 <= 27 taps fit one 32-deep reduction step.  Taps and weights
// are split exactly into three bfloat16 terms (split3), six of their nine products
// are summed from zero by v_mfma_f32_16x16x32_bf16 and the bias is added once, so
// an output takes 7 roundings where a chain of C * 9 fused multiply-adds took 27.
//
// k_conv_image_split: a wave takes 16 consecutive output pixels at a time, for all
// channels.  Its weight fragments stay in registers (NT tiles of 16 channels,
// split once per wave); lane (lrow, lgrp) gathers taps 8 lgrp .. +7 of pixel lrow
// straight from the planes, a tile ahead, and stores four channels of it.
//
// Bound by tanh (26 instructions per float32 value) beside the output's stores.
// k_conv_image runs C * 9 multiply-adds per value and two 16-byte LDS reads of
// weights per eight of them; with one plane those are few, and only large float32
// maps are faster here (a wave's weights take 3 us to load and split).  Measured,
// k_conv_image -> this (100 channels, us): float32 RGB 320 x 240 42 -> 23,
// 744 x 496 118 -> 51, 1256 x 389 154 -> 61, gray 320 x 240 18 -> 21, 744 x 496
// 56 -> 51, 1256 x 389 82 -> 65; bf16 RGB 744 x 496 74 -> 41, gray 37 -> 39.
// Four waves per SIMD's worth of workgroups took 86 instead of 65 us (RGB 744 x
// 496, with the profiler), three 70 us.
#include <type_traits>

#include "conv_split.hpp"

namespace ccs {

template <int C, int NT, typename TO>
__global__ __launch_bounds__(256, 2) void k_conv_image_split(const float* __restrict__ x, int Hin, int Win,
                                                             const float* __restrict__ w,
                                                             const float* __restrict__ bias, int K, int act,
                                                             TO* __restrict__ y, int Wo, long P, int Cs) {
  constexpr int T = C * 9;
  static_assert(T <= 32, "one reduction step");
  const int lane = threadIdx.x & 63, lrow = lane & 15, lgrp = lane >> 4;
  const long tiles = (P + 15) / 16, nw = (long)gridDim.x * 4;
  long tile = (long)blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  __shared__ __align__(16) float bs[16 * NT];
  for (int c = threadIdx.x; c < 16 * NT; c += 256) bs[c] = c < K && bias ? bias[c] : 0.f;
  __syncthreads();
  if (tile >= tiles) return;  // (uniform over the wave; no barrier follows)

  int off[8];  // of this lane's taps, from the output pixel's top left input
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int t = 8 * lgrp + e;
    off[e] = t < T ? (t / 9 * Hin + t % 9 / 3) * Win + t % 3 : 0;
  }
  float in[8], first;  // the taps, and the first plane's middle one
  auto load = [&](long tl) {
    const long p = min(tl * 16 + lrow, P - 1);
    const int ho = (int)(p / Wo), wo = (int)(p % Wo);
    const float* base = x + (long)ho * Win + wo;
#pragma unroll
    for (int e = 0; e < 8; ++e) in[e] = base[off[e]];
    if (sizeof(TO) == 4) first = base[Win + 1];
  };
  load(tile);

  bf16x8 wf[NT][3];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int n = 16 * t + lrow;
    float v[8];
    bf16 p[3][8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const int tap = 8 * lgrp + e;
      v[e] = tap < T && n < K ? w[(long)n * T + tap / 9 * 9 + 8 - tap % 9] : 0.f;
    }
    split3(v, p[0], p[1], p[2]);
#pragma unroll
    for (int k = 0; k < 3; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) wf[t][k][e] = p[k][e];
  }

  auto run = [&](auto f) {
    for (; tile < tiles; tile += nw) {
      const long p = tile * 16 + lrow;
      float v[8];
      bf16 s[3][8];
      bf16x8 a[3];
      // Half of a float32 map's pixels are multiplied negated (see kNegate).
      const unsigned neg = sizeof(TO) == 4 ? parity_sign(__float_as_uint(first)) : 0u;
      const float sg = with_sign(1.f, neg);
#pragma unroll
      for (int e = 0; e < 8; ++e) v[e] = 8 * lgrp + e < T ? with_sign(in[e], neg) : 0.f;
      split3(v, s[0], s[1], s[2]);
#pragma unroll
      for (int k = 0; k < 3; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) a[k][e] = s[k][e];
      load(min(tile + nw, tiles - 1));
      f32x4 c[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t)
        c[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][0], a[2], f32x4{0.f, 0.f, 0.f, 0.f}, 0, 0, 0);
      auto mm = [&](int kw, int kx) {
#pragma unroll
        for (int t = 0; t < NT; ++t) c[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[t][kw], a[kx], c[t], 0, 0, 0);
      };
      mm(2, 0);
      mm(1, 1);
      mm(0, 1);
      mm(1, 0);
      mm(0, 0);
      TO* row = y + p * Cs;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int n0 = 16 * t + 4 * lgrp;
        typedef __attribute__((ext_vector_type(4))) TO vec4;
        vec4 o;
        const f32x4 bn = *reinterpret_cast<const f32x4*>(bs + n0);
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (TO)(n0 + e < K ? f(fmaf(c[t][e], sg, bn[e])) : 0.f);
        if (p < P && n0 < Cs) *reinterpret_cast<vec4*>(row + n0) = o;
      }
    }
  };
  if (!act)
    run([](float v) { return v; });
  else if (sizeof(TO) == 2)
    run([](float v) { return tanh_for_bf16(v); });
  else
    run([](float v) { return tanh_fast(v); });
}

bool image_split_supported(int H, int W, int C, int K, int precision) {
  const bool worth = C > 1 || (precision == CCS_FP32 && (long)H * W >= 1l << 18);
  return C >= 1 && C <= 3 && ((K > 48 && K <= 64) || (K > 96 && K <= 112)) && worth;
}

void image_split_launch(const float* x, int H, int W, int C, const float* w, const float* b, int K, int act,
                        int precision, void* y, hipStream_t st) {
  const int Wo = W - 2;
  const long P = (long)(H - 2) * Wo, tiles = (P + 15) / 16;
  // As many workgroups as two waves per SIMD hold, with equal shares.
  const long rounds = (tiles + 2047) / 2048;
  const unsigned grid = ceil_div(tiles, 4 * rounds);
  auto go = [&](auto cc, auto nt, auto to) {
    k_conv_image_split<decltype(cc)::value, decltype(nt)::value, decltype(to)>
        <<<grid, 256, 0, st>>>(x, H, W, w, b, K, act, (decltype(to)*)y, Wo, P, feature_stride(K));
  };
  auto types = [&](auto cc, auto nt) { precision == CCS_BF16 ? go(cc, nt, bf16{}) : go(cc, nt, float{}); };
  auto widths = [&](auto cc) {
    K > 64 ? types(cc, std::integral_constant<int, 7>{}) : types(cc, std::integral_constant<int, 4>{});
  };
  if (C == 1) widths(std::integral_constant<int, 1>{});
  else if (C == 2) widths(std::integral_constant<int, 2>{});
  else widths(std::integral_constant<int, 3>{});
}

}  // namespace ccs
