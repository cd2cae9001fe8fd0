// float32 convolution layers on the 16-bit matrix cores (conv_split.hip).
#pragma once

#include "common.hpp"

namespace ccs {

// Whether a KH x KW layer from Cs_in = feature_stride(C) to K channels has a
// split kernel: the 100-channel layers (3x3 and 2x2) and the 64-channel 3x3 one.
bool split_supported(int K, int C, int KH, int KW);
size_t split_packed_bytes(int K, int C, int KH, int KW);
// adj: the filters of the input gradient, w holding C x K x KH x KW.
void split_pack(const float* w, int K, int C, int KH, int KW, int adj, void* packed, hipStream_t st);
void split_launch(const float* x, int H, int W, int C, const void* packed, const float* b, int K, int KH, int KW,
                  int act, float* y, hipStream_t st);

// The image layer (C planes, 3x3) of K channels (conv_image.hip).
bool image_split_supported(int H, int W, int C, int K, int precision);
void image_split_launch(const float* x, int H, int W, int C, const float* w, const float* b, int K, int act,
                        int precision, void* y, hipStream_t st);

// Input gradient of a layer with filters w (K x C x KH x KW) on the MFMA
// forward kernels: dx (C channels) = true convolution of the padded dz (H x W,
// K channels) with Wt[c][k][a][b] = w[k][c][KH-1-a][KW-1-b].  *done is false
// (and nothing is queued) where the shape has no MFMA kernel.  (conv.hip)
int conv_input_gradient(ccs_handle_t h, const void* dz, int H, int W, int K, const float* w, int C, int KH, int KW,
                        int precision, void* dx, bool* done);

// x = h + m + l in bfloat16, exactly for every finite float32 down to l's
// underflow: h is x rounded to nearest, m the residual x - h rounded to nearest
// (|m| <= 2^-9 |x|), l what is left (at most 6 significant bits).  A value that
// would round to infinity is clamped first; an infinity or a NaN goes to l
// alone (h = m = 0), so that a product with a split finite y, which takes
// l only with y's h, keeps its sign or its NaN.
template <int N>
__device__ __forceinline__ void split3(const float (&x)[N], bf16 (&h)[N], bf16 (&m)[N], bf16 (&l)[N]) {
  constexpr float kMaxBf16 = 3.38953139e38f;
#pragma unroll
  for (int e = 0; e < N; ++e) {
    const bool fin = (__float_as_uint(x[e]) & 0x7fffffffu) < 0x7f800000u;
    const float v = fin ? x[e] : 0.f;
    h[e] = (bf16)__builtin_amdgcn_fmed3f(v, -kMaxBf16, kMaxBf16);
    const float r = v - (float)h[e];
    m[e] = (bf16)r;
    l[e] = (bf16)(fin ? r - (float)m[e] : x[e]);
  }
}

typedef __attribute__((ext_vector_type(8))) _Float16 f16x8;

// A block's biased exponent from its largest |x| bits (from 29, so that the
// factors below are normal numbers: smaller blocks keep a share of the bits).
__device__ __forceinline__ int split_exp(unsigned mx) { return max((int)(mx >> 23), 29); }
// s, and 2^-28 / s: what a sum of products of two split blocks takes back, but
// for the other block's own scale 2^(eb - 127).
__device__ __forceinline__ float split_scale(int eb) { return __uint_as_float((unsigned)(268 - eb) << 23); }
__device__ __forceinline__ float split_unscale(int eb) { return __uint_as_float((unsigned)(eb - 28) << 23); }

// The matrix unit rounds its 16-bit products' sums down, whatever their sign: an
// output's error is small but always of one sign, and sums over a map's pixels (the
// gradients of earlier layers and of biases) gather it.  So one operand is negated
// for half of the pixels, rows or segments, and the sum is negated back where it is
// added up in the vector unit, which rounds to nearest: over a map the errors
// cancel.  Which half, the bits of an input value decide (parity_sign), so that equal
// inputs give equal outputs wherever they lie.  Six 3x3 layers' bias gradients from exact inputs (512 x 256) were off by
// 1.0e-6 to 2.0e-6 without it and are by 0.7e-7 to 0.9e-7 with it, at the same
// speed (v_mfma_f32_16x16x4_f32: 0.8e-7 to 1.1e-7).  kNegate is a float's sign bit.
constexpr unsigned kNegate = 0x80000000u;
__device__ __forceinline__ float with_sign(float x, unsigned sign) {  // x, negated by sign = kNegate
  return __uint_as_float(__float_as_uint(x) ^ sign);
}
// A sign from a value's bits: as good as a random one over a map, and the same wherever
// the value lies in it.
__device__ __forceinline__ unsigned parity_sign(unsigned bits) { return (unsigned)__popc(bits) << 31; }

// x s = h + l / kLowUnit in float16, for a power of two s that takes the largest |x| of
// a block to [2^14, 2^15): h is x s rounded to nearest, l the rest, scaled up to h's size
// and rounded to nearest.  (float16's subnormals are exact in the matrix core.)  What is
// left out is at most 2^-24 |x| down to 2^-16 of the block's largest and 2^-22 |x| down
// to 2^-29; with the rest in h's own unit it is a subnormal number below 2^-15 of the
// largest, and lost below 2^-39.  The products with a low term are summed apart from
// those without.  No value of the block may be infinite.
constexpr float kLowUnit = 4096.f;
__device__ __forceinline__ void split_value(float x, float s, _Float16& h, _Float16& l) {
  const float v = x * s;
  h = (_Float16)v;
  l = (_Float16)fmaf((float)h, -kLowUnit, v * kLowUnit);
}
__device__ __forceinline__ void split_pair(const float (&x)[8], float s, f16x8& h, f16x8& l) {
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    _Float16 a, b;
    split_value(x[e], s, a, b);
    h[e] = a;
    l[e] = b;
  }
}

// What a pair leaves out of a value below 2^-29 of its block's largest is 2^-52 of
// that largest, and the low products that are dropped are 2^-50 of the largest product.
// That is nothing beside the largest value's own product, unless this meets a zero or
// a very small factor: where all factors of a sum are within 2^-22 of their largest
// (even), 32 such values leave out 2^-23 of the sum's terms at most.  So a sum needs other
// products than the pairs' only where one side has values that far apart and the other
// is uneven.
//
// BlockRange collects what tells: the largest |x| of a block, the smallest (as ordered
// bits, one instruction per two values each; a NaN is passed over: both its terms
// are NaN), and the smallest that is not 0 (as 2 |x| - 2, which makes 0 the largest).
struct BlockRange {
  float above = 0.f, least = __builtin_huge_valf();
  unsigned below = ~0u;
  __device__ __forceinline__ void add_largest(float x, float y) {
    asm("v_max3_f32 %0, |%1|, |%2|, %0" : "+v"(above) : "v"(x), "v"(y));
  }
  __device__ __forceinline__ void add_least(float x, float y) {
    asm("v_min3_f32 %0, |%1|, |%2|, %0" : "+v"(least) : "v"(x), "v"(y));
  }
  __device__ __forceinline__ void add_nonzero(float x, float y) {
    below = min(below, min((__float_as_uint(x) << 1) - 2u, (__float_as_uint(y) << 1) - 2u));
  }
  __device__ __forceinline__ unsigned largest() const { return __float_as_uint(above); }
  // Sums of products may leave float32's range before their scales are taken back
  // (from 2^115), or a value is infinite.
  __device__ __forceinline__ bool huge(unsigned from = 242u << 23) const { return largest() >= from; }
  // A value that is not 0 is below 2^-29 of the block's largest; eb: its split_exp.
  __device__ __forceinline__ bool apart(int eb) const { return below < (unsigned)(eb - 29) << 24; }
  // A value, 0 or not, is below 2^-22 of the block's largest (its ordered bits).
  __device__ __forceinline__ bool uneven(unsigned block) const {
    return __float_as_int(least) < (int)block - (22 << 23);
  }
};

}  // namespace ccs
