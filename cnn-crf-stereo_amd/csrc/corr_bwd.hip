// Adjoint of the correlation volume on the bf16 matrix cores, for feature maps
// of 72 to 112 channels (with padding) and consecutive disparities.
//
//   out[p][c] = sum_k Gt[p][k] F[p + e_k][c],  e_k = e0 + s k,  s = -1 or 1
//   df0: F = f1, e_k = o_k,  Gt[p][k] = G[p][k]
//   df1: F = f0, e_k = -o_k, Gt[p][k] = G[p + e_k][k]
// (terms whose column leaves the image are zero).  For a run of pixels this is
// a banded product over a window of F's columns.  A chunk's window is staged in
// LDS transposed (channel-major, so a fragment is one 16-byte read), the columns
// in the order in which k grows with the column index R for every pixel:
//   R = k + shift(i),  shift(i) = i (s > 0) or MPW - 1 - i (s < 0)
// for pixel i of the workgroup's MPW.  G goes from memory straight into the
// fragments: a lane's eight reduction indices are eight consecutive k of one
// pixel (df0: two 16-byte loads), or one k of eight pixels in which 16 lanes
// hold 16 consecutive k (df1: eight 64-byte segments).
//
// G is float32 and is split exactly into three bfloat16 terms (split3): a
// product with a bfloat16 feature takes three products, each exact, with a
// float32 feature (split into three planes at staging) the six that are not
// below 2^-26 of it.  float32 maps sum each 32-deep step from zero before they
// add it, as conv_split.hip does.  The result rows are channels (F is the A
// operand), so a lane stores four consecutive channels of a pixel.
//
// The kernel it replaces (v_mfma_f32_16x16x4_f32 on operands gathered from LDS
// one float at a time) took 7.39 ms for both maps at 1488 x 992, D = 256 in
// bf16; this one takes 1.52 ms, of which reading G costs 0.5 and staging 0.4
// (timed without them).  G (1.51 GB) and the maps at copy rate are 0.57 ms; both
// maps of a row run on the same XCD one after the other, so that they share G
// through its L2.  64-disparity chunks with three workgroups per CU: 2.27 ms.
#include <type_traits>

#include "conv_split.hpp"
#include "corr_bwd.hpp"

namespace ccs {

template <typename T>
struct CorrBwdCfg;
template <>
struct CorrBwdCfg<bf16> {  // 4 waves of 32 pixels, 59 KB: two workgroups per CU
  static constexpr int WAVES = 4, MT = 2, KC = 128, PLANES = 1;
};
template <>
struct CorrBwdCfg<float> {  // 8 waves of 16 pixels, 145 KB
  static constexpr int WAVES = 8, MT = 1, KC = 64, PLANES = 3;
};

constexpr int kCorrNT = 7;  // channel tiles

template <typename T>
struct CorrBwdTile : CorrBwdCfg<T> {
  using B = CorrBwdCfg<T>;
  static constexpr int PW = 16 * B::MT, MPW = PW * B::WAVES, THREADS = 64 * B::WAVES;
  static constexpr int STEPS = (PW - 1 + B::KC + 31) / 32;  // 32-deep steps of a full chunk
  static constexpr int COLS = MPW - PW + 32 * STEPS;        // staged columns
  static constexpr int PITCH = COLS + 8;                    // elements; an odd multiple of 16 bytes
  static constexpr int plane = 16 * kCorrNT * PITCH * 2;
  static constexpr int lds_bytes = plane * B::PLANES;
  static_assert((PITCH * 2 / 16) % 2 == 1, "the fragment rows start on distinct bank groups");
};

// Exact three-term split of eight values.  The guards of split3 only run where
// a value needs them.
__device__ __forceinline__ void split_frag(const float (&x)[8], bf16x8& h, bf16x8& m, bf16x8& l) {
  float mx = 0.f;
#pragma unroll
  for (int e = 0; e < 8; ++e) mx = fmaxf(mx, fabsf(x[e]));
  float s = 0.f;  // NaN if one of them is
#pragma unroll
  for (int e = 0; e < 8; ++e) s += x[e];
  bf16 p[3][8];
  if (__any(!(mx < 1e38f) || s != s)) {
    split3(x, p[0], p[1], p[2]);
  } else {
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      p[0][e] = (bf16)x[e];
      const float r = x[e] - (float)p[0][e];
      p[1][e] = (bf16)r;
      p[2][e] = (bf16)(r - (float)p[1][e]);
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    h[e] = p[0][e];
    m[e] = p[1][e];
    l[e] = p[2][e];
  }
}

template <typename T>
__global__ __launch_bounds__(CorrBwdTile<T>::THREADS, 2) void k_corr_bwd_split(CorrBwdArgs a) {
  using Cfg = CorrBwdTile<T>;
  constexpr int MT = Cfg::MT, PW = Cfg::PW, MPW = Cfg::MPW, PITCH = Cfg::PITCH, COLS = Cfg::COLS, NT = kCorrNT;
  constexpr bool kF32 = sizeof(T) == 4;
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lrow = lane & 15, lgrp = lane >> 4;
  // Blocks b and b + 8 share an XCD: a row's blocks (both maps' tiles) follow
  // one another there.
  const int bpr = 2 * a.tiles;
  const int local = blockIdx.x >> 3;
  const int h = (blockIdx.x & 7) + 8 * (local / bpr);
  if (h >= a.H) return;  // (uniform) the grid is rounded up to 8 rows
  const int sub = local % bpr;
  const bool gather = sub >= a.tiles;  // df1
  const int P0 = (sub - (gather ? a.tiles : 0)) * MPW;
  const int W = a.W, D = a.D, Cs = a.Cs;
  const int s = gather ? -a.ostep : a.ostep, e0 = gather ? -a.o0 : a.o0;
  const long rowpix = (long)h * W;
  const T* frow = (const T*)(gather ? a.f0 : a.f1) + rowpix * Cs;
  const float* grow = a.G + rowpix * D;

  // Half of a float32 map's rows are multiplied negated (see kNegate): a sign from
  // the first pixel's features.  A bfloat16 result is rounded at 2^-9 of itself, to
  // nearest, which hides an offset of 1e-7 also in a sum over a frame (and the sign cost
  // 1361 -> 1610 us there).
  unsigned neg = 0;
  if constexpr (kF32) {
    const u32x4 v = *reinterpret_cast<const u32x4*>((const T*)a.f0 + rowpix * Cs);
    neg = parity_sign(__builtin_amdgcn_readfirstlane(v[0] ^ v[1] ^ v[2] ^ v[3]));
  }
  const float sg = with_sign(1.f, neg);

  // Rows Cs .. 112 of the planes stay zero.
  for (int v = tid; v < Cfg::PLANES * (16 * NT - Cs) * (PITCH / 8); v += Cfg::THREADS) {
    const int pl = v / ((16 * NT - Cs) * (PITCH / 8)), w = v % ((16 * NT - Cs) * (PITCH / 8));
    *reinterpret_cast<u32x4*>(lds + pl * Cfg::plane + (Cs * (PITCH / 8) + w) * 16) = u32x4{0u, 0u, 0u, 0u};
  }

  // Columns R = 0 .. COLS-1 of the chunk that starts at disparity kc, four
  // columns of one channel group per unit.
  auto stage = [&](int kc, int kn) {
    constexpr int VE = 16 / (int)sizeof(T);
    const int groups = Cs / VE, last = MPW - 1 + kn;  // columns past `last` are never multiplied by a G entry
    const int col0 = s > 0 ? P0 + e0 + kc : P0 + MPW - 1 + e0 - kc;
    constexpr int QB = (COLS + 63) / 64;  // blocks of 16 column quads
    for (int v = tid; v < (groups + 3) / 4 * QB * 64; v += Cfg::THREADS) {
      // 16 lanes take 16 column quads of one group, the wave four groups: a
      // pixel is read 64 bytes at a time, and 16 lanes store 128 bytes in a row.
      const int b = v >> 6, q = b % QB * 16 + (v & 15), g = b / QB * 4 + ((v >> 4) & 3);
      if (g >= groups || 4 * q >= COLS) continue;
      u32x4 r[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int R = 4 * q + i, col = col0 + s * R;
        const bool ok = R < last && col >= 0 && col < W;
        const u32x4 val = *reinterpret_cast<const u32x4*>(frow + (long)(ok ? col : 0) * Cs + g * VE);
        r[i] = ok ? (kF32 ? val ^ neg : val) : u32x4{0u, 0u, 0u, 0u};
      }
      unsigned char* d = lds + (g * VE * PITCH + 4 * q) * 2;
      if constexpr (kF32) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float f[4];
          bf16 p[3][4];
#pragma unroll
          for (int i = 0; i < 4; ++i) f[i] = __uint_as_float(r[i][e]);
          split3(f, p[0], p[1], p[2]);
          typedef __attribute__((ext_vector_type(4))) __bf16 bf16x4;
#pragma unroll
          for (int k = 0; k < 3; ++k)
            *reinterpret_cast<bf16x4*>(d + k * Cfg::plane + e * PITCH * 2) =
                bf16x4{p[k][0], p[k][1], p[k][2], p[k][3]};
        }
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const unsigned sel = (e & 1) ? 0x07060302u : 0x05040100u;
          const u32x2 o = {__builtin_amdgcn_perm(r[1][e >> 1], r[0][e >> 1], sel),
                           __builtin_amdgcn_perm(r[3][e >> 1], r[2][e >> 1], sel)};
          *reinterpret_cast<u32x2*>(d + e * PITCH * 2) = o;
        }
      }
    }
  };

  // This lane's pixels and where their band starts in the wave's columns.
  const int bw = s > 0 ? PW * wave : MPW - PW - PW * wave;
  int pix[MT], sm[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    pix[mt] = P0 + PW * wave + 16 * mt + lrow;
    sm[mt] = s > 0 ? 16 * mt + lrow : PW - 1 - 16 * mt - lrow;
  }
  // The G entries of step st of the chunk (kc, kn): k = 32 st + 8 lgrp + j - sm.
  // The row of G is a buffer resource: an entry that does not exist is read
  // past its range, which gives zero.  In the inner steps every entry exists,
  // and a lane's eight are 16-byte loads (df0) or a fixed stride of D + s apart
  // (df1), one address for all.
  const __amdgpu_buffer_rsrc_t rG =
      __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(grow), (short)0, W * D * 4, 0x00020000);
  constexpr int kNone = (int)0x80000000;
  const int gstep = (s * D + 1) * 4;  // bytes between a lane's entries of df1
  auto load_g = [&](int kc, int kn, int st, float (&x)[MT][8]) {
    bool inner = st >= 1 && 32 * st + 32 <= kn;  // (uniform) every lane's eight k exist
    if (gather) {  // and so do the columns of the wave's 32
      const int c0 = (s > 0 ? P0 + e0 + kc : P0 + MPW - 1 + e0 - kc) + s * (bw + 32 * st), c1 = c0 + 31 * s;
      inner = inner && min(c0, c1) >= 0 && max(c0, c1) < W;
    }
#pragma unroll
    for (int mt = 0; mt < MT; ++mt) {
      const int k0 = 32 * st + 8 * lgrp - sm[mt];
      if (!gather) {
        const int off = (pix[mt] * D + kc + k0) * 4;
        if (inner) {
          const int v = pix[mt] < W ? off : kNone;
          const u32x4 p = __builtin_amdgcn_raw_buffer_load_b128(rG, v, 0, 0);
          const u32x4 q = __builtin_amdgcn_raw_buffer_load_b128(rG, v, 16, 0);
#pragma unroll
          for (int j = 0; j < 8; ++j) x[mt][j] = __uint_as_float(j < 4 ? p[j & 3] : q[j & 3]);
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const bool ok = pix[mt] < W && k0 + j >= 0 && k0 + j < kn;
            x[mt][j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rG, ok ? off + 4 * j : kNone, 0, 0));
          }
        }
      } else {
        const int col0 = pix[mt] + e0 + s * (kc + k0);
        const int off = (col0 * D + kc + k0) * 4;
        if (inner) {
          const int v = gstep >= 0 ? off : off + 7 * gstep;
#pragma unroll
          for (int j = 0; j < 8; ++j)
            x[mt][j] = __uint_as_float(
                __builtin_amdgcn_raw_buffer_load_b32(rG, v, gstep >= 0 ? j * gstep : (j - 7) * gstep, 0));
        } else {
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int col = col0 + s * j;
            const bool ok = pix[mt] < W && k0 + j >= 0 && k0 + j < kn && col >= 0 && col < W;
            x[mt][j] =
                __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rG, ok ? off + j * gstep : kNone, 0, 0));
          }
        }
      }
    }
  };

  f32x4 acc[MT][NT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[mt][t] = f32x4{0.f, 0.f, 0.f, 0.f};

  for (int kc = 0; kc < D; kc += Cfg::KC) {
    const int kn = min(Cfg::KC, D - kc);
    const int steps = (PW - 1 + kn + 31) / 32;
    float x[MT][8];
    load_g(kc, kn, 0, x);
    __syncthreads();  // the previous chunk's columns are read
    stage(kc, kn);
    __syncthreads();
#pragma unroll 1
    for (int st = 0; st < steps; ++st) {
      bf16x8 g[3][MT];
#pragma unroll
      for (int mt = 0; mt < MT; ++mt) split_frag(x[mt], g[0][mt], g[1][mt], g[2][mt]);
      if (st + 1 < steps) load_g(kc, kn, st + 1, x);  // in flight under the MFMAs
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const unsigned char* fp = lds + ((16 * t + lrow) * PITCH + bw + 32 * st + 8 * lgrp) * 2;
        bf16x8 f[Cfg::PLANES];
#pragma unroll
        for (int k = 0; k < Cfg::PLANES; ++k) f[k] = *reinterpret_cast<const bf16x8*>(fp + k * Cfg::plane);
#pragma unroll
        for (int mt = 0; mt < MT; ++mt) {
          f32x4 c = kF32 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[mt][t];
          auto mm = [&](int kf, int kg) { c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[kf], g[kg][mt], c, 0, 0, 0); };
          if constexpr (kF32) {
            mm(0, 2);
            mm(Cfg::PLANES - 1, 0);
            mm(Cfg::PLANES / 2, 1);
            mm(0, 1);
            mm(Cfg::PLANES / 2, 0);
            mm(0, 0);
            acc[mt][t] += c;
          } else {
            mm(0, 2);
            mm(0, 1);
            mm(0, 0);
            acc[mt][t] = c;
          }
        }
      }
    }
  }
  T* out = (T*)(gather ? a.df1 : a.df0) + rowpix * Cs;
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    if (pix[mt] >= W) continue;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int c = 16 * t + 4 * lgrp;
      typedef __attribute__((ext_vector_type(4))) T vec4;
      const f32x4 v = kF32 ? acc[mt][t] * sg : acc[mt][t];
      if (c < Cs) *reinterpret_cast<vec4*>(out + (long)pix[mt] * Cs + c) = __builtin_convertvector(v, vec4);
    }
  }
}

// A row of G is addressed with 32-bit byte offsets, also a tile past its end.
bool corr_bwd_split_supported(int Cs, int W, int D, int ostep) {
  return Cs > 64 && Cs <= 16 * kCorrNT && (ostep == 1 || ostep == -1) && ((long)W + 1024) * D <= 0x7fffffffL / 4;
}

template <typename T>
static void launch(CorrBwdArgs a, hipStream_t st) {
  using Cfg = CorrBwdTile<T>;
  const auto kern = k_corr_bwd_split<T>;
  a.tiles = (int)ceil_div(a.W, Cfg::MPW);
  (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::lds_bytes);
  const unsigned blocks = 8u * (unsigned)(2 * a.tiles) * ceil_div(a.H, 8);
  kern<<<blocks, Cfg::THREADS, Cfg::lds_bytes, st>>>(a);
}

void corr_bwd_split(const CorrBwdArgs& a, int precision, hipStream_t st) {
  if (precision == CCS_BF16) launch<bf16>(a, st);
  else launch<float>(a, st);
}

}  // namespace ccs
