// Weight gradient of the 100-channel layers on the 16-bit matrix cores:
//   dW[tap][k][c] = sum over output pixels p of dz[p][k] x[p + tap][c]
// for bfloat16 maps and float32 maps (two float16 terms per operand with a scale
// per channel and segment, three products summed from zero per segment, as
// conv_split.hip).
//
// k_dw_split: a workgroup takes one tap row i (its KW taps) and a chunk of
// SEG-pixel segments of output rows; each of its seven waves owns 16 channels of
// dz, KW x 7 tiles of 16 input channels.  The reduction runs over pixels, so a
// fragment is eight consecutive pixels of one channel: dz and the input row go
// to LDS transposed (channel-major, pixel-minor).  A lane stages four pixels of
// a 16-byte channel group and stores four pixels of a channel with one 8-byte
// write.  The input row is stored once: the fragment of tap j starts j pixels
// later, which is the same dwords moved by a v_alignbit each (j = 1) or by one
// dword (j = 2), the fifth dword read beside them.  (A copy of the row per tap,
// stored two bytes at a time, took 64 LDS writes per thread and segment.)
//
// Bound by the steps' LDS reads and, with float32 maps, by splitting them.
// Measured with the reduction and k_dz_pad (the kernels it replaced -> with the
// zeros past a row's end selected beside the loads, which waited for each segment's
// reads -> now): bf16 3x3 at 524 x 268 190 -> 112 -> 94 us, at 1488 x 992
// 1490 -> 949 -> 708 us; float32 3x3 at 524 x 268 473 -> 328 -> 263 us (301 with
// three bfloat16 terms and six products).  Two input halves per chunk on four-wave
// workgroups, two or three per CU, measured the same as one (110, 990, 357 us): they
// read dz twice as often.
//
// Blocks b and b + 8 share an XCD: the tap rows of a chunk, which read the same
// dz and overlapping inputs, are consecutive there.  The block's sums go to
// part[chunk][tap], added in a fixed order by k_dw_reduce.
#include <type_traits>

#include "conv_grad.hpp"
#include "conv_split.hpp"

namespace ccs {

template <typename T>
struct DwCfg {
  static constexpr bool kF32 = sizeof(T) == 4;
  static constexpr int PLANES = kF32 ? 2 : 1;
  static constexpr int SEG = kF32 ? 32 : 64;  // output pixels per segment
  static constexpr int NT = 7, CP = 16 * NT, THREADS = 64 * NT;  // channel tiles, one wave each for dz
  static constexpr int VE = 16 / (int)sizeof(T);                 // channels per 16-byte vector
  // Staging blocks of 64 units (four pixels of a 16-byte channel group): QL
  // pixel quads times GL groups; four blocks of dz and four of the input row.  The
  // pixels past the segment that the shifted taps read: bfloat16 a ninth block
  // with the input row's last quad, float32 two more pixels in its blocks (their
  // channel's scale must cover them).  Two blocks per wave at most.
  static constexpr int QL = SEG / 4, GL = 64 / QL, NU = 2, BLOCKS = kF32 ? 8 : 9;
  static_assert(4 * GL >= CP / VE && BLOCKS <= NU * NT, "the blocks cover the channels");
  static constexpr int PITCH = SEG + 8;         // pixels; an odd multiple of 16 bytes
  static constexpr int plane = CP * PITCH * 2;  // bytes
  static constexpr int scales = 2 * PLANES * plane;  // float32: a scale per channel of dz, then of the input
  static constexpr int buffer = scales + (kF32 ? 2 * CP * 4 : 0);
  static constexpr int lds_bytes = 2 * buffer;
};

template <typename T, int KW>
__global__ __launch_bounds__(DwCfg<T>::THREADS, 2) void k_dw_split(const T* __restrict__ x, int Win, int Csx,
                                                                   const T* __restrict__ dz, int zpitch, int Ho,
                                                                   int Wo, int Csk, int KH, int nch, int segs_per_row,
                                                                   long nseg, long spc, float* __restrict__ part) {
  using Cfg = DwCfg<T>;
  constexpr int PLANES = Cfg::PLANES, NT = Cfg::NT, CP = Cfg::CP, VE = Cfg::VE, PITCH = Cfg::PITCH, SEG = Cfg::SEG;
  extern __shared__ __align__(16) unsigned char lds[];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int lrow = lane & 15, lgrp = lane >> 4;
  const int local = blockIdx.x >> 3;
  const int ti = local % KH, chunk = local / KH * 8 + (blockIdx.x & 7);
  if (chunk >= nch) return;  // (uniform) the grid is rounded up to whole groups of 8 chunks
  const int k0 = 16 * wave;
  const long s0 = (long)chunk * spc;
  const long s1 = s0 + spc < nseg ? s0 + spc : nseg;
  for (int i = tid; i < Cfg::lds_bytes / 16; i += Cfg::THREADS)  // the pad channels stay zero
    reinterpret_cast<u32x4*>(lds)[i] = u32x4{0u, 0u, 0u, 0u};

  // This lane's units: block 0-3 dz, 4-7 the input row, 8 the input row's last
  // quad (block and kind are uniform over the wave).  16 (float32: 8) lanes take
  // consecutive quads of one group, so a pixel is read 64 (128) bytes at a time
  // and the stores of a channel are contiguous.
  u32x4 reg[Cfg::NU][4];
  u32x4 ext[Cfg::NU][2];  // float32: input pixels SEG, SEG + 1
  struct Unit {
    bool z, ok;
    int q, g;
  };
  auto unit = [&](int b) {
    Unit u;
    u.z = b < 4;
    u.q = b == 8 ? Cfg::QL : lane % Cfg::QL;
    u.g = b == 8 ? lane : (b & 3) * Cfg::GL + lane / Cfg::QL;
    u.ok = u.g < (u.z ? Csk : Csx) / VE;
    return u;
  };
  // The next segment to load, as an output row and its first pixel, and the first
  // pixel of the loaded one.  A pixel past its row is loaded from the row's start
  // and zeroed when it is stored: a select beside the load would wait for it.
  int wo_loaded = 0;
  int lho = (int)(s0 / segs_per_row), lseg = (int)(s0 % segs_per_row);
  auto load_next = [&]() {
    const int ho = lho, wo0 = lseg * SEG;
    wo_loaded = wo0;
#pragma unroll
    for (int n = 0; n < Cfg::NU; ++n) {
      const int b = wave + NT * n;
      if (b >= Cfg::BLOCKS) break;
      const Unit u = unit(b);
      const T* row = u.z ? dz + ((long)ho * zpitch + wo0) * Csk : x + ((long)(ho + ti) * Win + wo0) * Csx;
      const int cs = u.z ? Csk : Csx, left = (u.z ? Wo : Win) - wo0;  // pixels of the row from wo0 on
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int px = 4 * u.q + i;
        const bool ok = u.ok && px < left;
        reg[n][i] = *reinterpret_cast<const u32x4*>(row + (ok ? px * cs + u.g * VE : 0));
      }
      if constexpr (Cfg::kF32) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const bool ok = !u.z && u.ok && SEG + i < left;
          ext[n][i] = *reinterpret_cast<const u32x4*>(row + (ok ? (SEG + i) * cs + u.g * VE : 0));
        }
      }
    }
    if (++lseg == segs_per_row) {
      lseg = 0;
      ++lho;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int n = 0; n < Cfg::NU; ++n) {
      const int b = wave + NT * n;
      if (b >= Cfg::BLOCKS) break;
      const Unit u = unit(b);
      if (!Cfg::kF32 && !u.ok) continue;
      const int left = (u.z ? Wo : Win) - wo_loaded;
      if (left < SEG + 4) {  // (uniform) the row may end in this segment
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (4 * u.q + i >= left) reg[n][i] = u32x4{0u, 0u, 0u, 0u};
        if constexpr (Cfg::kF32) {
#pragma unroll
          for (int i = 0; i < 2; ++i)
            if (SEG + i >= left) ext[n][i] = u32x4{0u, 0u, 0u, 0u};
        }
      }
      unsigned char* d =
          lds + buf * Cfg::buffer + (u.z ? 0 : PLANES * Cfg::plane) + (u.g * VE * PITCH + 4 * u.q) * 2;
      if constexpr (Cfg::kF32) {
        // Four pixels and the two past the segment of four channels; the eight
        // lanes of a group agree on each channel's scale.
        unsigned mx[4], all = 0;
        auto bits = [&](int e, int i) { return i < 4 ? reg[n][i][e] : ext[n][i - 4][e]; };
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          mx[e] = 0;
#pragma unroll
          for (int i = 0; i < 6; ++i)
            if (i < 4 || !u.z) mx[e] = max(mx[e], bits(e, i) & 0x7fffffffu);
          all = max(all, mx[e]);
        }
        const bool finite = !__any(all >= 0x7f800000u);
        const unsigned neg = u.z && buf ? kNegate : 0u;  // every other segment's dz
        const unsigned scale0 = (268u << 23) + neg, unscale0 = u.z ? neg - (28u << 23) : 0u;
        f32x4 unscale;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          if (!finite) {
            mx[e] = 0;
#pragma unroll
            for (int i = 0; i < 6; ++i)
              if (i < 4 || !u.z) mx[e] = max(mx[e], finite_bits(__uint_as_float(bits(e, i))));
#pragma unroll
            for (int i = 0; i < 4; ++i)  // (a value that the scale does not reach)
              if ((reg[n][i][e] & 0x7fffffffu) >= 0x7f800000u) reg[n][i][e] ^= neg;
          }
          mx[e] = max(mx[e], (unsigned)__builtin_amdgcn_mov_dpp((int)mx[e], 0xb1, 0xf, 0xf, true));
          mx[e] = max(mx[e], (unsigned)__builtin_amdgcn_mov_dpp((int)mx[e], 0x4e, 0xf, 0xf, true));
          mx[e] = max(mx[e], (unsigned)__builtin_amdgcn_mov_dpp((int)mx[e], 0x141, 0xf, 0xf, true));  // row_half_mirror
          const int eb = split_exp(mx[e]);
          // split_scale and split_unscale (x's side: 2^(eb - 127)) with the sign,
          // which is carried through by sums modulo 2^32
          const float sc = __uint_as_float(scale0 - ((unsigned)eb << 23));
          unscale[e] = __uint_as_float(((unsigned)eb << 23) + unscale0);
          typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
          typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
          f16x4 hi, lo;
          f16x2 hx, lx;
#pragma unroll
          for (int i = 0; i < 6; ++i) {
            if (i >= 4 && u.z) break;
            const float f = __uint_as_float(bits(e, i));
            const bool fin = finite || (__float_as_uint(f) & 0x7fffffffu) < 0x7f800000u;
            const float v = fin ? f * sc : 0.f;
            const _Float16 h = (_Float16)v, l = (_Float16)(fin ? v - (float)h : f);
            if (i < 4) hi[i] = h, lo[i] = l;
            else hx[i - 4] = h, lx[i - 4] = l;
          }
          if (u.ok) {
            *reinterpret_cast<f16x4*>(d + e * PITCH * 2) = hi;
            *reinterpret_cast<f16x4*>(d + Cfg::plane + e * PITCH * 2) = lo;
            if (!u.z && u.q == Cfg::QL - 1) {  // (the next quad's first half)
              *reinterpret_cast<f16x2*>(d + (e * PITCH + 4) * 2) = hx;
              *reinterpret_cast<f16x2*>(d + Cfg::plane + (e * PITCH + 4) * 2) = lx;
            }
          }
        }
        if (u.ok && u.q == 0)
          *reinterpret_cast<f32x4*>(lds + buf * Cfg::buffer + Cfg::scales + ((u.z ? 0 : CP) + u.g * VE) * 4) = unscale;
      } else {
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          const unsigned sel = (e & 1) ? 0x07060302u : 0x05040100u;
          *reinterpret_cast<u32x2*>(d + e * PITCH * 2) =
              u32x2{__builtin_amdgcn_perm(reg[n][1][e >> 1], reg[n][0][e >> 1], sel),
                    __builtin_amdgcn_perm(reg[n][3][e >> 1], reg[n][2][e >> 1], sel)};
        }
      }
    }
  };

  f32x4 acc[KW][NT];
#pragma unroll
  for (int j = 0; j < KW; ++j)
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[j][t] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto multiply = [&](int buf) {
    const unsigned char* zb = lds + buf * Cfg::buffer;
    const unsigned char* xb = zb + PLANES * Cfg::plane;
    const float* scale = reinterpret_cast<const float*>(zb + Cfg::scales);  // (float32)
    f32x4 sz;
    if constexpr (Cfg::kF32) sz = *reinterpret_cast<const f32x4*>(scale + k0 + 4 * lgrp);
#pragma unroll
    for (int st = 0; st < SEG / 32; ++st) {
      const int off = (32 * st + 8 * lgrp) * 2;
      bf16x8 a[PLANES];
#pragma unroll
      for (int k = 0; k < PLANES; ++k)
        a[k] = *reinterpret_cast<const bf16x8*>(zb + k * Cfg::plane + (k0 + lrow) * PITCH * 2 + off);
      // Fragments of channel tile t: five dwords, read one tile ahead.
      u32x4 d[PLANES];
      unsigned d4[PLANES];
      float sx = 0.f;
      auto read_x = [&](int t) {
        if constexpr (Cfg::kF32) sx = scale[CP + 16 * t + lrow];
#pragma unroll
        for (int k = 0; k < PLANES; ++k) {
          const unsigned char* src = xb + k * Cfg::plane + (16 * t + lrow) * PITCH * 2 + off;
          d[k] = *reinterpret_cast<const u32x4*>(src);
          d4[k] = *reinterpret_cast<const unsigned*>(src + 16);
        }
      };
      read_x(0);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        bf16x8 b[PLANES][KW];
#pragma unroll
        for (int k = 0; k < PLANES; ++k) {
          // (the shifted fragments come from these registers, not from more reads
          // of LDS at odd dwords, which meet a quarter of the banks)
          asm("" : "+v"(d[k]));
          asm("" : "+v"(d4[k]));
          const u32x4 e = d[k];
          b[k][0] = __builtin_bit_cast(bf16x8, e);
          b[k][1] = __builtin_bit_cast(
              bf16x8, u32x4{__builtin_amdgcn_alignbit(e[1], e[0], 16), __builtin_amdgcn_alignbit(e[2], e[1], 16),
                            __builtin_amdgcn_alignbit(e[3], e[2], 16), __builtin_amdgcn_alignbit(d4[k], e[3], 16)});
          if constexpr (KW == 3) b[k][2] = __builtin_bit_cast(bf16x8, u32x4{e[1], e[2], e[3], d4[k]});
        }
        f32x4 both;  // the scales of this lane's four sums
        if constexpr (Cfg::kF32) both = sz * sx;
        if (t + 1 < NT) read_x(t + 1);
        __builtin_amdgcn_sched_barrier(0);
        f32x4 c[KW];
#pragma unroll
        for (int j = 0; j < KW; ++j) c[j] = Cfg::kF32 ? f32x4{0.f, 0.f, 0.f, 0.f} : acc[j][t];
        auto mm = [&](int ka, int kb) {
#pragma unroll
          for (int j = 0; j < KW; ++j) {
            if constexpr (Cfg::kF32)
              c[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[ka]),
                                                           __builtin_bit_cast(f16x8, b[kb][j]), c[j], 0, 0, 0);
            else
              c[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[ka], b[kb][j], c[j], 0, 0, 0);
          }
        };
        if constexpr (Cfg::kF32) {
          mm(PLANES - 1, 0);
          mm(0, PLANES - 1);
        }
        mm(0, 0);
#pragma unroll
        for (int j = 0; j < KW; ++j) {
          if constexpr (Cfg::kF32) {
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[j][t][e] = fmaf(c[j][e], both[e], acc[j][t][e]);
          } else {
            acc[j][t] = c[j];
          }
        }
      }
    }
  };

  __syncthreads();  // the zero fill is done
  if (s0 < s1) {
    load_next();
    store(0);
    if (s0 + 1 < s1) load_next();
  }
  __syncthreads();
  // Segment s is multiplied from buffer (s - s0) % 2 while the next one's
  // registers go into the other (whose readers finished before the barrier).
  // Waves w and w + 4 share a SIMD: with bf16 maps one stages while the other
  // multiplies (float32 maps would spill: 477 us).
  for (long s = s0; s < s1; ++s) {
    const int buf = (int)((s - s0) & 1);
    auto stage = [&]() {
      if (s + 1 < s1) {
        store(buf ^ 1);
        if (s + 2 < s1) load_next();
      }
    };
    if (Cfg::kF32 || wave < 4) stage();
    multiply(buf);
    if (!Cfg::kF32 && wave >= 4) stage();
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < KW; ++j) {
    float* out = part + ((long)chunk * KH * KW + ti * KW + j) * CP * CP;
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) out[(k0 + 4 * lgrp + e) * CP + 16 * t + lrow] = acc[j][t][e];
  }
}

bool dw_split_supported(int Csx, int Csk, int KW) {
  return Csx > 64 && Csk > 64 && Csx <= 112 && Csk <= 112 && (KW == 2 || KW == 3);
}

int dw_split_segment(int precision) { return precision == CCS_BF16 ? DwCfg<bf16>::SEG : DwCfg<float>::SEG; }

template <typename T>
static void launch(const DwArgs& a, int KH, int KW, hipStream_t st) {
  using Cfg = DwCfg<T>;
  const unsigned blocks = (unsigned)(8 * KH * ((a.nch + 7) / 8));
  auto go = [&](auto kwc) {
    const auto kern = k_dw_split<T, decltype(kwc)::value>;
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, Cfg::lds_bytes);
    kern<<<blocks, Cfg::THREADS, Cfg::lds_bytes, st>>>((const T*)a.x, a.Win, a.Csx, (const T*)a.dz, a.zpitch, a.Ho,
                                                      a.Wo, a.Csk, KH, a.nch, a.segs_per_row, a.nseg, a.spc, a.part);
  };
  if (KW == 3) go(std::integral_constant<int, 3>{});
  else go(std::integral_constant<int, 2>{});
}

void dw_split(const DwArgs& a, int precision, int KH, int KW, hipStream_t st) {
  if (precision == CCS_BF16) launch<bf16>(a, KH, KW, st);
  else launch<float>(a, KH, KW, st);
}

}  // namespace ccs
