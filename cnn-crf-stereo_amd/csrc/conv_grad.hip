// Weight gradient of the 100-channel layers on the 16-bit matrix cores:
//   dW[tap][k][c] = sum over output pixels p of dz[p][k] x[p + tap][c]
// for bfloat16 maps and float32 maps (two float16 terms per operand with a scale
// per channel and segment, three products in two sums from zero per segment, as
// conv_split.hip; a segment in which that does not do, see BlockRange, takes
// v_mfma_f32_16x16x4_f32 from memory after the others).
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
// three bfloat16 terms and six products), and 271 with both units and the range tests
// (850 where every segment goes to float32 products).  Two input halves per chunk on four-wave
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
  // float32: per buffer and wave the DwFlags of its units, then a bit per segment of the chunk
  static constexpr int flag_off = 2 * buffer, float_off = flag_off + 2 * 8 * 4;
  static constexpr int lds_bytes(long spc) { return kF32 ? float_off + (int)((spc + 127) / 128) * 16 : 2 * buffer; }
};

// What the channels of a segment's input (X) and dz (Z) have: values of 2^64 and more, with
// which the product of two channels' scales may be infinite; uneven() ones; apart() ones.
enum DwFlag { kUnevenX = 1, kUnevenZ = 2, kApartX = 4, kApartZ = 8, kHuge = 16 };

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
  for (int i = tid; i < Cfg::lds_bytes(spc) / 16; i += Cfg::THREADS)  // the pad channels stay zero
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
  // Stores the loaded segment s into a buffer.
  auto store = [&](int buf, long s) {
    int flags = 0;  // float32: the units' DwFlags (uniform over the wave)
#pragma unroll
    for (int n = 0; n < Cfg::NU; ++n) {
      const int b = wave + NT * n;
      if (b >= Cfg::BLOCKS) break;
      const Unit u = unit(b);
      if (!Cfg::kF32 && !u.ok) continue;
      const int left = (u.z ? Wo : Win) - wo_loaded;
      // Fills the pixels past the row's end, if it is in this segment (uniform).
      auto fill_end = [&](unsigned v) {
        if (left >= SEG + 4) return;
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (4 * u.q + i >= left) reg[n][i] = u32x4{v, v, v, v};
        if constexpr (Cfg::kF32) {
#pragma unroll
          for (int i = 0; i < 2; ++i)
            if (SEG + i >= left) ext[n][i] = u32x4{v, v, v, v};
        }
      };
      [[maybe_unused]] auto at = [&](int e, int i) {
        return __uint_as_float(i < 4 ? reg[n][i][e] : ext[n][i - 4][e]);
      };
      [[maybe_unused]] int eb[4];
      if constexpr (Cfg::kF32) {
        // Four pixels and the two past the segment of four channels; the eight
        // lanes of a group agree on each channel's scale.
        fill_end(0x7fc00000u);  // (a NaN, which the ranges pass over)
        unsigned long huge = 0, uneven = 0, apart = 0;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          BlockRange r;
#pragma unroll
          for (int i = 0; i < 6; i += 2) {
            if (i >= 4 && u.z) break;
            r.add_largest(at(e, i), at(e, i + 1));
            r.add_least(at(e, i), at(e, i + 1));
          }
          unsigned mx = r.largest();
          mx = max(mx, (unsigned)__builtin_amdgcn_mov_dpp((int)mx, 0xb1, 0xf, 0xf, true));
          mx = max(mx, (unsigned)__builtin_amdgcn_mov_dpp((int)mx, 0x4e, 0xf, 0xf, true));
          mx = max(mx, (unsigned)__builtin_amdgcn_mov_dpp((int)mx, 0x141, 0xf, 0xf, true));  // row_half_mirror
          eb[e] = split_exp(mx);
          huge |= __ballot(u.ok && r.huge(191u << 23));
          uneven |= __ballot(u.ok && r.uneven(mx));
        }
        if (uneven) {  // (uniform; a value that is apart is uneven too)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            BlockRange r;
#pragma unroll
            for (int i = 0; i < 6; i += 2) {
              if (i >= 4 && u.z) break;
              r.add_nonzero(at(e, i), at(e, i + 1));
            }
            apart |= __ballot(u.ok && r.apart(eb[e]));
          }
        }
        flags |= (huge ? kHuge : 0) | (uneven ? u.z ? kUnevenZ : kUnevenX : 0) | (apart ? u.z ? kApartZ : kApartX : 0);
      }
      fill_end(0u);
      unsigned char* d =
          lds + buf * Cfg::buffer + (u.z ? 0 : PLANES * Cfg::plane) + (u.g * VE * PITCH + 4 * u.q) * 2;
      if constexpr (Cfg::kF32) {
        const unsigned neg = u.z && (s & 1) ? kNegate : 0u;  // every other segment's dz
        const unsigned scale0 = (268u << 23) + neg, unscale0 = u.z ? neg - (28u << 23) : 0u;
        f32x4 unscale;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          // split_scale and split_unscale (x's side: 2^(eb - 127)) with the sign,
          // which is carried through by sums modulo 2^32
          const float sc = __uint_as_float(scale0 - ((unsigned)eb[e] << 23));
          unscale[e] = __uint_as_float(((unsigned)eb[e] << 23) + unscale0);
          typedef __attribute__((ext_vector_type(4))) _Float16 f16x4;
          typedef __attribute__((ext_vector_type(2))) _Float16 f16x2;
          f16x4 hi, lo;
          f16x2 hx, lx;
#pragma unroll
          for (int i = 0; i < 6; ++i) {
            if (i >= 4 && u.z) break;
            _Float16 h, l;
            split_value(at(e, i), sc, h, l);
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
    if constexpr (Cfg::kF32) {
      if (lane == 0) *reinterpret_cast<int*>(lds + Cfg::flag_off + (8 * buf + wave) * 4) = flags;
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
        f32x4 c[KW], low[KW];  // low (float32): the products with a low term
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
#pragma unroll
          for (int j = 0; j < KW; ++j) low[j] = c[j], c[j] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
        mm(0, 0);
#pragma unroll
        for (int j = 0; j < KW; ++j) {
          if constexpr (Cfg::kF32) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
              acc[j][t][e] = fmaf(fmaf(low[j][e], 1.f / kLowUnit, c[j][e]), both[e], acc[j][t][e]);
          } else {
            acc[j][t] = c[j];
          }
        }
      }
    }
  };

  auto failed = [&](int buf) {  // (behind the barrier)
    const u32x4* f = reinterpret_cast<const u32x4*>(lds + Cfg::flag_off + 8 * buf * 4);
    const u32x4 a = f[0], b = f[1];
    const int any = __builtin_amdgcn_readfirstlane(a[0] | a[1] | a[2] | a[3] | b[0] | b[1] | b[2]);
    return (any & kHuge) || ((any & kApartX) && (any & kUnevenZ)) || ((any & kApartZ) && (any & kUnevenX));
  };

  __syncthreads();  // the zero fill is done
  if (s0 < s1) {
    load_next();
    store(0, s0);
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
        store(buf ^ 1, s + 1);
        if (s + 2 < s1) load_next();
      }
    };
    if (Cfg::kF32 || wave < 4) stage();
    if constexpr (Cfg::kF32) {
      if (failed(buf)) {  // its products become zeros (a branch around multiply() spills)
        if (tid == 0) reinterpret_cast<unsigned*>(lds + Cfg::float_off)[(s - s0) >> 5] |= 1u << ((s - s0) & 31);
        for (int i = tid; i < Cfg::buffer / 16; i += Cfg::THREADS)
          reinterpret_cast<u32x4*>(lds + buf * Cfg::buffer)[i] = u32x4{0u, 0u, 0u, 0u};
        __syncthreads();
      }
    }
    multiply(buf);
    if (!Cfg::kF32 && wave >= 4) stage();
    __syncthreads();
  }
  if constexpr (Cfg::kF32) {
    // The segments left out, on v_mfma_f32_16x16x4_f32 with operands from memory (here,
    // where the staged values are dead: beside multiply() this spills).
    for (long w0 = s0; w0 < s1; w0 += 32) {
      unsigned bits = __builtin_amdgcn_readfirstlane(reinterpret_cast<unsigned*>(lds + Cfg::float_off)[(w0 - s0) >> 5]);
      for (; bits; bits &= bits - 1) {
        const long s = w0 + __builtin_ctz(bits);
        const int ho = (int)(s / segs_per_row), wo0 = (int)(s % segs_per_row) * SEG;
        const T* zrow = dz + ((long)ho * zpitch + wo0) * Csk;
        const T* xrow = x + ((long)(ho + ti) * Win + wo0) * Csx;
        const int left = min(SEG, Wo - wo0);
#pragma unroll 1
        for (int p0 = 0; p0 < left; p0 += 4) {
          // Past the row and the channels another value is loaded (no branches); those
          // channels' sums are not used.
          const int p = min(p0 + lgrp, left - 1);
          const bool in = p0 + lgrp < left;
          const float zv = in ? (float)zrow[p * Csk + min(k0 + lrow, Csk - 1)] : 0.f;
          float xv[KW][NT];
#pragma unroll
          for (int j = 0; j < KW; ++j)
#pragma unroll
            for (int t = 0; t < NT; ++t) xv[j][t] = (float)xrow[(p + j) * Csx + min(16 * t + lrow, Csx - 1)];
#pragma unroll
          for (int j = 0; j < KW; ++j)
#pragma unroll
            for (int t = 0; t < NT; ++t)
              acc[j][t] = __builtin_amdgcn_mfma_f32_16x16x4f32(zv, in ? xv[j][t] : 0.f, acc[j][t], 0, 0, 0);
        }
      }
    }
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
    const int lds = Cfg::lds_bytes(a.spc);
    (void)hipFuncSetAttribute((const void*)kern, hipFuncAttributeMaxDynamicSharedMemorySize, lds);
    kern<<<blocks, Cfg::THREADS, lds, st>>>((const T*)a.x, a.Win, a.Csx, (const T*)a.dz, a.zpitch, a.Ho,
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
