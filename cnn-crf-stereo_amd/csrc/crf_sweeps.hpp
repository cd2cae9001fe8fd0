// SlackProp CRF inference on MI355X: dual minorize-maximize over row and column
// chains of the 4-connected grid.
//
// The reference calls slack_prop_2D_alg from an un-vendored library
// (stereo/stereo.cpp:140-154, stereo/operators/slackprop.cpp:96-105); this file
// implements a restatement of that published method:
//
//   A = C                                   (row unaries; columns hold C - A)
//   repeat iters times:
//     rows:    g = minorant(A_row, wx_row);       A_row -= g
//     columns: g = minorant((C-A)_col, wy_col);   A_col += g
//   decode rows: label = argmin of the row min-marginals
//
// with the pairwise term w * rho(x_p - x_q), rho = 0 / L1 (0 < |d| < delta) /
// L2 (|d| >= delta).  minorant() is a tight, maximal modular minorant of one
// chain: a backward min-sum pass stores normalised messages Bh, then a forward
// pass keeps g_i = 1/4 (R_i + B_i) + excess_i at every node and passes the rest
// on.  The dual bound Phi_rows(A) + Phi_cols(C - A) never decreases; its float64
// bookkeeping (chain minima S, kept constants K) runs beside the float32 min-sum.
//
// The sweeps keep one state volume that alternates between the two halves'
// unaries: a row sweep reads A and stores B = C - (A - g), a column sweep reads
// B and stores A = (C - B) + g, so each reads one volume in each of its two
// passes and the cost volume only in its forward pass (4 volume passes per
// sweep instead of 3 for rows and 5 for columns).
//
// GPU mapping: one wavefront per chain (k_chain; with few chains two more waves
// move its data, k_line), label s = lane * LPL + j held in VGPRs,
// DPP wave_shr/wave_shl for the label neighbours and a DPP tree for the minimum
// over labels.  The volume streams through HBM once per pass (node i is D
// contiguous floats), backward messages go to a scratch volume (column sweeps
// of large volumes store every seg_len()-th one and recompute the rest), and the
// per-node minima go to LDS; their float64 sums are formed by wave scans after
// each pass.  The row decode runs its two message passes on two wavefronts at
// once, and two more waves take its decisions (k_decode4).
//
// This file holds the chain sweeps only.  It is compiled with -fno-honor-nans:
// the min/max trees then run as fused DPP instructions without NaN-quieting
// moves.  Costs must be finite or +inf; a NaN cost gives unspecified labels
// (never an out-of-range memory access: labels are only stored, and every
// address is computed from chain/node/lane indices).  The row minorant can
// flag NaN unaries per chain (ChainArgs::nan_flags) with a class test of every
// value it reads, which the host turns into a status code.
#pragma once

#include <type_traits>
#include <utility>

#include "crf_chain.hpp"

namespace ccs {

constexpr float kInfF = __builtin_huge_valf();
// Relative tolerance under which two decoded min-marginals count as tied.
#ifndef CCS_CRF_TIE_EPS
#define CCS_CRF_TIE_EPS 1e-5f
#endif
constexpr float kTieEps = CCS_CRF_TIE_EPS;

// Scheduling fence between a ring slot's read and its refill: memory, LDS and
// scalar instructions keep their side of it, VALU instructions may cross (they
// fill the DPP/permlane wait states of the neighbouring step).
constexpr int kSchedValu = 0x2;

// kNoWideStores: no chain kernel stores more than 64 bits per lane in one
// instruction.  A vector store of 96 or 128 bits reads its data VGPRs after
// issue, and hipcc (ROCm 7.2) for gfx950 was seen to place a VALU write of those
// VGPRs (a DPP min of the next step) directly behind such a store with no wait
// state; the D = 256 sweeps then stored partly overwritten data, varying from
// run to run.  With two 64-bit stores (kept apart by a compiler barrier, which
// stops them being merged back) the sweeps are deterministic and bit-identical
// between the column schemes.

template <int LPL>
constexpr int seg_len() {
  return seg_length(LPL);
}

template <int LPL>
struct Vec {
  float v[LPL];
};

// How the D labels lie in the wave's 64 * LPL places.  kFitFull: D == 64 * LPL.
// kFitLanes: D is a multiple of LPL, so a lane's labels all exist or none does:
// a node is one vector access per lane, as with kFitFull, and the lanes without
// labels only need +inf unaries (their messages are never stored and never
// reach a label).  kFitHalf: kFitLanes with labels in two of the wave's four rows
// only, whose minimum over the labels is five instructions shorter.  kFitAny:
// element-wise accesses and a mask per label.
enum { kFitAny = 0, kFitLanes = 1, kFitFull = 2, kFitHalf = 3 };

// Row sweeps with a message wave (SEG rows): the backward pass keeps every
// seg_len()-th message in the scratch volume, and a second wave of the
// workgroup recomputes each segment's messages from those checkpoints into an
// LDS ring of kRowRing segments, two segments ahead of the forward pass.  The
// ring holds a node's messages at a stride of 64 * LPL floats.
// Workgroup barrier that orders LDS accesses only: the waves wait for their
// own LDS operations (lgkmcnt) but keep their global loads in flight.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// A node's messages in the LDS ring (lane-major, LPL floats per lane; stores
// of at most 64 bits, as for global memory).
template <int LPL>
__device__ __forceinline__ void st_ring(float* p, int lane, const Vec<LPL>& x) {
  if constexpr (LPL == 4) {
    *reinterpret_cast<float2*>(p + lane * 4) = make_float2(x.v[0], x.v[1]);
    *reinterpret_cast<float2*>(p + lane * 4 + 2) = make_float2(x.v[2], x.v[3]);
  } else if constexpr (LPL == 2) {
    *reinterpret_cast<float2*>(p + lane * 2) = make_float2(x.v[0], x.v[1]);
  } else {
    p[lane] = x.v[0];
  }
}

template <int LPL>
__device__ __forceinline__ Vec<LPL> ld_ring(const float* p, int lane) {
  Vec<LPL> o;
  if constexpr (LPL == 4) {
    const float4 t = *reinterpret_cast<const float4*>(p + lane * 4);
    o.v[0] = t.x; o.v[1] = t.y; o.v[2] = t.z; o.v[3] = t.w;
  } else if constexpr (LPL == 2) {
    const float2 t = *reinterpret_cast<const float2*>(p + lane * 2);
    o.v[0] = t.x; o.v[1] = t.y;
  } else {
    o.v[0] = p[lane];
  }
  return o;
}

// Vector shifted by one label: out(s) = x(s - 1) (dir < 0) or x(s + 1) (dir > 0).
template <int LPL>
__device__ __forceinline__ Vec<LPL> shift_label(const Vec<LPL>& x, int dir, float fill) {
  Vec<LPL> o;
  if (dir < 0) {
    o.v[0] = lane_prev(x.v[LPL - 1], fill);
#pragma unroll
    for (int j = 1; j < LPL; ++j) o.v[j] = x.v[j - 1];
  } else {
    o.v[LPL - 1] = lane_next(x.v[0], fill);
#pragma unroll
    for (int j = 0; j + 1 < LPL; ++j) o.v[j] = x.v[j + 1];
  }
  return o;
}

// The destinations of the one-label lane shifts, carried from step to step.  A
// shift by one lane writes every lane but the boundary one (lane 0 for the
// shift towards higher labels, lane 63 for the other), which keeps the value of
// the destination register; set to the fill once, that lane holds the fill for
// good, and no step re-initialises it.  mn_*: fill +inf (minimum of the
// neighbours), mx_*: fill -inf (maximum).
struct ShiftCarry {
  float mn_prev = kInfF, mn_next = kInfF, mx_prev = -kInfF, mx_next = -kInfF;
};

template <int LPL>
__device__ __forceinline__ Vec<LPL> shift_carry(const Vec<LPL>& x, int dir, float& carry) {
  Vec<LPL> o;
  if (dir < 0) {
    carry = dpp_f<0x138, 0xf, 0xf, false>(carry, x.v[LPL - 1]);  // wave_shr:1
    o.v[0] = carry;
#pragma unroll
    for (int j = 1; j < LPL; ++j) o.v[j] = x.v[j - 1];
  } else {
    carry = dpp_f<0x130, 0xf, 0xf, false>(carry, x.v[0]);  // wave_shl:1
    o.v[LPL - 1] = carry;
#pragma unroll
    for (int j = 0; j + 1 < LPL; ++j) o.v[j] = x.v[j + 1];
  }
  return o;
}

template <int LPL>
__device__ __forceinline__ Vec<LPL> plus(const Vec<LPL>& x, const Vec<LPL>& y) {
  Vec<LPL> o;
#pragma unroll
  for (int j = 0; j < LPL; ++j) o.v[j] = x.v[j] + y.v[j];
  return o;
}

template <int LPL>
__device__ __forceinline__ float local_min(const Vec<LPL>& x) {
  float m = x.v[0];
#pragma unroll
  for (int j = 1; j < LPL; ++j) m = fminf(m, x.v[j]);
  return m;
}

// True in a lane if any of its values is a NaN.  Under -fno-honor-nans the
// compiler may fold any floating-point NaN test (and an integer test of the
// value's bits, which it turns into one) to false, so the bits pass through an
// empty asm first: an integer the compiler knows nothing about.
template <int LPL>
__device__ __forceinline__ bool any_nan(const Vec<LPL>& x) {
  bool r = false;
#pragma unroll
  for (int j = 0; j < LPL; ++j) {
    unsigned u = __float_as_uint(x.v[j]);
    asm volatile("" : "+v"(u));
    r |= (u & 0x7fffffffu) > 0x7f800000u;  // exponent all ones, mantissa not zero
  }
  return r;
}

// The same values in new registers.  The sweeps keep their prefetched nodes in
// a register ring and refill a slot right after reading it; a value read from
// the slot that stays live past the refill would share its register with the
// refill load, and the register allocator would then copy the whole ring at the
// loop back-edge -- a copy that waits for every load in flight.  Copying such
// values first (the copy waits only for this slot's load, issued a ring length
// earlier) keeps each slot in fixed registers.
template <int LPL>
__device__ __forceinline__ Vec<LPL> fresh(const Vec<LPL>& x) {
  Vec<LPL> o;
#pragma unroll
  for (int j = 0; j < LPL; ++j) asm volatile("v_mov_b32 %0, %1" : "=v"(o.v[j]) : "v"(x.v[j]));
  return o;
}

// Makes the values opaque at this point, so that the arithmetic that formed them
// stays ahead of the slot refill that follows (otherwise it may be sunk past the
// refill, which again makes the slot's old value outlive it).
template <int LPL>
__device__ __forceinline__ void pin(Vec<LPL>& x) {
#pragma unroll
  for (int j = 0; j < LPL; ++j) asm volatile("" : "+v"(x.v[j]));
}

// f(integral_constant 0) ... f(integral_constant N-1): steps whose position is a
// compile-time constant.
template <int... I, typename F>
__device__ __forceinline__ void unroll_seq(std::integer_sequence<int, I...>, F&& f) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void unroll_steps(F&& f) {
  unroll_seq(std::make_integer_sequence<int, N>{}, static_cast<F&&>(f));
}

// Minimum over the 64 lanes of a value, left in every lane.  A wave alone on
// its SIMD takes 4 cycles per instruction (measured, stand-alone), wait states
// included, so the tree's length is what a sweep's step costs: four DPP levels
// inside each row of 16 lanes (two wait states before each), then the four rows'
// minima through v_readlane: 9 instructions against 10 with v_permlane16_swap
// and v_permlane32_swap, whose copies and wait states cannot be filled.
// ROWS = 2: the other two rows hold +inf (32 labels, kFitHalf: 4 instructions).
template <int ROWS = 4>
__device__ __forceinline__ float rows_min(float x) {
  auto row = [&](int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(x), l)); };
  if constexpr (ROWS == 2) return fminf(fminf(x, row(0)), row(16));
  const float s0 = row(0), s1 = row(16), s2 = row(32), s3 = row(48);
  // (one scalar operand per instruction, so no value has to be moved first)
  return fminf(fminf(fminf(s0, x), fminf(s1, x)), fminf(fminf(s2, x), fminf(s3, x)));
}
template <int ROWS = 4>
__device__ __forceinline__ float chain_min(float x) {
  x = fminf(x, dpp_rot<0xb1>(x));
  x = fminf(x, dpp_rot<0x4e>(x));
  x = fminf(x, dpp_rot<0x124>(x));
  x = fminf(x, dpp_rot<0x128>(x));
  return rows_min<ROWS>(x);
}

// A kernel-uniform value kept in a VGPR.  The steps multiply the edge weight
// (an SGPR, taken with v_readlane) by L1 and L2; with L1 and L2 in VGPRs each of
// those FMAs has one scalar operand, as a VALU instruction allows, and the weight
// needs no copy into a VGPR per step.
__device__ __forceinline__ float in_vgpr(float x) {
  asm volatile("" : "+v"(x));
  return x;
}

// near(s) = min over 0 < |s - t| < delta of x(t)  (+inf if delta == 1).
// DC = 2 fixes delta = 2 at compile time (no branch in the step); DC = 0 reads it.
template <int LPL, int DC>
__device__ __forceinline__ Vec<LPL> near_min(const Vec<LPL>& x, int delta, ShiftCarry& c) {
  if (DC == 2 || delta == 2) {  // the common case, straight-line
    const Vec<LPL> l = shift_carry(x, -1, c.mn_prev), r = shift_carry(x, +1, c.mn_next);
    Vec<LPL> o;
#pragma unroll
    for (int j = 0; j < LPL; ++j) o.v[j] = fminf(l.v[j], r.v[j]);
    return o;
  }
  Vec<LPL> acc;
#pragma unroll
  for (int j = 0; j < LPL; ++j) acc.v[j] = kInfF;
  Vec<LPL> l = x, r = x;
  for (int d = 1; d < delta; ++d) {
    l = shift_label(l, -1, kInfF);
    r = shift_label(r, +1, kInfF);
#pragma unroll
    for (int j = 0; j < LPL; ++j) acc.v[j] = fminf(acc.v[j], fminf(l.v[j], r.v[j]));
  }
  return acc;
}

template <int LPL, int DC>
__device__ __forceinline__ Vec<LPL> near_max(const Vec<LPL>& x, int delta, ShiftCarry& c) {
  if (DC == 2 || delta == 2) {
    const Vec<LPL> l = shift_carry(x, -1, c.mx_prev), r = shift_carry(x, +1, c.mx_next);
    Vec<LPL> o;
#pragma unroll
    for (int j = 0; j < LPL; ++j) o.v[j] = fmaxf(l.v[j], r.v[j]);
    return o;
  }
  Vec<LPL> acc;
#pragma unroll
  for (int j = 0; j < LPL; ++j) acc.v[j] = -kInfF;
  Vec<LPL> l = x, r = x;
  for (int d = 1; d < delta; ++d) {
    l = shift_label(l, -1, -kInfF);
    r = shift_label(r, +1, -kInfF);
#pragma unroll
    for (int j = 0; j < LPL; ++j) acc.v[j] = fmaxf(acc.v[j], fmaxf(l.v[j], r.v[j]));
  }
  return acc;
}

// near(s) + P1 for every label and the minimum over all labels, the two parts
// of the min-convolution that do not wait for each other.  P1 = w L1 (PE false)
// or w (PE).  fma(w, L1, .) is monotone, so it may be taken before the minimum
// over the neighbours as well as after it, with the same bits; with two labels
// per lane (LPL = 2, delta = 2) that saves an instruction per label: a label's
// neighbours are the other label of its own lane and the one of an adjacent
// lane, so t_j = P1 + x_{1-j} turns into the result by one v_min with a DPP
// operand, in place.  The lane at the border has no source: its destination
// stays, which is the one neighbour it has.
//
// The blocks fix the order so that every DPP operand is two instructions old
// (the wait states DPP needs after a VALU write), and so is w, which the caller
// takes with v_readlane: the sum that forms U and the neighbour terms fill the
// first two levels of the minimum's tree, with no instruction spent on waiting.
//
// near_block returns the minimum's tree after two levels (near_min_rest goes
// on).  FORM 0: U is given; 1: U = x + y; 2: U = x - (x + y) / 4 (fused, as the
// forward pass's V from R and Bh).
template <int LPL, int DC, bool PE, int FORM>
__device__ __forceinline__ float near_block(Vec<LPL>& U, const Vec<LPL>& x, const Vec<LPL>& y, float w, float L1,
                                            int delta, ShiftCarry& c, Vec<LPL>& nr) {
  if constexpr (LPL == 2 && DC == 2) {
    float lm, t0, t1;
#define CCS_NEAR_P1 "v_add_f32 %4, %[w], %1\n\tv_add_f32 %3, %[w], %0\n\t"
#define CCS_NEAR_L1 "v_fma_f32 %4, %[w], %[l1], %1\n\tv_fma_f32 %3, %[w], %[l1], %0\n\t"
#define CCS_NEAR_TREE                                                            \
  "v_min_f32_dpp %2, %2, %2 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n\t" \
  "v_min_f32_dpp %4, %4, %4 wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"          \
  "v_min_f32_dpp %3, %3, %3 wave_shl:1 row_mask:0xf bank_mask:0xf\n\t"          \
  "v_min_f32_dpp %2, %2, %2 quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf"
    if constexpr (FORM == 0) {
#define CCS_NEAR_U "s_nop 0\n\tv_min_f32 %2, %0, %1\n\t"
      if constexpr (PE)
        asm(CCS_NEAR_U CCS_NEAR_P1 CCS_NEAR_TREE
            : "+&v"(U.v[0]), "+&v"(U.v[1]), "=&v"(lm), "=&v"(t0), "=&v"(t1) : [w] "s"(w));
      else
        asm(CCS_NEAR_U CCS_NEAR_L1 CCS_NEAR_TREE
            : "+&v"(U.v[0]), "+&v"(U.v[1]), "=&v"(lm), "=&v"(t0), "=&v"(t1) : [w] "s"(w), [l1] "v"(L1));
#undef CCS_NEAR_U
    } else if constexpr (FORM == 1) {
#define CCS_NEAR_U "v_add_f32 %1, %[x1], %[y1]\n\tv_add_f32 %0, %[x0], %[y0]\n\tv_min_f32 %2, %0, %1\n\t"
      if constexpr (PE)
        asm(CCS_NEAR_U CCS_NEAR_P1 CCS_NEAR_TREE
            : "=&v"(U.v[0]), "=&v"(U.v[1]), "=&v"(lm), "=&v"(t0), "=&v"(t1)
            : [w] "s"(w), [x0] "v"(x.v[0]), [x1] "v"(x.v[1]), [y0] "v"(y.v[0]), [y1] "v"(y.v[1]));
      else
        asm(CCS_NEAR_U CCS_NEAR_L1 CCS_NEAR_TREE
            : "=&v"(U.v[0]), "=&v"(U.v[1]), "=&v"(lm), "=&v"(t0), "=&v"(t1)
            : [w] "s"(w), [l1] "v"(L1), [x0] "v"(x.v[0]), [x1] "v"(x.v[1]), [y0] "v"(y.v[0]), [y1] "v"(y.v[1]));
#undef CCS_NEAR_U
    } else {
      static_assert(kGamma == 0.25f, "the constant below");
#define CCS_NEAR_U                                                            \
  "v_add_f32 %1, %[x1], %[y1]\n\tv_add_f32 %0, %[x0], %[y0]\n\t"             \
  "v_fmamk_f32 %1, %1, 0xbe800000, %[x1]\n\t"                                 \
  "v_fmamk_f32 %0, %0, 0xbe800000, %[x0]\n\tv_min_f32 %2, %0, %1\n\t"
      if constexpr (PE)
        asm(CCS_NEAR_U CCS_NEAR_P1 CCS_NEAR_TREE
            : "=&v"(U.v[0]), "=&v"(U.v[1]), "=&v"(lm), "=&v"(t0), "=&v"(t1)
            : [w] "s"(w), [x0] "v"(x.v[0]), [x1] "v"(x.v[1]), [y0] "v"(y.v[0]), [y1] "v"(y.v[1]));
      else
        asm(CCS_NEAR_U CCS_NEAR_L1 CCS_NEAR_TREE
            : "=&v"(U.v[0]), "=&v"(U.v[1]), "=&v"(lm), "=&v"(t0), "=&v"(t1)
            : [w] "s"(w), [l1] "v"(L1), [x0] "v"(x.v[0]), [x1] "v"(x.v[1]), [y0] "v"(y.v[0]), [y1] "v"(y.v[1]));
#undef CCS_NEAR_U
    }
#undef CCS_NEAR_P1
#undef CCS_NEAR_L1
#undef CCS_NEAR_TREE
    nr.v[0] = t1;  // label 2 lane: its neighbours are x_1 of this lane and of the previous one
    nr.v[1] = t0;
    return lm;
  } else {
    if constexpr (FORM == 1) {
#pragma unroll
      for (int j = 0; j < LPL; ++j) U.v[j] = x.v[j] + y.v[j];
    } else if constexpr (FORM == 2) {
#pragma unroll
      for (int j = 0; j < LPL; ++j) U.v[j] = fmaf(-kGamma, x.v[j] + y.v[j], x.v[j]);
    }
    const Vec<LPL> n0 = near_min<LPL, DC>(U, delta, c);
#pragma unroll
    for (int j = 0; j < LPL; ++j) nr.v[j] = PE ? n0.v[j] + w : fmaf(w, L1, n0.v[j]);
    return local_min(U);
  }
}

// The rest of the minimum's tree, from near_block's partial minimum.
template <int LPL, int DC, int ROWS = 4>
__device__ __forceinline__ float near_min_rest(float lm) {
  if constexpr (!(LPL == 2 && DC == 2)) return chain_min<ROWS>(lm);
  lm = fminf(lm, dpp_rot<0x124>(lm));
  lm = fminf(lm, dpp_rot<0x128>(lm));
  return rows_min<ROWS>(lm);
}

// U = x + y and its neighbour terms alone (the recomputed messages, whose
// minimum is stored).
template <int LPL, int DC, bool PE>
__device__ __forceinline__ void near_only(Vec<LPL>& U, const Vec<LPL>& x, const Vec<LPL>& y, float w, float L1,
                                          int delta, ShiftCarry& c, Vec<LPL>& nr) {
  if constexpr (LPL == 2 && DC == 2) {
    float t0, t1;
    if constexpr (PE)
      asm("v_add_f32 %1, %[x1], %[y1]\n\t"
          "v_add_f32 %0, %[x0], %[y0]\n\t"
          "v_add_f32 %3, %[w], %1\n\t"
          "v_add_f32 %2, %[w], %0\n\t"
          "s_nop 0\n\t"
          "v_min_f32_dpp %3, %3, %3 wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
          "v_min_f32_dpp %2, %2, %2 wave_shl:1 row_mask:0xf bank_mask:0xf"
          : "=&v"(U.v[0]), "=&v"(U.v[1]), "=&v"(t0), "=&v"(t1)
          : [w] "s"(w), [x0] "v"(x.v[0]), [x1] "v"(x.v[1]), [y0] "v"(y.v[0]), [y1] "v"(y.v[1]));
    else
      asm("v_add_f32 %1, %[x1], %[y1]\n\t"
          "v_add_f32 %0, %[x0], %[y0]\n\t"
          "v_fma_f32 %3, %[w], %[l1], %1\n\t"
          "v_fma_f32 %2, %[w], %[l1], %0\n\t"
          "s_nop 0\n\t"
          "v_min_f32_dpp %3, %3, %3 wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
          "v_min_f32_dpp %2, %2, %2 wave_shl:1 row_mask:0xf bank_mask:0xf"
          : "=&v"(U.v[0]), "=&v"(U.v[1]), "=&v"(t0), "=&v"(t1)
          : [w] "s"(w), [l1] "v"(L1), [x0] "v"(x.v[0]), [x1] "v"(x.v[1]), [y0] "v"(y.v[0]), [y1] "v"(y.v[1]));
    nr.v[0] = t1;
    nr.v[1] = t0;
  } else {
#pragma unroll
    for (int j = 0; j < LPL; ++j) U.v[j] = x.v[j] + y.v[j];
    const Vec<LPL> n0 = near_min<LPL, DC>(U, delta, c);
#pragma unroll
    for (int j = 0; j < LPL; ++j) nr.v[j] = PE ? n0.v[j] + w : fmaf(w, L1, n0.v[j]);
  }
}

// max over the neighbours of m, minus P1, for every label (-fma(-L1, w, .) is
// monotone too), and a = th + m, whose first sum fills the block's wait state.
// mx: m with -inf in the lanes without a label.
template <int LPL, int DC, bool PE>
__device__ __forceinline__ void near_max_minus(const Vec<LPL>& mx, const Vec<LPL>& m, const Vec<LPL>& th, float w,
                                               float L1, int delta, ShiftCarry& c, Vec<LPL>& nx, Vec<LPL>& a) {
  if constexpr (LPL == 2 && DC == 2) {
    float t0, t1;
    if constexpr (PE)
      asm("v_subrev_f32 %1, %[w], %[m1]\n\t"
          "v_subrev_f32 %0, %[w], %[m0]\n\t"
          "v_add_f32 %2, %[th], %[m]\n\t"
          "v_max_f32_dpp %1, %1, %1 wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
          "v_max_f32_dpp %0, %0, %0 wave_shl:1 row_mask:0xf bank_mask:0xf"
          : "=&v"(t0), "=&v"(t1), "=&v"(a.v[0])
          : [w] "s"(w), [m0] "v"(mx.v[0]), [m1] "v"(mx.v[1]), [m] "v"(m.v[0]), [th] "v"(th.v[0]));
    else
      asm("v_fma_f32 %1, -%[l1], %[w], %[m1]\n\t"
          "v_fma_f32 %0, -%[l1], %[w], %[m0]\n\t"
          "v_add_f32 %2, %[th], %[m]\n\t"
          "v_max_f32_dpp %1, %1, %1 wave_shr:1 row_mask:0xf bank_mask:0xf\n\t"
          "v_max_f32_dpp %0, %0, %0 wave_shl:1 row_mask:0xf bank_mask:0xf"
          : "=&v"(t0), "=&v"(t1), "=&v"(a.v[0])
          : [w] "s"(w), [l1] "v"(L1), [m0] "v"(mx.v[0]), [m1] "v"(mx.v[1]), [m] "v"(m.v[0]), [th] "v"(th.v[0]));
    nx.v[0] = t1;
    nx.v[1] = t0;
    a.v[1] = th.v[1] + m.v[1];
  } else {
    const Vec<LPL> n0 = near_max<LPL, DC>(mx, delta, c);
#pragma unroll
    for (int j = 0; j < LPL; ++j) {
      nx.v[j] = PE ? n0.v[j] - w : fmaf(-L1, w, n0.v[j]);
      a.v[j] = th.v[j] + m.v[j];
    }
  }
}

// m(s) = min(U(s), near(U)(s) + P1, min U + P2) from the parts above: nr =
// near + P1, umin = min U, P2 = w L2 or (PE) w2.
template <int LPL, bool PE>
__device__ __forceinline__ Vec<LPL> minconv(const Vec<LPL>& U, const Vec<LPL>& nr, float umin, float w, float w2,
                                            float L2) {
  const float far = PE ? umin + w2 : fmaf(w, L2, umin);
  Vec<LPL> m;
#pragma unroll
  for (int j = 0; j < LPL; ++j) m.v[j] = fminf(fminf(U.v[j], nr.v[j]), far);
  return m;
}

// Node loads never sit under divergent control flow (that would make the
// compiler drain every outstanding load at the join): with kFitFull every lane
// owns LPL labels and loads them as one vector, with kFitLanes the lanes without
// labels load the last lane's again; with kFitAny the lane loads clamped
// addresses element by element.  What the places without a label load is replaced
// where it is used (masked()), never beside the load: a select there is scheduled
// with the load and waits for it, which empties the register rings (320 x 240 x 32
// rows 58 us, x 64 52 us; a streamed wave waits once per segment).
template <int LPL, int FIT>
__device__ __forceinline__ Vec<LPL> masked(const Vec<LPL>& x, int lane, int D, float fill) {
  Vec<LPL> o;
#pragma unroll
  for (int j = 0; j < LPL; ++j)
    o.v[j] = FIT == kFitFull || lane * LPL + (FIT == kFitAny ? j : 0) < D ? x.v[j] : fill;
  return o;
}

template <int LPL, int FIT>
__device__ __forceinline__ Vec<LPL> ld_node(const float* __restrict__ base, int lane, int D) {
  Vec<LPL> out;
  if constexpr (FIT != kFitAny) {
    const int l = FIT == kFitFull ? lane * LPL : min(lane * LPL, D - LPL);
    if constexpr (LPL == 4) {
      const float4 t = *reinterpret_cast<const float4*>(base + l);
      out.v[0] = t.x; out.v[1] = t.y; out.v[2] = t.z; out.v[3] = t.w;
    } else if constexpr (LPL == 2) {
      const float2 t = *reinterpret_cast<const float2*>(base + l);
      out.v[0] = t.x; out.v[1] = t.y;
    } else {
      out.v[0] = base[l];
    }
  } else {
#pragma unroll
    for (int j = 0; j < LPL; ++j) {
      const int s = lane * LPL + j;
      out.v[j] = base[s < D ? s : D - 1];
    }
  }
  return out;
}

template <int LPL, int FIT>
__device__ __forceinline__ void st_node(float* __restrict__ base, int lane, int D, const Vec<LPL>& x) {
  if constexpr (FIT != kFitAny) {
    if (FIT != kFitFull && lane * LPL >= D) return;
    if constexpr (LPL == 4) {  // two 64-bit stores (see kNoWideStores)
      *reinterpret_cast<float2*>(base + lane * 4) = make_float2(x.v[0], x.v[1]);
      asm volatile("" ::: "memory");
      *reinterpret_cast<float2*>(base + lane * 4 + 2) = make_float2(x.v[2], x.v[3]);
    } else if constexpr (LPL == 2) {
      *reinterpret_cast<float2*>(base + lane * 2) = make_float2(x.v[0], x.v[1]);
    } else {
      base[lane] = x.v[0];
    }
  } else {
#pragma unroll
    for (int j = 0; j < LPL; ++j)
      if (lane * LPL + j < D) base[lane * LPL + j] = x.v[j];
  }
}

// Buffer-resource access for the row sweeps.  A row chain's nodes (and its
// message buffer) are contiguous, so a node address is the chain's base, held in
// a buffer resource, plus a 32-bit byte offset in an SGPR: one or two scalar
// instructions per node instead of 64-bit address arithmetic.  Every offset
// passed here is that of a node inside the resource's range.
typedef __amdgpu_buffer_rsrc_t Rsrc;

__device__ __forceinline__ Rsrc chain_rsrc(const float* base, long nfloats) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(base), (short)0, (int)(nfloats * 4), 0x00020000);
}

// AUX: cache policy of the access (0, or kStream for costs that a sweep reads
// once and that do not stay in the cache until the next one: they then leave the
// cached part to the unaries, which every sweep reads twice).
constexpr int kStream = 2;  // non-temporal
template <int LPL, int FIT, int AUX = 0>
__device__ __forceinline__ Vec<LPL> ld_buf(Rsrc r, int soff, int lane, int D) {
  Vec<LPL> out;
  if constexpr (FIT != kFitAny) {
    const int voff = (FIT == kFitFull ? lane * LPL : min(lane * LPL, D - LPL)) * 4;
    if constexpr (LPL == 4) {
      const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(r, voff, soff, AUX);
#pragma unroll
      for (int j = 0; j < 4; ++j) out.v[j] = __uint_as_float(t[j]);
    } else if constexpr (LPL == 2) {
      const u32x2 t = __builtin_amdgcn_raw_buffer_load_b64(r, voff, soff, AUX);
      out.v[0] = __uint_as_float(t[0]);
      out.v[1] = __uint_as_float(t[1]);
    } else {
      out.v[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, voff, soff, AUX));
    }
  } else {
#pragma unroll
    for (int j = 0; j < LPL; ++j) {
      const int s = lane * LPL + j;
      out.v[j] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, (s < D ? s : D - 1) * 4, soff, AUX));
    }
  }
  return out;
}

template <int LPL, int FIT>
__device__ __forceinline__ void st_buf(Rsrc r, int soff, int lane, int D, const Vec<LPL>& x) {
  if constexpr (FIT != kFitAny) {
    // The lanes without labels store past the resource's range, which the
    // hardware drops: no branch around the store.
    const int voff = FIT == kFitFull || lane * LPL < D ? lane * LPL * 4 : (int)0x80000000;
    if constexpr (LPL == 4) {  // two 64-bit stores (see kNoWideStores)
      const u32x2 t = {__float_as_uint(x.v[0]), __float_as_uint(x.v[1])};
      const u32x2 u = {__float_as_uint(x.v[2]), __float_as_uint(x.v[3])};
      __builtin_amdgcn_raw_buffer_store_b64(t, r, voff, soff, 0);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_raw_buffer_store_b64(u, r, voff + 8, soff, 0);
    } else if constexpr (LPL == 2) {
      const u32x2 t = {__float_as_uint(x.v[0]), __float_as_uint(x.v[1])};
      __builtin_amdgcn_raw_buffer_store_b64(t, r, voff, soff, 0);
    } else {
      __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x.v[0]), r, voff, soff, 0);
    }
  } else {
#pragma unroll
    for (int j = 0; j < LPL; ++j) {
      const int s = lane * LPL + j;
      if (s < D) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x.v[j]), r, s * 4, soff, 0);
    }
  }
}

// Edge weights of a block of up to 64 steps sit one per lane (lane j: the
// block's step j), read from LDS a block ahead; a step takes its weight with
// v_readlane, as an SGPR operand, so the step itself waits on no LDS access.
__device__ __forceinline__ float lane_weight(float wv, int j) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(wv), j));
}

// Suffix sums b_i = u_i + ... + u_{n-2} (b_{n-1} = 0) of the backward-pass
// minima, in float64, the 64 lanes each taking a contiguous segment; returns b_0.
// Done once after the pass so the per-node step carries no float64 work.
__device__ double chain_offsets(const float* u, double* b, int n, int lane) {
  const int m = n - 1;
  const int L = (m + 63) / 64;
  const int s0 = min(lane * L, m), s1 = min(s0 + L, m);
  double tot = 0.0;
  for (int j = s0; j < s1; ++j) tot += (double)u[j];
  double incl = tot;  // sum over this lane and the lanes above it
  for (int o = 1; o < 64; o <<= 1) {
    const double t = __shfl_down(incl, o, 64);
    if (lane + o < 64) incl += t;
  }
  double acc = __shfl_down(incl, 1, 64);
  if (lane == 63) acc = 0.0;
  for (int j = s1 - 1; j >= s0; --j) {
    acc += (double)u[j];
    b[j] = acc;
  }
  if (lane == 0) b[m] = 0.0;
  return __shfl(incl, 0, 64);
}

// Kept constant of the forward pass: r_0 = 0, r_{i+1} = a r_i + v_i - g b_i with
// a = 1 - g for i < m = n - 1; returns g * sum_{i<m} (r_i + b_i) + r_m.  Each
// lane runs its segment from r = 0 and the segments are joined by a scan of the
// affine maps x -> a^len x + r_end.
__device__ double chain_kept(const float* v, const double* b, int n, int lane, double g) {
  const int m = n - 1;
  const double a = 1.0 - g;
  const int L = (m + 63) / 64;
  const int s0 = min(lane * L, m), s1 = min(s0 + L, m);
  double r = 0.0, sr = 0.0, sb = 0.0, geo = 0.0, ap = 1.0;
  for (int j = s0; j < s1; ++j) {
    sr += r;
    geo += ap;
    sb += b[j];
    r = a * r + ((double)v[j] - g * b[j]);
    ap *= a;
  }
  double A = ap, B = r;  // this lane's map, then the composition of lanes 0..lane
  for (int o = 1; o < 64; o <<= 1) {
    const double Ap = __shfl_up(A, o, 64), Bp = __shfl_up(B, o, 64);
    if (lane >= o) {
      B = A * Bp + B;
      A = A * Ap;
    }
  }
  double rin = __shfl_up(B, 1, 64);  // r at the start of this lane's segment
  if (lane == 0) rin = 0.0;
  const double total = wave_sum_f64(g * (sr + rin * geo + sb));
  return total + __shfl(B, 63, 64);
}

// Pipelined chain sweep.  Every input stream of a pass (unaries, cost, backward
// messages, edge weights) runs P nodes ahead of the node being processed: the
// main loop handles blocks of P nodes, unrolled, so ring slot j is a fixed set
// of registers and the load for node s + P is issued right after slot s is read
// (clamped to the last node, so it never leaves the chain).  The last partial
// block is an unrolled tail that issues no loads.
//
// SEG: 0 every message is stored; 1 checkpointed; 2 checkpointed, costs streamed.
template <int LPL, int MODE, int P, int FIT, int DC, int SEG, bool NANCHK, bool PE>
__global__ __launch_bounds__(MODE != kColsMinorant && SEG ? 256 : 64) void k_chain(ChainArgs a) {
  extern __shared__ double lds_all[];
  constexpr bool kCols = MODE == kColsMinorant;
  // Rows with a message wave: wave 0 runs both passes, wave 1 recomputes the
  // forward pass's messages into the LDS ring (see kRowRing).  A workgroup of
  // 256 threads runs two chains (waves 0-1 and 2-3, each with its own LDS), so
  // that between one and two times as many chains as CUs need not put two
  // workgroups on a CU.
  constexpr bool kRowSeg = !kCols && SEG != 0;
  constexpr int kCostAux = SEG == 2 ? kStream : 0;
  constexpr int KR = kRowSeg ? seg_len<LPL>() : 1;
  static_assert(!kRowSeg || P == kRowRing * KR, "the forward ring spans the message ring");
  static_assert(P <= 64, "one weight per lane and step of a block");
  constexpr int kNS = 64 * LPL;  // ring stride per node, floats
  const int n = a.n, D = a.D;
  const int cs = kRowSeg ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 7) : 0;  // chain slot of the workgroup
  const int cpw = kRowSeg ? (int)(blockDim.x >> 7) : 1;
  const int c_slot = blockIdx.x * cpw + cs;
  const int c = min(c_slot, a.n_chains - 1);  // a missing second chain only keeps the barriers
  const int lane = threadIdx.x & 63;
  const int wid = __builtin_amdgcn_readfirstlane((threadIdx.x >> 6) & (kRowSeg ? 1 : 63));  // wave in the chain
  // per chain: b (doubles), w, u, [w2], v, then the ring (floats, 16-byte aligned)
  const int chain_floats = (((PE ? 6 : 5) * n + 3) & ~3) + (kRowSeg ? kRowRing * KR * kNS : 0);
  double* b_lds = lds_all + cs * (chain_floats / 2);  // b_i = offset of the true backward message at node i
  ShiftCarry cc;
  const float L1v = in_vgpr(a.L1), L2v = in_vgpr(a.L2);
  const long pbase = (long)c * a.pcs;
  const long nstride = a.pns * (long)D;  // floats between consecutive nodes
  // The running state alternates between the two subproblems' unaries, so
  // that each sweep reads one volume for its chain unaries:
  //   rows read A from A_in (A, or the cost volume in a run's first sweep) and
  //     write the column unaries C - A' (A' = A - g);
  //   columns read B = C - A from A and write the row unaries A' = (C - B) + g.
  // Both convert with the cost volume in their forward pass only.  The decode
  // reads A.
  const float* __restrict__ Ab = (kCols ? a.A : a.A_in) + pbase * D;
  float* __restrict__ Aw = a.A + pbase * D;
  const float* __restrict__ Cb = MODE != kRowsDecode ? a.cost + pbase * D : nullptr;
  const float* __restrict__ wb = a.w + pbase * a.wmul;
  const float* __restrict__ wb2 = PE ? a.w2 + pbase * a.wmul : nullptr;
  float* __restrict__ msg = a.msg + (long)c * n * D;
  bool valid[LPL];
#pragma unroll
  for (int j = 0; j < LPL; ++j) valid[j] = FIT == kFitFull || lane * LPL + (FIT == kFitLanes ? 0 : j) < D;
  // (with kFitLanes +inf unaries alone keep the lanes without labels out)
  auto keep = [&](int j) { return FIT != kFitAny || valid[j]; };

  // The chain unaries: what the sweep reads (A for rows, B for columns).
  auto theta_of = [&](const Vec<LPL>& av) { return masked<LPL, FIT>(av, lane, D, kInfF); };
  // Columns: the row unaries C - B of a node.
  auto row_unaries = [&](const Vec<LPL>& bv, const Vec<LPL>& cv) {
    Vec<LPL> r;
#pragma unroll
    for (int j = 0; j < LPL; ++j) r.v[j] = cv.v[j] - bv.v[j];
    return r;
  };
  // Rows: the column unaries C - A' stored for a node.
  auto col_unaries = [&](const Vec<LPL>& out, const Vec<LPL>& cv) {
    Vec<LPL> r;
#pragma unroll
    for (int j = 0; j < LPL; ++j) r.v[j] = cv.v[j] - out.v[j];
    return r;
  };

  // The chain's edge weights (per-edge P1 and P2 with PE) go to LDS once (the
  // sweeps read them a block of steps at a time, one per lane).  u_lds takes
  // the per-node minima of a pass (float64 sums are formed after it).
  float* w_lds = reinterpret_cast<float*>(b_lds + n);
  float* u_lds = w_lds + n;
  float* w2_lds = u_lds + n;  // PE only
  // kRowSeg: the forward minima go to v_lds (u_lds keeps the backward minima
  // that the message wave reads), then the message ring at a 16-byte boundary.
  float* v_lds = w2_lds + (PE ? n : 0);
  // (offset arithmetic on the LDS pointer itself keeps its address space)
  float* ring = reinterpret_cast<float*>(b_lds) + (((PE ? 6 : 5) * n + 3) & ~3);
  float* fw_lds = kRowSeg ? v_lds : u_lds;
  const long wstep = a.pns * a.wmul;
  constexpr int kChainThreads = kRowSeg ? 128 : 64;
  for (int i = threadIdx.x & (kChainThreads - 1); i < n - 1; i += kChainThreads) {
    w_lds[i] = wb[(long)i * wstep];
    if constexpr (PE) w2_lds[i] = wb2[(long)i * wstep];
  }
  __syncthreads();
  if constexpr (kRowSeg) {
    if (c_slot >= a.n_chains) {  // the workgroup's second chain is missing: the same barriers, no work
      const int M = (n - 1 + KR - 1) / KR;
      __syncthreads();
      for (int k = 0; k < (M == 0 ? 0 : (M > 2 ? M - 1 : 1)); ++k) lds_barrier();
      return;
    }
  }

  Vec<LPL> ra[P], rc[P], rb[P];
  // Row chains (the host guarantees a row's byte extent fits in 31 bits): the
  // unaries and the messages through buffer resources; columns use 64-bit
  // addresses (their nodes span the whole volume).
  const int strideB = (int)(nstride * 4);
  const Rsrc rA = chain_rsrc(Ab, (long)(n - 1) * nstride + D);
  const Rsrc rW = chain_rsrc(Aw, (long)(n - 1) * nstride + D);
  const Rsrc rM = chain_rsrc(msg, (long)n * D);

  // ---- backward pass: step s handles i = n-2-s: Bh[i] = minconv(theta[i+1] + Bh[i+1]) - min(...)
  // kRowSeg: wave 0 only; it stores the messages at i = nb - m*KR (m >= 1), so
  // a step s0 + j of a block (s0 a multiple of P, itself a multiple of KR) is a
  // checkpoint exactly when (j + 1) % KR == 0.
  const int nb = n - 1;
  Vec<LPL> bh;
  bool nan_seen = false;  // NANCHK: a unary read by this lane was NaN
  double bsum = 0.0;
  Vec<LPL> a0, c0, th0;
  // kRowSeg, wave 1: the forward pass's messages.  Segment s holds the forward
  // steps i' = s*KR + t (t < KR) of node i = i' - g, where the g = M*KR - nb
  // virtual steps before node 0 end-align the segments with the checkpoints
  // (Bh at (s+1)*KR - g is one; Bh_{n-1} = 0).  Each message is recomputed
  // with the backward step's own operations and operands (theta_{i+1} + Bh_{i+1},
  // the stored minimum u_i, the edge's penalties), so it equals the message
  // the backward pass formed, and goes to ring slot i' % (kRowRing*KR).
  // Segments 0 and 1 are done before the first barrier, then segment s before
  // the barrier that wave 0 passes at the start of segment s - 1.
  auto row_messages = [&]() {
    if constexpr (kRowSeg) {
      constexpr int K = KR;
      const int M = (nb + K - 1) / K;
      // NANCHK: this wave tests node 0 and every unary its segments consume
      // (nodes 1 .. n-1) and sets the chain's flag, off the forward wave.
      bool nan1 = NANCHK && any_nan(ld_buf<LPL, FIT>(rA, 0, lane, D));
      auto put_flag = [&]() {
        if constexpr (NANCHK) {
          const bool any = __ballot(nan1) != 0;  // all lanes take part
          if (lane == 0) a.nan_flags[c] = any ? 1 : 0;
        }
      };
      if (M == 0) {
        put_flag();
        return;
      }
      const int g = M * K - nb;
      struct HSeg {
        Vec<LPL> a[K], m;
        float u, w, w2;
      };
      HSeg X, Y;
      auto load_h = [&](int s, HSeg& B) {  // s is clamped by the caller to a segment
        const int ib = s * K - g;            // node of t = 0 (negative only in segment 0)
#pragma unroll
        for (int t = 0; t < K; ++t)
          B.a[t] = ld_buf<LPL, FIT>(rA, min(max(ib + t + 1, 1), n - 1) * strideB, lane, D);
        B.m = ld_buf<LPL, FIT>(rM, (ib + K) * D * 4, lane, D);
        const int e = max(min(ib + lane, n - 2), 0);
        B.u = u_lds[e];
        B.w = w_lds[e];
        B.w2 = PE ? w2_lds[e] : 0.f;
      };
      auto run_h = [&](int s, const HSeg& B) {
        const int ib = s * K - g;
        float* slot = ring + (s % kRowRing) * K * kNS;
        Vec<LPL> Xb = B.m;
#pragma unroll
        for (int t = K - 1; t >= 0; --t) {
          if (ib + t >= 0) {
            if constexpr (NANCHK) nan1 |= any_nan(B.a[t]);
            const float u = lane_weight(B.u, t);
            Vec<LPL> U, nr;
            near_only<LPL, DC, PE>(U, theta_of(B.a[t]), Xb, lane_weight(B.w, t), L1v, a.delta, cc, nr);
            const Vec<LPL> m = minconv<LPL, PE>(U, nr, u, lane_weight(B.w, t), PE ? lane_weight(B.w2, t) : 0.f, L2v);
#pragma unroll
            for (int k = 0; k < LPL; ++k) Xb.v[k] = keep(k) ? m.v[k] - u : 0.f;
            st_ring<LPL>(slot + t * kNS, lane, Xb);
          }
        }
      };
      load_h(0, X);
      load_h(min(1, M - 1), Y);
      run_h(0, X);
      load_h(min(2, M - 1), X);
      if (M > 1) run_h(1, Y);
      lds_barrier();  // segments 0 and 1 are in the ring
      for (int s = 2; s < M;) {
        load_h(min(s + 1, M - 1), Y);
        __builtin_amdgcn_sched_barrier(0);
        run_h(s, X);
        lds_barrier();
        if (++s >= M) break;
        load_h(min(s + 1, M - 1), X);
        __builtin_amdgcn_sched_barrier(0);
        run_h(s, Y);
        lds_barrier();
        ++s;
      }
      put_flag();
    }
  };
  if (!kRowSeg || wid == 0) {
  auto load_b = [&](int s, Vec<LPL>& av) {
    const int node = s < nb ? n - 1 - s : 1;  // clamped: beyond the chain re-read node 1
    if constexpr (kCols)
      av = ld_node<LPL, FIT>(Ab + node * nstride, lane, D);
    else
      av = ld_buf<LPL, FIT>(rA, node * strideB, lane, D);
  };
  // weights of steps s0 .. s0+63 of the backward pass (edge n-2-s)
  auto wlane_b = [&](int s0) { return w_lds[max(n - 2 - (s0 + lane), 0)]; };
  auto wlane_b2 = [&](int s0) { return PE ? w2_lds[max(n - 2 - (s0 + lane), 0)] : 0.f; };
#pragma unroll
  for (int j = 0; j < LPL; ++j) bh.v[j] = 0.f;
  st_node<LPL, FIT>(msg + (long)(n - 1) * D, lane, D, bh);
  // th: theta_{i+1}; refill() re-issues the ring slot th came from, once its
  // value is read; ck: (kRowSeg) this step's message is a checkpoint
  auto step_b = [&](int s, const Vec<LPL>& th, float wi, float wi2, bool ck, auto&& refill) {
    const int i = n - 2 - s;
    Vec<LPL> U, nr;
    const float lm = near_block<LPL, DC, PE, 1>(U, th, bh, wi, L1v, a.delta, cc, nr);
    __builtin_amdgcn_sched_barrier(kSchedValu);
    refill();
    const float u = near_min_rest<LPL, DC>(lm);
    const Vec<LPL> m = minconv<LPL, PE>(U, nr, u, wi, wi2, L2v);
#pragma unroll
    for (int k = 0; k < LPL; ++k) bh.v[k] = keep(k) ? m.v[k] - u : 0.f;
    if constexpr (kCols) {
      constexpr int K = SEG != 0 ? seg_len<LPL>() : 0;
      if (K == 0 || i % K == 0) st_node<LPL, FIT>(msg + (long)i * D, lane, D, bh);  // i is wave-uniform
    } else if constexpr (kRowSeg) {
      if (ck) st_buf<LPL, FIT>(rM, i * D * 4, lane, D, bh);
    } else {
      st_buf<LPL, FIT>(rM, i * D * 4, lane, D, bh);
    }
    u_lds[i] = u;  // every lane writes the same value
  };
  if (nb > 0) {
#pragma unroll
    for (int j = 0; j < P; ++j) load_b(j, ra[j]);
  }
  int s0 = 0;
  float wv = wlane_b(0), wv2 = wlane_b2(0);
  for (; s0 + P <= nb; s0 += P) {
    const float wnext = wlane_b(s0 + P), wnext2 = wlane_b2(s0 + P);
    // kRowSeg: byte offsets of the block's refills, one per lane (v_readlane
    // per step instead of clamping each offset with scalar instructions)
    const int bo = kRowSeg ? (s0 + P + lane < nb ? n - 1 - (s0 + P + lane) : 1) * strideB : 0;
#pragma unroll
    for (int j = 0; j < P; ++j) {
      if constexpr (NANCHK && !kRowSeg) nan_seen |= any_nan(ra[j]);
      // Slot j is consumed (U is a new value) before it is refilled, so the
      // refill reuses the slot's registers.
      step_b(s0 + j, theta_of(ra[j]), lane_weight(wv, j), PE ? lane_weight(wv2, j) : 0.f, (j + 1) % KR == 0, [&]() {
        if constexpr (kRowSeg)
          ra[j] = ld_buf<LPL, FIT>(rA, __builtin_amdgcn_readlane(bo, j), lane, D);
        else
          load_b(s0 + j + P, ra[j]);
      });
    }
    wv = wnext;
    wv2 = wnext2;
  }
#pragma unroll
  for (int j = 0; j < P; ++j)
    if (s0 + j < nb) {
      if constexpr (NANCHK && !kRowSeg) nan_seen |= any_nan(ra[j]);
      step_b(s0 + j, theta_of(ra[j]), lane_weight(wv, j), PE ? lane_weight(wv2, j) : 0.f, (j + 1) % KR == 0, []() {});
    }
  bsum = chain_offsets(u_lds, b_lds, n, lane);  // b_0 = sum of all minima

  // bh holds Bh[0]; theta[0] is read directly.
  a0 = ld_node<LPL, FIT>(Ab, lane, D);
  if constexpr (NANCHK && !kRowSeg) {  // (kRowSeg: the message wave tests the unaries)
    nan_seen |= any_nan(a0);
    const bool any = __ballot(nan_seen) != 0;  // all lanes take part
    if (lane == 0) a.nan_flags[c] = any ? 1 : 0;
  }
  if constexpr (MODE != kRowsDecode) c0 = ld_node<LPL, FIT>(Cb, lane, D);
  th0 = theta_of(a0);
  }
  __syncthreads();  // kRowSeg: the checkpoints and u_lds are now visible to wave 1
  if constexpr (kRowSeg) {
    if (wid == 1) {
      row_messages();
      return;
    }
  }
  Vec<LPL> M0;
#pragma unroll
  for (int k = 0; k < LPL; ++k) M0.v[k] = th0.v[k] + bh.v[k];
  const double Lambda = bsum + (double)chain_min(local_min(M0));

  {
    // Forward pass: keep g_i = gamma (R + Bh) + excess, pass V = R - gamma (R + Bh) on.
    // Step i's operands: Bh_i, the read unaries of node i+1 and the costs of
    // node i+1 (columns: they form A_{i+1}) or of node i (rows: they form the
    // stored C - A'_i).
    const Rsrc rC = chain_rsrc(Cb, kCols ? 0 : (long)(n - 1) * nstride + D);  // (rows)
    auto load_f = [&](int i, Vec<LPL>& bv, Vec<LPL>& av, Vec<LPL>& cv) {
      const int node = i < nb ? i : nb - 1;
      if constexpr (kCols) {
        bv = ld_node<LPL, FIT>(msg + (long)node * D, lane, D);
        av = ld_node<LPL, FIT>(Ab + (node + 1) * nstride, lane, D);
        cv = ld_node<LPL, FIT>(Cb + (node + 1) * nstride, lane, D);
      } else {
        bv = ld_buf<LPL, FIT>(rM, node * D * 4, lane, D);
        av = ld_buf<LPL, FIT>(rA, (node + 1) * strideB, lane, D);
        cv = ld_buf<LPL, FIT>(rC, node * strideB, lane, D);
      }
    };
    // weights of steps i0 .. i0+63 of the forward pass (edge i)
    auto wlane_f = [&](int i0) { return w_lds[max(min(i0 + lane, n - 2), 0)]; };
    auto wlane_f2 = [&](int i0) { return PE ? w2_lds[max(min(i0 + lane, n - 2), 0)] : 0.f; };
    Vec<LPL> R = th0;
    Vec<LPL> a_cur = kCols ? row_unaries(a0, c0) : a0;  // A_0
    // Rows: the costs of the last node, for its stored C - A'.
    Vec<LPL> c_last;
    if constexpr (!kCols) c_last = ld_buf<LPL, FIT>(rC, (n - 1) * strideB, lane, D);
    // The float64 kept constant (the chain minimum this pass leaves behind) is
    // formed from the per-node minima v_i after the pass: chain_kept().
    // step_f takes Bh_i, A_{i+1} and theta_{i+1} (the read unaries) and returns
    // the node's new unaries; the caller stores them.  used() runs once Bh_i is
    // read.
    auto step_f = [&](int i, const Vec<LPL>& Bi, const Vec<LPL>& an, const Vec<LPL>& thn, float wi, float wi2,
                      auto&& used) {
      Vec<LPL> V, nr;
      float lm;
      if constexpr (FIT == kFitFull) {
        lm = near_block<LPL, DC, PE, 2>(V, R, Bi, wi, L1v, a.delta, cc, nr);
      } else {
#pragma unroll
        for (int k = 0; k < LPL; ++k) V.v[k] = valid[k] ? fmaf(-kGamma, R.v[k] + Bi.v[k], R.v[k]) : kInfF;
        lm = near_block<LPL, DC, PE, 0>(V, V, V, wi, L1v, a.delta, cc, nr);
      }
      __builtin_amdgcn_sched_barrier(kSchedValu);
      used();
      const float v = near_min_rest<LPL, DC>(lm);
      fw_lds[i] = v;  // every lane writes the same value
      const Vec<LPL> m = minconv<LPL, PE>(V, nr, v, wi, wi2, L2v);
      Vec<LPL> mm;
#pragma unroll
      for (int k = 0; k < LPL; ++k) mm.v[k] = valid[k] ? m.v[k] : -kInfF;
      Vec<LPL> nx, am;
      near_max_minus<LPL, DC, PE>(mm, m, thn, wi, L1v, a.delta, cc, nx, am);
      Vec<LPL> out;
#pragma unroll
      for (int k = 0; k < LPL; ++k) {
        // g = gamma (R + Bh) + excess, excess = V - max(m, near_max(m) - w L1); with
        // V = R - gamma (R + Bh) that is R - max(...), formed directly.
        const float g = keep(k) ? R.v[k] - fmaxf(m.v[k], nx.v[k]) : 0.f;
        out.v[k] = MODE == kRowsMinorant ? a_cur.v[k] - g : a_cur.v[k] + g;
        R.v[k] = keep(k) ? am.v[k] - v : kInfF;
      }
      a_cur = an;
      return out;
    };
    // Stores node i's result: columns A'_i, rows C_i - A'_i (ci: C_i).
    auto store_f = [&](int i, const Vec<LPL>& out, const Vec<LPL>& ci) {
      if constexpr (kCols) st_node<LPL, FIT>(Aw + i * nstride, lane, D, out);
      else st_buf<LPL, FIT>(rW, i * strideB, lane, D, col_unaries(out, ci));
    };
    if constexpr (kRowSeg) {
      // Forward step i' = i + g (see row_messages): A_{i+1} in register ring
      // slot i' % P (P = kRowRing*KR, so the segments i' = q*KR .. q*KR+KR-1
      // line up with the blocks), Bh_i from LDS ring slot i' % P, read two
      // steps ahead.  Segments 0 and 1 are complete at the first barrier;
      // before the first step of segment q (1 <= q <= M-2) a barrier pairs
      // with wave 1's barrier after segment q+1, which also frees the slots of
      // segment q-1 for segment q+2.
      constexpr int K = KR;
      const int M = (nb + K - 1) / K;
      const int g = M * K - nb;
      const int nbp = M * K;
      // Register ring slot j (steps ip = j mod P) holds A_{i+1}, read by step
      // ip as theta_{i+1} and by step ip + 1 as its own node's unaries A_i; it
      // is refilled after that second read, so neither read copies it out.
      // Node of step ip's A (A_{i+1}, i = ip - g); virtual steps (i < 0) read
      // A_0, which the first real step reads as its own node's unaries.
      auto node_a = [&](int ip) { return max(min(ip - g, nb - 1) + 1, 0); };
      // rc slot j holds C_i of the node step ip stores, refilled after the store.
      auto node_c = [&](int ip) { return max(min(ip - g, nb - 1), 0); };
      // Byte offsets of a block's refills (A of step ip0 + P + lane), one per
      // lane: a step takes its offset with v_readlane instead of clamping it.
      auto refill_offsets = [&](int ip0) { return node_a(ip0 + P + lane) * strideB; };
      auto wl = [&](int ip0) { return w_lds[max(min(ip0 - g + lane, n - 2), 0)]; };
      auto wl2 = [&](int ip0) { return PE ? w2_lds[max(min(ip0 - g + lane, n - 2), 0)] : 0.f; };
      Vec<LPL> bm[3];
      if (nb > 0) {
        // slots 0 .. P-2: steps 0 .. P-2; slot P-1: A of step -1 (A_0, the first
        // step's own unaries), its C that of step P-1
#pragma unroll
        for (int j = 0; j < P; ++j) {
          ra[j] = ld_buf<LPL, FIT>(rA, node_a(j < P - 1 ? j : -1) * strideB, lane, D);
          rc[j] = ld_buf<LPL, FIT, kCostAux>(rC, node_c(j) * strideB, lane, D);
        }
        lds_barrier();  // segments 0 and 1 are in the ring
        bm[0] = ld_ring<LPL>(ring, lane);
        bm[1] = ld_ring<LPL>(ring + kNS, lane);
      }
      float wf = wl(0), wf2 = wl2(0);
      // Step j of the block at ip0 (ao: the block's refill offsets, aop: the
      // previous block's).  LOW: the block may start with virtual steps (i < 0,
      // skipped); TAIL: no refills, steps past the chain skipped.
      auto fstep = [&](int ip0, int ao, int aop, int j, bool LOW, bool TAIL) {
        const int ip = ip0 + j;
        if (TAIL && ip >= nbp) return;
        if (j % K == 0) {
          const int q = ip / K;
          if (q >= 1 && q <= M - 2) lds_barrier();
        }
        const int i = ip - g;
        const int jp = (j + P - 1) % P;  // the previous step's slot
        a_cur = ra[jp];                  // A_i
        auto next_msg = [&]() { bm[(j + 2) % 3] = ld_ring<LPL>(ring + ((j + 2) % P) * kNS, lane); };
        if (!LOW || i >= 0)
          store_f(i,
                  step_f(i, bm[j % 3], ra[j], theta_of(ra[j]), lane_weight(wf, j), PE ? lane_weight(wf2, j) : 0.f,
                         next_msg),
                  rc[j]);
        else
          next_msg();
        if (!TAIL) {
          // C_i and A_i are read: their slots take C of step ip + P and A of
          // step ip - 1 + P.
          rc[j] = ld_buf<LPL, FIT, kCostAux>(rC, __builtin_amdgcn_readlane(ao, j) - strideB, lane, D);
          ra[jp] = ld_buf<LPL, FIT>(rA, j > 0 ? __builtin_amdgcn_readlane(ao, j - 1) : __builtin_amdgcn_readlane(aop, P - 1),
                                     lane, D);
        }
      };
      int i0p = 0;
      if (nbp >= P) {
        int aop = refill_offsets(-P);
        {
          const float wn = wl(P), wn2 = wl2(P);
          const int ao = refill_offsets(0);
#pragma unroll
          for (int j = 0; j < P; ++j) fstep(0, ao, aop, j, true, false);
          aop = ao;
          wf = wn;
          wf2 = wn2;
        }
        for (i0p = P; i0p + P <= nbp; i0p += P) {
          const float wn = wl(i0p + P), wn2 = wl2(i0p + P);
          const int ao = refill_offsets(i0p);
#pragma unroll
          for (int j = 0; j < P; ++j) fstep(i0p, ao, aop, j, false, false);
          aop = ao;
          wf = wn;
          wf2 = wn2;
        }
      }
      // (the last node's own unaries: a_cur as the last step left it)
#pragma unroll
      for (int j = 0; j < P; ++j) fstep(i0p, 0, 0, j, true, true);
    } else
    if constexpr (kCols && SEG != 0 && seg_len<LPL>() > 0) {
      // Segments of K forward steps i0 .. i0+K-1.  Their nodes i0+1 .. i0+K
      // (unaries and costs), the checkpoint Bh_{min(i0+K, n-1)} (Bh_{n-1} = 0
      // is stored) and the segment's minima u_i and weights w_i (one per lane)
      // are loaded a segment ahead.  Bh_i for the segment is recomputed
      // backwards from the checkpoint with the backward step's own operations
      // and operands (theta_{i+1}, u_i, w_i), so it equals the message the
      // backward pass formed; u_lds[i] still holds the backward minimum until
      // forward step i overwrites it.
      constexpr int K = seg_len<LPL>();
      struct Seg {
        Vec<LPL> a[K], c[K], m;
        float u, w, w2;
      };
      Seg X, Y;
      Vec<LPL> bs[K];
      // Nodes first .. first+K-1 (clamped to the chain) through buffer
      // resources based at the segment: 32-bit offsets, one scalar multiply
      // per node (the host bounds K nodes of a column by 2 GiB).
      auto load_seg = [&](int i0, Seg& B) {
        const int first = min(i0 + 1, n - 1);
        const long span = (long)(K - 1) * nstride + D;
        const Rsrc sA = chain_rsrc(Ab + first * nstride, span);
        const Rsrc sC = chain_rsrc(Cb + first * nstride, span);
#pragma unroll
        for (int t = 0; t < K; ++t) {
          const int off = min(t, n - 1 - first) * strideB;
          B.a[t] = ld_buf<LPL, FIT>(sA, off, lane, D);
          B.c[t] = ld_buf<LPL, FIT, kCostAux>(sC, off, lane, D);
        }
        B.m = ld_node<LPL, FIT>(msg + (long)min(i0 + K, nb) * D, lane, D);
        const int e = max(min(i0 + lane, n - 2), 0);
        B.u = u_lds[e];
        B.w = w_lds[e];
        B.w2 = PE ? w2_lds[e] : 0.f;
      };
      // The segment of cnt (1 .. K) steps from i0, its data in B.
      auto run_seg = [&](int i0, int cnt, const Seg& B) {
        Vec<LPL> Xb = B.m;
#pragma unroll
        for (int t = K - 1; t >= 0; --t) {
          if (t < cnt) {
            const float u = lane_weight(B.u, t);
            Vec<LPL> U, nr;
            near_only<LPL, DC, PE>(U, theta_of(B.a[t]), Xb, lane_weight(B.w, t), L1v, a.delta, cc, nr);
            const Vec<LPL> m = minconv<LPL, PE>(U, nr, u, lane_weight(B.w, t), PE ? lane_weight(B.w2, t) : 0.f, L2v);
#pragma unroll
            for (int k = 0; k < LPL; ++k) Xb.v[k] = keep(k) ? m.v[k] - u : 0.f;
            bs[t] = Xb;
          }
        }
        const Rsrc sW = chain_rsrc(Aw + i0 * nstride, (long)(K - 1) * nstride + D);
#pragma unroll
        for (int t = 0; t < K; ++t)
          if (t < cnt)
            st_buf<LPL, FIT>(sW, t * strideB, lane, D,
                              step_f(i0 + t, bs[t], row_unaries(B.a[t], B.c[t]), theta_of(B.a[t]),
                                     lane_weight(B.w, t), PE ? lane_weight(B.w2, t) : 0.f, []() {}));
      };
      // Two segments per iteration, alternating between X and Y; the next
      // segment's loads are issued before the current segment's steps.
      load_seg(0, X);
      int i0 = 0;
      for (;;) {
        if (i0 + K >= nb) break;  // X holds the last segment
        load_seg(i0 + K, Y);
        __builtin_amdgcn_sched_barrier(0);
        run_seg(i0, K, X);
        i0 += K;
        if (i0 + K >= nb) {
          X = Y;
          break;
        }
        load_seg(i0 + K, X);
        __builtin_amdgcn_sched_barrier(0);
        run_seg(i0, K, Y);
        i0 += K;
      }
      if (i0 < nb) run_seg(i0, nb - i0, X);
    } else {
    if (nb > 0) {
#pragma unroll
      for (int j = 0; j < P; ++j) load_f(j, rb[j], ra[j], rc[j]);
    }
    int i0 = 0;
    float wf = wlane_f(0), wf2 = wlane_f2(0);
    for (; i0 + P <= nb; i0 += P) {
      const float wnext = wlane_f(i0 + P), wnext2 = wlane_f2(i0 + P);
#pragma unroll
      for (int j = 0; j < P; ++j) {
        // A_{i+1} lives on as the next step's a_cur: copied out of the slot
        // (columns form it from C and B).
        Vec<LPL> an, thn;
        if constexpr (kCols) {
          an = row_unaries(ra[j], rc[j]);
          thn = theta_of(ra[j]);
          pin(an);
          pin(thn);
        } else {
          an = fresh(ra[j]);
          thn = an;
        }
        const Vec<LPL> ci = fresh(rc[j]);  // (rows: C_i)
        store_f(i0 + j,
                step_f(i0 + j, rb[j], an, thn, lane_weight(wf, j), PE ? lane_weight(wf2, j) : 0.f,
                       [&]() { load_f(i0 + j + P, rb[j], ra[j], rc[j]); }),
                ci);
      }
      wf = wnext;
      wf2 = wnext2;
    }
#pragma unroll
    for (int j = 0; j < P; ++j)
      if (i0 + j < nb)
        store_f(i0 + j,
                step_f(i0 + j, rb[j], kCols ? row_unaries(ra[j], rc[j]) : ra[j], theta_of(ra[j]),
                       lane_weight(wf, j), PE ? lane_weight(wf2, j) : 0.f, []() {}),
                rc[j]);
    }
    {
      Vec<LPL> out;
#pragma unroll
      for (int k = 0; k < LPL; ++k)
        out.v[k] = MODE == kRowsMinorant ? a_cur.v[k] - R.v[k] : a_cur.v[k] + R.v[k];
      if constexpr (kCols)
        st_node<LPL, FIT>(Aw + (n - 1) * nstride, lane, D, out);
      else
        st_node<LPL, FIT>(Aw + (n - 1) * nstride, lane, D, col_unaries(out, c_last));
    }
    const double kept = chain_kept(fw_lds, b_lds, n, lane, kGammaD);
    if (lane == 0) {
      a.lam[c] = Lambda;
      a.kept[c] = kept;
    }
  }
}

// Chain sweep on three waves per chain (delta = 2), for the sweeps whose time is
// the steps of one resident set of chains and not the bytes they move
// (use_line()).
//
// A wave alone on its SIMD pays 4 cycles for every instruction, dependent or
// not, but 16-24 for a global load or store, 16-20 for an LDS store and 12 for
// an LDS read (measured, stand-alone).  A forward step of k_chain spends 100 of
// its 304 cycles on its memory instructions (two loads, a store, an LDS read and
// an LDS store; 128 ns measured at 1242 x 375 x 128).  Here the chain wave
// touches no global memory in its forward pass: 47 instructions, one LDS read
// and one LDS store per step (103 ns).
//
//   Backward pass (chain wave): theta through a register ring, every K-th
//     message stored as a checkpoint (end-aligned, at nodes n-1 - m K).  The
//     per-node minimum is kept in a register: one DPP move writes it to the
//     step's quad of lanes, and 16 steps' values go to LDS at once.  The messages
//     of the first three segments, the pass's last, go straight to the ring, so
//     that the forward pass starts without waiting for a recomputation.
//   Forward pass, in segments of K steps (forward step i' = i + g of node i, g
//     virtual steps align the segments with the checkpoints).  Between barriers
//     q and q + 1
//       the chain wave runs segment q: it reads (Bh_i, theta_{i+1}) as one vector
//         from an LDS ring of three segments, two steps ahead, and writes its
//         result (rows: A'_i = A_i - g_i; columns: g_i) to a ring of two;
//       the output wave stores segment q - 1 (rows: C_i - A'_i; columns:
//         (C_i - B_i) + g_i);
//       the message wave (first: the float64 offsets b_i) recomputes the messages
//         of segment q + 2 from the checkpoint at its end into the slot that
//         segment q - 1 has left, with the backward step's own operations and
//         operands, so they are the messages it formed, bit for bit.
//
// Loads run 4 (costs) and 6 segments (theta) ahead: 1242 x 256 chains of 128
// labels 242 -> 237 us against 2 and 3.  Up to two chains per CU share a
// workgroup of eight waves, two of them idle: waves go to the four SIMDs in turn,
// so that each chain wave keeps a SIMD to itself.
//
// Measured, one sweep (us, k_chain -> this): rows 320 x 240 x 32 72 -> 50,
// 744 x 496 x 64 141 -> 115, 1242 x 128 x 128 261 -> 212 (88 of them backward),
// 1242 x 375 x 128 270 -> 262 (streaming the costs; 954 MB, 3.6 TB/s); columns
// 320 x 240 x 32 73 -> 40, 744 x 496 x 64 126 -> 95.
constexpr int kLineK = 8;
constexpr int kLineRing = 3 * 2 + 2;  // segments of node vectors in the two rings
enum LineRole { kChain = 0, kMessages = 1, kOut = 2, kIdle = 3 };

// LDS of one chain: b and their sum, w, u, v, [w2], rounded to 16 bytes, then the rings.
constexpr size_t line_lds(int lpl, bool per_edge, int n) {
  return sizeof(float) *
         ((((per_edge ? 6 : 5) * (size_t)n + 5) & ~(size_t)3) + (size_t)kLineRing * kLineK * 64 * lpl);
}

template <int LPL, int FIT, bool PE, bool COLS, bool NANCHK>
__global__ __launch_bounds__(512) void k_line(ChainArgs a) {
  extern __shared__ double lds_line[];
  constexpr int K = kLineK, DC = 2, P = 32, NS = 64 * LPL;
  const int n = a.n, D = a.D;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const bool two = blockDim.x > 256;  // two chains in the workgroup
  const int cs = two ? (wave >> 1) & 1 : 0;
  const int role = !two ? wave : wave < 4 ? wave & 1 : wave & 1 ? kOut : kIdle;
  const int c_slot = blockIdx.x * (two ? 2 : 1) + cs;
  const int c = min(c_slot, a.n_chains - 1);
  // per chain: b and their sum (doubles), w, u, v, [w2], then the rings at a 16-byte boundary
  const int head = ((PE ? 6 : 5) * n + 5) & ~3;
  const int chain_floats = head + kLineRing * K * NS;
  double* b_lds = lds_line + cs * (chain_floats / 2);
  float* w_lds = reinterpret_cast<float*>(b_lds + n + 1);
  float* u_lds = w_lds + n;
  float* v_lds = u_lds + n;
  float* w2_lds = v_lds + n;  // PE only
  float* msg_ring = reinterpret_cast<float*>(b_lds) + head;  // [3][K] nodes of 64 x (Bh, theta)
  float* out_ring = msg_ring + 3 * K * 2 * NS;               // [2][K] nodes, by segment
  ShiftCarry cc;
  const float L1v = in_vgpr(a.L1), L2v = in_vgpr(a.L2);
  const long pbase = (long)c * a.pcs;
  const int strideB = (int)(a.pns * D * 4);
  const long span = (long)(n - 1) * a.pns * D + D;
  const Rsrc rT = chain_rsrc((COLS ? a.A : a.A_in) + pbase * D, span);  // theta: the sweep's unaries
  const Rsrc rC = chain_rsrc(a.cost + pbase * D, span);
  const Rsrc rW = chain_rsrc(a.A + pbase * D, span);
  const Rsrc rM = chain_rsrc(a.msg + (long)c * n * D, (long)n * D);
  const bool valid = FIT == kFitFull || lane * LPL < D;  // this lane has labels
  const float* __restrict__ wb = a.w + pbase * a.wmul;
  const float* __restrict__ wb2 = PE ? a.w2 + pbase * a.wmul : nullptr;
  const long wstep = a.pns * a.wmul;
  const int nb = n - 1, M = (nb + K - 1) / K, g = M * K - nb;
  auto fill_weights = [&]() {  // by the message and the output wave
    for (int i = (role - kMessages) * 64 + lane; i < nb; i += 128) {
      w_lds[i] = wb[(long)i * wstep];
      if constexpr (PE) w2_lds[i] = wb2[(long)i * wstep];
    }
  };
  if (role == kIdle || c_slot >= a.n_chains) {  // the same barriers, no work
    __syncthreads();
    __syncthreads();
    for (int q = 1; q <= M; ++q) lds_barrier();
    return;
  }
  auto theta_of = [&](const Vec<LPL>& x) { return masked<LPL, FIT>(x, lane, D, kInfF); };
  auto ld_theta = [&](int node) { return ld_buf<LPL, FIT>(rT, node * strideB, lane, D); };

  auto ib = [&](int q) { return q * K - g; };  // node of a segment's first step
  // The two halves of a lane's vector in the message ring (64-bit stores, as everywhere).
  auto put_msg = [&](float* d, const Vec<LPL>& x) {
    if constexpr (LPL == 2) {
      *reinterpret_cast<float2*>(d) = make_float2(x.v[0], x.v[1]);
      asm volatile("" ::: "memory");
    } else {
      d[0] = x.v[0];
    }
  };
  auto put_theta = [&](float* d, const Vec<LPL>& x) {
    if constexpr (LPL == 2)
      *reinterpret_cast<float2*>(d + 2) = make_float2(x.v[0], x.v[1]);
    else
      d[1] = x.v[0];
  };

  if (role == kOut) {
    // ---- output wave: the costs run four segments ahead
    constexpr int F = 4;
    Vec<LPL> C[F][K], B[COLS ? F : 1][K];
    auto load = [&](int q, auto k) {
      constexpr int kk = decltype(k)::value;
      auto off = [&](int t) { return min(max(ib(min(q, M - 1)) + t, 0), n - 1) * strideB; };
      if (a.stream) {
#pragma unroll
        for (int t = 0; t < K; ++t) C[kk][t] = ld_buf<LPL, FIT, kStream>(rC, off(t), lane, D);
      } else {
#pragma unroll
        for (int t = 0; t < K; ++t) C[kk][t] = ld_buf<LPL, FIT>(rC, off(t), lane, D);
      }
      if constexpr (COLS) {
#pragma unroll
        for (int t = 0; t < K; ++t) B[kk][t] = ld_buf<LPL, FIT>(rT, off(t), lane, D);
      }
    };
    // Stores segment q (q % F = k) after barrier q + 1, then loads segment q + F.
    auto store = [&](int q, auto k) {
      constexpr int kk = decltype(k)::value;
      const float* src = out_ring + (kk % 2) * K * NS;
      Vec<LPL> r[K];
#pragma unroll
      for (int t = 0; t < K; ++t) r[t] = ld_ring<LPL>(src + t * NS, lane);
#pragma unroll
      for (int t = 0; t < K; ++t) {
#pragma unroll
        for (int e = 0; e < LPL; ++e)
          r[t].v[e] = COLS ? (C[kk][t].v[e] - B[COLS ? kk : 0][t].v[e]) + r[t].v[e] : C[kk][t].v[e] - r[t].v[e];
        const int i = ib(q) + t;
        if (kk != 0 || i >= 0) st_buf<LPL, FIT>(rW, i * strideB, lane, D, r[t]);
      }
      load(q + F, k);
    };
    fill_weights();
    __syncthreads();
    __syncthreads();
    unroll_steps<F>([&](auto k) { load(decltype(k)::value, k); });
    for (int q = 0; q < M; q += F)
      unroll_steps<F>([&](auto k) {
        const int qk = q + decltype(k)::value;
        if (qk < M) {
          lds_barrier();  // qk + 1
          store(qk, k);
        }
      });
    return;
  }
  if (role == kMessages) {
    // ---- message wave
    struct Seg {
      Vec<LPL> a[K], m;
      float u, w, w2;
    };
    constexpr int F = 6;  // segments in flight
    Seg T[F];
    auto load_t = [&](int q, Seg& S) {           // theta of nodes ib + 1 .. ib + K
#pragma unroll
      for (int t = 0; t < K; ++t) S.a[t] = ld_theta(min(max(ib(min(q, M - 1)) + t + 1, 1), n - 1));
    };
    auto load_m = [&](int q, Seg& S) {  // the checkpoint and the segment's minima and weights, one per lane
      S.m = ld_buf<LPL, FIT>(rM, min(ib(q) + K, n - 1) * D * 4, lane, D);
      const int e = max(min(ib(q) + lane, n - 2), 0);
      S.u = u_lds[e];
      S.w = w_lds[e];
      S.w2 = PE ? w2_lds[e] : 0.f;
    };
    fill_weights();
    bool nan1 = false;
    if constexpr (NANCHK) {  // the nodes that its segments do not read
#pragma unroll
      for (int i = 0; i <= 3 * K; ++i) nan1 |= any_nan(ld_theta(min(i, n - 1)));
    }
    unroll_steps<F>([&](auto k) { load_t(3 + decltype(k)::value, T[(3 + decltype(k)::value) % F]); });
    __syncthreads();  // the weights are in LDS
    __syncthreads();  // the checkpoints, the minima and segments 0 .. 2 are visible
    // The messages of segment q >= 3 into ring slot q % 3.
    auto messages = [&](int q, const Seg& S, int slot) {
      float* dst = msg_ring + slot * K * 2 * NS + lane * 2 * LPL;
      Vec<LPL> X = S.m;
#pragma unroll
      for (int t = K - 1; t >= 0; --t) {
        if constexpr (NANCHK) nan1 |= any_nan(S.a[t]);
        const Vec<LPL> th = theta_of(S.a[t]);
        const float u = lane_weight(S.u, t);
        Vec<LPL> U, nr;
        near_only<LPL, DC, PE>(U, th, X, lane_weight(S.w, t), L1v, 2, cc, nr);
        const Vec<LPL> m = minconv<LPL, PE>(U, nr, u, lane_weight(S.w, t), PE ? lane_weight(S.w2, t) : 0.f, L2v);
#pragma unroll
        for (int k = 0; k < LPL; ++k) X.v[k] = m.v[k] - u;
        float* d = dst + t * 2 * NS;
        put_msg(d, X);
        put_theta(d, th);
      }
    };
    unroll_steps<3>([&](auto k) { load_m(3 + decltype(k)::value, T[3 + decltype(k)::value]); });
    const double bsum = chain_offsets(u_lds, b_lds, n, lane);  // b_0 = sum of all minima
    if (lane == 0) b_lds[n] = bsum;
    // Segment q (q % F = k) between barriers q - 2 and q - 1, then the checkpoint
    // of segment q + 3 and theta of q + F.
    for (int q = 1; q <= min(M, 2); ++q)
      if (q < 2 || M < 4) lds_barrier();
    for (int q0 = 0; q0 < M; q0 += F)
      unroll_steps<F>([&](auto k) {
        constexpr int kk = decltype(k)::value;
        const int q = q0 + kk;
        if ((kk >= 3 || q0 > 0) && q < M) {
          messages(q, T[kk], kk % 3);
          load_m(q + 3, T[(kk + 3) % F]);
          load_t(q + F, T[kk]);
          lds_barrier();  // q - 1
        }
      });
    for (int q = max(M - 1, 3); q <= M; ++q) lds_barrier();
    if constexpr (NANCHK) {
      const bool any = __ballot(nan1) != 0;  // all lanes take part
      if (lane == 0) a.nan_flags[c] = any ? 1 : 0;
    }
    return;
  }

  // ---- chain wave, backward pass: step s handles i = n-2-s
  Vec<LPL> bh;
#pragma unroll
  for (int k = 0; k < LPL; ++k) bh.v[k] = 0.f;
  st_buf<LPL, FIT>(rM, (n - 1) * D * 4, lane, D, bh);  // Bh_{n-1} = 0, the last segment's checkpoint
  auto wlane_b = [&](int s0) { return w_lds[max(n - 2 - (s0 + lane), 0)]; };
  auto wlane_b2 = [&](int s0) { return PE ? w2_lds[max(n - 2 - (s0 + lane), 0)] : 0.f; };
  // Returns the minimum; refill() re-issues the ring slot th came from.
  auto step_b = [&](const Vec<LPL>& th, float wi, float wi2, auto&& refill) {
    Vec<LPL> U, nr;
    const float lm = near_block<LPL, DC, PE, 1>(U, th, bh, wi, L1v, 2, cc, nr);
    __builtin_amdgcn_sched_barrier(kSchedValu);
    refill();
    const float u = near_min_rest<LPL, DC, FIT == kFitHalf ? 2 : 4>(lm);
    const Vec<LPL> m = minconv<LPL, PE>(U, nr, u, wi, wi2, L2v);
#pragma unroll
    for (int k = 0; k < LPL; ++k) bh.v[k] = m.v[k] - u;
    return u;
  };
  // Puts a uniform value into the lanes 4 slot .. 4 slot + 3 of col.
  auto collect = [&](float& col, float x, auto slot) {
    constexpr int S = decltype(slot)::value;
    col = dpp_f<0xe4, 1 << (S >> 2), 1 << (S & 3), false>(col, x);
  };
  // The steps down to the first three segments run through the register ring;
  // those of the first three segments, the last, have their unaries from the start.
  const int nhi = max(nb - (3 * K - g), 0);
  Vec<LPL> ra[P], lo[3 * K];
#pragma unroll
  for (int j = 0; j < P; ++j) ra[j] = ld_theta(j < nhi ? n - 1 - j : min(1, nb));
#pragma unroll
  for (int t = 0; t < 3 * K; ++t) lo[t] = ld_theta(max(min(t - g, nb - 1) + 1, 0));
  const Vec<LPL> a0 = theta_of(ld_theta(0)), c_end = ld_buf<LPL, FIT>(rC, nb * strideB, lane, D);
  __syncthreads();  // the weights are in LDS
  int s0 = 0;
  float wv = wlane_b(0), wv2 = wlane_b2(0);
  for (; s0 + P <= nhi; s0 += P) {
    const float wnext = wlane_b(s0 + P), wnext2 = wlane_b2(s0 + P);
    const int bo = (s0 + P + lane < nhi ? n - 1 - (s0 + P + lane) : 1) * strideB;  // refill offsets, one per lane
    float uc = 0.f;
    unroll_steps<P>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      const float u = step_b(theta_of(ra[j]), lane_weight(wv, j), PE ? lane_weight(wv2, j) : 0.f, [&]() {
        ra[j] = ld_buf<LPL, FIT>(rT, __builtin_amdgcn_readlane(bo, j), lane, D);
      });
      collect(uc, u, std::integral_constant<int, j % 16>{});
      if constexpr (j % 16 == 15) u_lds[nb - 1 - (s0 + j - 15 + (lane >> 2))] = uc;
      if constexpr ((j + 1) % K == 0) st_buf<LPL, FIT>(rM, (nb - 1 - (s0 + j)) * D * 4, lane, D, bh);
    });
    wv = wnext;
    wv2 = wnext2;
  }
#pragma unroll
  for (int j = 0; j < P; ++j)
    if (s0 + j < nhi) {
      u_lds[nb - 1 - (s0 + j)] = step_b(theta_of(ra[j]), lane_weight(wv, j), PE ? lane_weight(wv2, j) : 0.f, []() {});
      if ((j + 1) % K == 0) st_buf<LPL, FIT>(rM, (nb - 1 - (s0 + j)) * D * 4, lane, D, bh);
    }
  {
    const int e = max(min(lane - g, nb - 1), 0);
    const float wlow = w_lds[e], wlow2 = PE ? w2_lds[e] : 0.f;
    float* d = msg_ring + lane * 2 * LPL;
    float uc = 0.f;
    unroll_steps<3 * K>([&](auto tc) {
      constexpr int t = 3 * K - 1 - decltype(tc)::value;  // the node's forward step
      if (t < M * K && t >= g) {
        const Vec<LPL> th = theta_of(lo[t]);
        const float u = step_b(th, lane_weight(wlow, t), PE ? lane_weight(wlow2, t) : 0.f, []() {});
        collect(uc, u, std::integral_constant<int, t % 16>{});
        put_msg(d + t * 2 * NS, bh);
        put_theta(d + t * 2 * NS, th);
      }
      if constexpr (t % 16 == 0) {
        const int i = t - g + (lane >> 2);
        if (i >= 0 && i < nb - nhi) u_lds[i] = uc;  // (a quad writes its step's value)
      }
    });
  }
  __syncthreads();
  Vec<LPL> M0;
#pragma unroll
  for (int k = 0; k < LPL; ++k) M0.v[k] = a0.v[k] + bh.v[k];
  const float m0 = chain_min(local_min(M0));

  // ---- chain wave, forward pass
  Vec<LPL> R = a0, t_cur = a0;  // theta of the current node
  struct Pair {
    Vec<LPL> b, t;
  };
  auto rd = [&](int slot) {  // node slot 0 .. 3K-1 of the message ring
    const float* p = msg_ring + slot * 2 * NS + lane * 2 * LPL;
    Pair r;
    if constexpr (LPL == 2) {
      const float4 x = *reinterpret_cast<const float4*>(p);
      r.b.v[0] = x.x; r.b.v[1] = x.y; r.t.v[0] = x.z; r.t.v[1] = x.w;
    } else {
      const float2 x = *reinterpret_cast<const float2*>(p);
      r.b.v[0] = x.x; r.t.v[0] = x.y;
    }
    return r;
  };
  auto wl = [&](int q) { return w_lds[max(min(q * K - g + lane, n - 2), 0)]; };
  auto wl2 = [&](int q) { return PE ? w2_lds[max(min(q * K - g + lane, n - 2), 0)] : 0.f; };
  if (M > 0) {
    Pair pr[3];
    pr[0] = rd(0);
    pr[1] = rd(1);
    float wf = wl(0), wf2 = wl2(0);
    // Segment q in ring slots q % 3 (messages) and q % 2 (results); low: it may
    // start with virtual steps.
    auto segment = [&](int q, auto slotc, auto outc, bool low) {
      constexpr int slot = decltype(slotc)::value, oslot = decltype(outc)::value;
      const float wn = wl(q + 1), wn2 = wl2(q + 1);
      float vc = 0.f;
      unroll_steps<K>([&](auto tc) {
        constexpr int t = decltype(tc)::value, j = slot * K + t;
        const Pair x = pr[j % 3];
        auto next = [&]() { pr[(j + 2) % 3] = rd((j + 2) % (3 * K)); };
        if (!low || q * K + t >= g) {
          const float wi = lane_weight(wf, t), wi2 = PE ? lane_weight(wf2, t) : 0.f;
          Vec<LPL> V, nr;
          float lm;
          if constexpr (FIT == kFitFull) {
            lm = near_block<LPL, DC, PE, 2>(V, R, x.b, wi, L1v, 2, cc, nr);
          } else {
#pragma unroll
            for (int k = 0; k < LPL; ++k) V.v[k] = valid ? fmaf(-kGamma, R.v[k] + x.b.v[k], R.v[k]) : kInfF;
            lm = near_block<LPL, DC, PE, 0>(V, V, V, wi, L1v, 2, cc, nr);
          }
          __builtin_amdgcn_sched_barrier(kSchedValu);
          next();
          const float v = near_min_rest<LPL, DC, FIT == kFitHalf ? 2 : 4>(lm);
          collect(vc, v, tc);
          const Vec<LPL> m = minconv<LPL, PE>(V, nr, v, wi, wi2, L2v);
          Vec<LPL> mm, nx, am, o;
#pragma unroll
          for (int k = 0; k < LPL; ++k) mm.v[k] = FIT == kFitFull || valid ? m.v[k] : -kInfF;
          near_max_minus<LPL, DC, PE>(mm, m, x.t, wi, L1v, 2, cc, nx, am);
#pragma unroll
          for (int k = 0; k < LPL; ++k) {
            const float gk = R.v[k] - fmaxf(m.v[k], nx.v[k]);
            o.v[k] = COLS ? gk : t_cur.v[k] - gk;
            R.v[k] = am.v[k] - v;
          }
          st_ring<LPL>(out_ring + (oslot * K + t) * NS, lane, o);
          t_cur = x.t;
        } else {
          next();
        }
      });
      // lanes 4 t .. 4 t + 3 hold step t's minimum
      const int i = q * K - g + (lane >> 2);
      if (lane < 4 * K && i >= 0) v_lds[i] = vc;
      wf = wn;
      wf2 = wn2;
      lds_barrier();  // q + 1
    };
    // six segments bring both rings back to their first slots
    constexpr std::integral_constant<int, 0> s0c;
    constexpr std::integral_constant<int, 1> s1c;
    constexpr std::integral_constant<int, 2> s2c;
    segment(0, s0c, s0c, true);
    for (int q = 1;; q += 6) {
      if (q >= M) break;
      segment(q, s1c, s1c, false);
      if (q + 1 >= M) break;
      segment(q + 1, s2c, s0c, false);
      if (q + 2 >= M) break;
      segment(q + 2, s0c, s1c, false);
      if (q + 3 >= M) break;
      segment(q + 3, s1c, s0c, false);
      if (q + 4 >= M) break;
      segment(q + 4, s2c, s1c, false);
      if (q + 5 >= M) break;
      segment(q + 5, s0c, s0c, false);
    }
  }
  Vec<LPL> out;
#pragma unroll
  for (int k = 0; k < LPL; ++k)
    out.v[k] = COLS ? (c_end.v[k] - t_cur.v[k]) + R.v[k] : c_end.v[k] - (t_cur.v[k] - R.v[k]);
  st_buf<LPL, FIT>(rW, (n - 1) * strideB, lane, D, out);
  const double kept = chain_kept(v_lds, b_lds, n, lane, kGammaD);
  if (lane == 0) {
    a.lam[c] = (M > 0 ? b_lds[n] : 0.0) + (double)m0;  // (n = 1: nothing orders the waves)
    a.kept[c] = kept;
  }
}

// Sum of u_0 .. u_{n-2} in float64 (64 lanes, contiguous segments).
__device__ double chain_total(const float* u, int n, int lane) {
  const int m = n - 1;
  const int L = (m + 63) / 64;
  const int s0 = min(lane * L, m), s1 = min(s0 + L, m);
  double tot = 0.0;
  for (int j = s0; j < s1; ++j) tot += (double)u[j];
  return wave_sum_f64(tot);
}

// Runs step(i, A_{i+aoff}, msg_i, w_{i+woff}) for the cnt nodes i = first,
// first + dir, ..., with the unaries (and, with MSG, the message buffer) P nodes
// ahead in a register ring, as in k_chain, and the edge weights w (in LDS, n - 1
// of them) one block ahead in lanes.
template <int LPL, int FIT, int P, bool MSG, bool PE, typename Step>
__device__ __forceinline__ void ring_pass(Rsrc rA, int strideB, Rsrc rM, const float* w_lds, const float* w2_lds,
                                          int n, int D, int lane, int first, int cnt, int dir, int aoff, int woff,
                                          Step&& step) {
  static_assert(P <= 64, "one weight per lane and step of a block");
  if (cnt <= 0) return;
  Vec<LPL> ra[P], rm[P];
  auto load = [&](int s, Vec<LPL>& av, Vec<LPL>& mv) {
    const int i = first + dir * (s < cnt ? s : cnt - 1);
    av = ld_buf<LPL, FIT>(rA, (i + aoff) * strideB, lane, D);
    if constexpr (MSG) mv = ld_buf<LPL, FIT>(rM, i * D * 4, lane, D);
  };
  auto wlane = [&](int s0) { return w_lds[max(min(first + dir * (s0 + lane) + woff, n - 2), 0)]; };
  auto wlane2 = [&](int s0) { return PE ? w2_lds[max(min(first + dir * (s0 + lane) + woff, n - 2), 0)] : 0.f; };
#pragma unroll
  for (int j = 0; j < P; ++j) load(j, ra[j], rm[j]);
  int s0 = 0;
  float wv = wlane(0), wv2 = wlane2(0);
  for (; s0 + P <= cnt; s0 += P) {
    const float wnext = wlane(s0 + P), wnext2 = wlane2(s0 + P);
#pragma unroll
    for (int j = 0; j < P; ++j) {
      const Vec<LPL> av = fresh(ra[j]);
      Vec<LPL> mv;
      if constexpr (MSG) mv = fresh(rm[j]);
      __builtin_amdgcn_sched_barrier(kSchedValu);
      load(s0 + j + P, ra[j], rm[j]);
      step(first + dir * (s0 + j), av, mv, lane_weight(wv, j), PE ? lane_weight(wv2, j) : 0.f);
    }
    wv = wnext;
    wv2 = wnext2;
  }
#pragma unroll
  for (int j = 0; j < P; ++j)
    if (s0 + j < cnt) step(first + dir * (s0 + j), ra[j], rm[j], lane_weight(wv, j), PE ? lane_weight(wv2, j) : 0.f);
}

// Row decode on four waves.  Wave 0 runs the forward messages F from node 0,
// wave 1 the backward messages Bh from node n-1.  Until the midpoint each
// stores its messages in the scratch volume (phase 1); then each goes on into
// the other half (phase 2) and hands its messages to a decision wave through
// an LDS ring of two segments of K nodes: wave 2 decides the nodes mid .. n-1
// (F_i from wave 0's ring, Bh_i from the scratch volume), wave 3 the nodes
// mid-1 .. 0 (Bh_i from wave 1's ring, F_i from the scratch volume).  Phase 2
// runs in rounds: in round r the message waves write segment r into slot r % 2
// and the decision waves decide segment r - 1 from slot (r - 1) % 2; all four
// waves meet at a barrier after every round.  F_i + Bh_i and the decision rule
// are those of the single-wave decode, so the labels are the same; the chain
// latency is n message steps, with no decision work on the message waves.
template <int LPL, int P, int FIT, int DC, bool GAP, bool PE>
__global__ __launch_bounds__(256) void k_decode4(ChainArgs a) {
  extern __shared__ double lds2[];
  constexpr int K = seg_len<LPL>();
  constexpr int ROWS = FIT == kFitHalf ? 2 : 4;
  static_assert(P == kRowRing * K, "the message waves' register ring spans three segments");
  static_assert(P <= 64, "one weight per lane and step of a block");
  constexpr int kNS = 64 * LPL;  // ring stride per node, floats
  const int c = blockIdx.x;
  const int wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // wave-uniform branches
  const int lane = threadIdx.x & 63;
  const int n = a.n, D = a.D;
  ShiftCarry cc;
  const float L1v = in_vgpr(a.L1), L2v = in_vgpr(a.L2);
  const long pbase = (long)c * a.pcs;
  const long nstride = a.pns * (long)D;
  const float* __restrict__ Ab = a.A + pbase * D;
  const float* __restrict__ wb = a.w + pbase * a.wmul;
  const float* __restrict__ wb2 = PE ? a.w2 + pbase * a.wmul : nullptr;
  float* msg = a.msg + (long)c * n * D;
  float* w_lds = reinterpret_cast<float*>(lds2);
  float* u_lds = w_lds + n;
  float* w2_lds = u_lds + n;  // PE only
  float* ring = w_lds + (((PE ? 3 : 2) * n + 3) & ~3);  // [half][slot][K][kNS]
  const int strideB = (int)(nstride * 4);
  const Rsrc rA = chain_rsrc(Ab, (long)(n - 1) * nstride + D);
  const Rsrc rM = chain_rsrc(msg, (long)n * D);
  bool valid[LPL];
#pragma unroll
  for (int j = 0; j < LPL; ++j) valid[j] = FIT == kFitFull || lane * LPL + (FIT == kFitLanes ? 0 : j) < D;
  // (with kFitLanes +inf unaries alone keep the lanes without labels out)
  auto keep = [&](int j) { return FIT != kFitAny || valid[j]; };
  const long wstep = a.pns * a.wmul;
  for (int i = threadIdx.x; i < n - 1; i += 256) {
    w_lds[i] = wb[(long)i * wstep];
    if constexpr (PE) w2_lds[i] = wb2[(long)i * wstep];
  }
  __syncthreads();
  const int mid = n / 2;
  const int len0 = n - mid, len1 = mid;  // phase-2 nodes of waves 0 / 1
  const int S = ((len0 > len1 ? len0 : len1) + K - 1) / K;  // rounds with a segment

  Vec<LPL> X;  // wave 0: F_i, wave 1: Bh_i
  auto fwd = [&](const Vec<LPL>& an, float w, float w2) {  // F_i = A_i + minconv(F_{i-1}; w_{i-1}) - min F_{i-1}
    Vec<LPL> nr;
    const float f = near_min_rest<LPL, DC, ROWS>(near_block<LPL, DC, PE, 0>(X, X, X, w, L1v, a.delta, cc, nr));
    const Vec<LPL> m = minconv<LPL, PE>(X, nr, f, w, w2, L2v);
#pragma unroll
    for (int k = 0; k < LPL; ++k) X.v[k] = an.v[k] + m.v[k] - f;
    X = masked<LPL, FIT>(X, lane, D, kInfF);
  };
  auto bwd = [&](int i, const Vec<LPL>& an1, float w, float w2) {  // Bh_i from Bh_{i+1}, A_{i+1} and w_i
    Vec<LPL> U, nr;
    const Vec<LPL> th = masked<LPL, FIT>(an1, lane, D, kInfF);
    const float u = near_min_rest<LPL, DC, ROWS>(near_block<LPL, DC, PE, 1>(U, th, X, w, L1v, a.delta, cc, nr));
    const Vec<LPL> m = minconv<LPL, PE>(U, nr, u, w, w2, L2v);
#pragma unroll
    for (int k = 0; k < LPL; ++k) X.v[k] = keep(k) ? m.v[k] - u : 0.f;
    u_lds[i] = u;  // every lane writes the same value
  };
  // Label (and, with GAP, the min-marginal gap) of node i from F_i + Bh_i.
  // Every lane stores the same value to the same address (one write, no
  // branch).
  auto decide = [&](int i, const Vec<LPL>& F, const Vec<LPL>& b) {
    const long p = pbase + (long)i * a.pns;
    float best = kInfF;
#pragma unroll
    for (int k = 0; k < LPL; ++k) best = fminf(best, valid[k] ? F.v[k] + b.v[k] : kInfF);
    const float gbest = chain_min<ROWS>(best);
    const float thr = gbest + kTieEps * fmaxf(1.f, fabsf(gbest));
    int bj = LPL;
#pragma unroll
    for (int k = LPL - 1; k >= 0; --k)
      if (valid[k] && F.v[k] + b.v[k] <= thr) bj = k;
    const unsigned long long ball = __ballot(bj < LPL);
    const int first = ball ? __builtin_ctzll(ball) : 0;  // empty only for NaN costs
    const int label = __builtin_amdgcn_readlane(lane * LPL + (bj < LPL ? bj : 0), first);
    if constexpr (GAP) {
      float second = kInfF;
#pragma unroll
      for (int k = 0; k < LPL; ++k) {
        const float mm = valid[k] ? F.v[k] + b.v[k] : kInfF;
        if (lane * LPL + k != label) second = fminf(second, mm);
      }
      a.gap[p] = chain_min<ROWS>(second) - gbest;
    }
    a.labels[p] = label;
  };

  // Phase 1: waves 0 and 1 walk to the midpoint, storing their messages.
  if (wv == 0) {
    X = masked<LPL, FIT>(ld_node<LPL, FIT>(Ab, lane, D), lane, D, kInfF);  // F_0 = A_0
    if (mid > 0) st_node<LPL, FIT>(msg, lane, D, X);
    ring_pass<LPL, FIT, P, false, PE>(rA, strideB, rM, w_lds, w2_lds, n, D, lane, 1, mid - 1, 1, 0, -1,
                                       [&](int i, const Vec<LPL>& an, const Vec<LPL>&, float w, float w2) {
                                         fwd(an, w, w2);
                                         st_buf<LPL, FIT>(rM, i * D * 4, lane, D, X);
                                       });
  } else if (wv == 1) {
#pragma unroll
    for (int k = 0; k < LPL; ++k) X.v[k] = 0.f;  // Bh_{n-1} = 0
    st_node<LPL, FIT>(msg + (long)(n - 1) * D, lane, D, X);
    ring_pass<LPL, FIT, P, false, PE>(rA, strideB, rM, w_lds, w2_lds, n, D, lane, n - 2, n - 1 - mid, -1, 1, 0,
                                       [&](int i, const Vec<LPL>& an1, const Vec<LPL>&, float w, float w2) {
                                         bwd(i, an1, w, w2);
                                         st_buf<LPL, FIT>(rM, i * D * 4, lane, D, X);
                                       });
  }
  __threadfence_block();
  __syncthreads();  // the phase-1 messages are visible to the decision waves

  if (wv < 2) {
    // Phase 2, message waves.  Step j: wave 0 forms F at node mid + j (from
    // A_{mid+j} and w_{mid+j-1}; F_0 = A_0 is X already when mid = 0), wave 1
    // Bh at node mid-1-j (from A_{mid-j} and w_{mid-1-j}).  A runs P steps ahead
    // in a register ring; the block's weights and refill offsets sit one per
    // lane (v_readlane per step).
    const int len = wv == 0 ? len0 : len1;
    float* rbase = ring + wv * 2 * K * kNS;
    auto anode = [&](int j) { return wv == 0 ? min(mid + j, n - 1) : max(mid - j, 0); };
    auto wnode = [&](int j) { return max(min(wv == 0 ? mid + j - 1 : mid - 1 - j, n - 2), 0); };
    Vec<LPL> ra[P];
#pragma unroll
    for (int t = 0; t < P; ++t) ra[t] = ld_buf<LPL, FIT>(rA, anode(t) * strideB, lane, D);
    for (int jb = 0; jb < S * K; jb += P) {
      const float wl = w_lds[wnode(jb + lane)];
      const float wl2 = PE ? w2_lds[wnode(jb + lane)] : 0.f;
      const int ao = anode(jb + P + lane) * strideB;
      const int r0 = jb / K;
#pragma unroll
      for (int t = 0; t < P; ++t) {
        const int j = jb + t;
        const Vec<LPL> an = fresh(ra[t]);
        __builtin_amdgcn_sched_barrier(kSchedValu);
        ra[t] = ld_buf<LPL, FIT>(rA, __builtin_amdgcn_readlane(ao, t), lane, D);
        if (j < len) {
          if (wv == 0) {
            if (j > 0 || mid > 0) fwd(an, lane_weight(wl, t), PE ? lane_weight(wl2, t) : 0.f);
          } else {
            bwd(mid - 1 - j, an, lane_weight(wl, t), PE ? lane_weight(wl2, t) : 0.f);
          }
          st_ring<LPL>(rbase + (((r0 + t / K) & 1) * K + t % K) * kNS, lane, X);
        }
        if ((t + 1) % K == 0 && r0 + t / K < S) lds_barrier();  // end of round r0 + t / K
      }
    }
    lds_barrier();  // round S (the decision waves' last segment)
    if (wv == 1) {
      // Chain minimum: sum of the backward minima + min(A_0 + Bh_0).
      const Vec<LPL> a0 = masked<LPL, FIT>(ld_node<LPL, FIT>(Ab, lane, D), lane, D, kInfF);
      Vec<LPL> M0;
#pragma unroll
      for (int k = 0; k < LPL; ++k) M0.v[k] = a0.v[k] + X.v[k];
      const double Lambda = chain_total(u_lds, n, lane) + (double)chain_min<ROWS>(local_min(M0));
      if (lane == 0) a.lam[c] = Lambda;
    }
  } else {
    // Phase 2, decision waves: wave 2 takes node mid + j with F from wave 0's
    // ring and Bh from the scratch volume, wave 3 node mid-1-j with Bh from
    // wave 1's ring and F from the scratch volume.  The scratch messages of the
    // next segment are loaded while this one is decided.
    const int h = wv - 2;
    const int len = h == 0 ? len0 : len1;
    const float* rbase = ring + h * 2 * K * kNS;
    auto node_of = [&](int j) { return h == 0 ? mid + j : mid - 1 - j; };
    auto load_other = [&](int s, Vec<LPL> (&o)[K]) {
#pragma unroll
      for (int t = 0; t < K; ++t) {
        const int i = min(max(node_of(s * K + t), 0), n - 1);
        o[t] = ld_buf<LPL, FIT>(rM, i * D * 4, lane, D);
      }
    };
    auto decide_seg = [&](int s, const Vec<LPL> (&o)[K]) {
      const float* slot = rbase + (s & 1) * K * kNS;
#pragma unroll
      for (int t = 0; t < K; ++t) {
        const int j = s * K + t;
        if (j < len) {
          const Vec<LPL> mine = ld_ring<LPL>(slot + t * kNS, lane);
          if (h == 0)
            decide(node_of(j), mine, o[t]);
          else
            decide(node_of(j), o[t], mine);
        }
      }
    };
    Vec<LPL> OX[K], OY[K];
    load_other(0, OX);
    lds_barrier();  // round 0: segment 0 is written
    for (int r = 1; r <= S;) {
      load_other(min(r, S - 1), OY);
      decide_seg(r - 1, OX);
      lds_barrier();
      if (++r > S) break;
      load_other(min(r, S - 1), OX);
      decide_seg(r - 1, OY);
      lds_barrier();
      ++r;
    }
  }
}

template <int LPL, int MODE, int P, int FIT, int DC, int SEG, bool NANCHK, bool PE>
static void launch_sweep(ChainArgs& a, size_t lds, hipStream_t st) {
  constexpr bool kRowSeg = MODE != kColsMinorant && SEG != 0;
  int cpw = 1;
  if constexpr (kRowSeg) {
    lds = row_seg_lds(LPL, PE, a.n);
    const int cus = cu_count();
    if (a.n_chains > cus && a.n_chains <= 2 * cus && 2 * lds <= kLdsPerCu) cpw = 2;  // one workgroup per CU
    lds *= cpw;
  }
  if (lds > 64 * 1024)  // long chains: allow the LDS beyond the default 64 KB
    (void)hipFuncSetAttribute((const void*)k_chain<LPL, MODE, P, FIT, DC, SEG, NANCHK, PE>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  k_chain<LPL, MODE, P, FIT, DC, SEG, NANCHK, PE><<<(a.n_chains + cpw - 1) / cpw, kRowSeg ? 128 * cpw : 64, lds, st>>>(a);
}

template <int LPL, int FIT, bool PE, bool COLS, bool NANCHK>
static void launch_line(ChainArgs& a, hipStream_t st) {
  size_t lds = line_lds(LPL, PE, a.n);
  const bool two = a.n_chains > cu_count() && 2 * lds <= kLdsPerCu;
  if (two) lds *= 2;
  if (lds > 64 * 1024)
    (void)hipFuncSetAttribute((const void*)k_line<LPL, FIT, PE, COLS, NANCHK>,
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  k_line<LPL, FIT, PE, COLS, NANCHK><<<two ? (a.n_chains + 1) / 2 : a.n_chains, two ? 512 : 192, lds, st>>>(a);
}

// Whether a sweep runs on k_line: where its time is the steps of one resident
// set of chains.  With more chains than LINE_ROUNDS per CU the sweep is bound by
// what it moves, and the three waves of a chain only take the CUs' wave slots
// from other chains.  Measured, k_line against k_chain (us):
//   rows, D = 64:  320 x 240 53 / 62, 640 x 480 102 / 119, 1000 x 1000 232 / 217
//   rows, D = 128: 320 x 240 63 / 72, 744 x 496 166 / 169, 1000 x 1000 458 / 414
//   columns, D = 64:  320 x 240 43 / 63, 1000 x 1000 238 / 281, 1242 x 375 141 / 129
//   columns, D = 128: 320 x 240 50 / 66, 512 x 256 62 / 74, 640 x 480 206 / 154
// Long chains take more LDS here than in k_chain, so that fewer share a CU and they may
// take more rounds of workgroups, of two thirds of the time each:
//   rows, two rounds / one: 400 of 3000 nodes, D = 128 1140 / 633; 500 of 3300, D = 64 1004 / 570
//   columns, two / one: 1000 of 2000 nodes, D = 64 712 / 558; 400 of 3000, D = 128 1160 / 796
//   columns, three / two: 700 of 4096 nodes, D = 32 1811 / 1993
template <int LPL, int MODE>
static bool use_line(const ChainArgs& a, bool seg) {
  constexpr bool kCols = MODE == kColsMinorant;
  constexpr int kPerCu = kCols && LPL == 1 ? 4 : 2;
  const bool pe = a.w2 != nullptr;
  const int cus = cu_count();
  const long extent = ((long)(a.n - 1) * a.pns * a.D + a.D) * (long)sizeof(float);  // 32-bit byte offsets
  const long msg = (long)a.n * a.D * (long)sizeof(float);
  const size_t lds = line_lds(LPL, pe, a.n);
  if (a.n_chains > kPerCu * cus || lds > kLdsPerCu || extent > 0x7fffffffL || msg > 0x7fffffffL) return false;
  // Rounds of chains, `per` to a workgroup of per * l bytes (0: not launchable).
  auto rounds = [&](size_t l, int per) {
    const long resident = (long)(kLdsPerCu / (per * l)) * per * cus;
    return resident ? (a.n_chains + resident - 1) / resident : 0x7fffffffL;
  };
  const bool many = a.n_chains > cus;
  const size_t chain = !kCols && seg ? row_seg_lds(LPL, pe, a.n) : chain_lds(pe, a.n);
  const bool pairs = !kCols && seg && many && a.n_chains <= 2 * cus && 2 * chain <= kLdsPerCu;
  return 2 * rounds(lds, many && 2 * lds <= kLdsPerCu ? 2 : 1) <= 3 * rounds(chain, pairs ? 2 : 1);
}

// Register-ring depth of the row sweeps with a message wave: three segments.
template <int LPL>
constexpr int row_seg_p() {
  return kRowRing * seg_len<LPL>();
}

template <int LPL, int MODE, int P, int FIT, int DC, bool PE>
static void launch_one(ChainArgs& a, size_t lds, bool seg, hipStream_t st) {
  if constexpr (MODE == kRowsDecode) {
    // w (and w2), u, then the two halves' two-segment message rings at a 16-byte boundary
    const size_t lds2 = sizeof(float) * ((((PE ? 3 : 2) * (size_t)a.n + 3) & ~(size_t)3) +
                                         (size_t)2 * 2 * seg_len<LPL>() * 64 * LPL);
    constexpr int PD = row_seg_p<LPL>();
    auto decode = [&](auto fit, auto gap) {
      constexpr int F = decltype(fit)::value;
      constexpr bool GAP = decltype(gap)::value;
      if (lds2 > 64 * 1024)
        (void)hipFuncSetAttribute((const void*)k_decode4<LPL, PD, F, DC, GAP, PE>,
                                  hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds2);
      k_decode4<LPL, PD, F, DC, GAP, PE><<<a.n_chains, 256, lds2, st>>>(a);
    };
    auto either = [&](auto fit) { a.gap ? decode(fit, std::true_type{}) : decode(fit, std::false_type{}); };
    if constexpr (LPL == 1 && FIT == kFitLanes)
      if (a.D <= 32) return either(std::integral_constant<int, kFitHalf>{});
    either(std::integral_constant<int, FIT>{});
  } else {
    constexpr bool kCols = MODE == kColsMinorant;
    constexpr int PS = kCols ? P : row_seg_p<LPL>();  // ring depth of the checkpointed sweep
    if constexpr (DC == 2 && LPL <= 2) {
      if (use_line<LPL, MODE>(a, seg)) {
        auto line = [&](auto fit) {
          constexpr int F = decltype(fit)::value;
          if constexpr (!kCols)
            if (a.nan_flags) return launch_line<LPL, F, PE, false, true>(a, st);
          launch_line<LPL, F, PE, kCols, false>(a, st);
        };
        if constexpr (LPL == 1 && FIT == kFitLanes)
          if (a.D <= 32) return line(std::integral_constant<int, kFitHalf>{});
        return line(std::integral_constant<int, FIT>{});
      }
    }
    auto sweep = [&](auto nan) {
      constexpr bool NAN_ = decltype(nan)::value;
      if (!seg) return launch_sweep<LPL, MODE, P, FIT, DC, 0, NAN_, PE>(a, lds, st);
      if constexpr (DC == 2)
        if (a.stream) return launch_sweep<LPL, MODE, PS, FIT, DC, 2, NAN_, PE>(a, lds, st);
      launch_sweep<LPL, MODE, PS, FIT, DC, 1, NAN_, PE>(a, lds, st);
    };
    if constexpr (!kCols)
      if (a.nan_flags) return sweep(std::true_type{});
    sweep(std::false_type{});
  }
}

// delta = 2 (the networks' penalty) runs straight-line code when the labels fit
// the lanes; the vector accesses of kFitLanes also need the volumes aligned to
// them (kFitFull has always taken any float pointer).
template <int MODE, int LPL, int P>
static void launch_lpl(ChainArgs& a, size_t lds, bool seg, hipStream_t st) {
  const auto off = reinterpret_cast<uintptr_t>(a.cost) | reinterpret_cast<uintptr_t>(a.A) |
                   reinterpret_cast<uintptr_t>(a.A_in) | reinterpret_cast<uintptr_t>(a.msg);
  const bool full = a.D == 64 * LPL, lanes = a.D % LPL == 0 && off % (LPL * sizeof(float)) == 0;
  if (a.w2) {  // per-edge penalties
    if (full && a.delta == 2) launch_one<LPL, MODE, P, kFitFull, 2, true>(a, lds, seg, st);
    else if (lanes && a.delta == 2) launch_one<LPL, MODE, P, kFitLanes, 2, true>(a, lds, seg, st);
    else launch_one<LPL, MODE, P, kFitAny, 0, true>(a, lds, seg, st);
  } else if (full && a.delta == 2) {
    launch_one<LPL, MODE, P, kFitFull, 2, false>(a, lds, seg, st);
  } else if (lanes && a.delta == 2) {
    launch_one<LPL, MODE, P, kFitLanes, 2, false>(a, lds, seg, st);
  } else if (full) {
    launch_one<LPL, MODE, P, kFitFull, 0, false>(a, lds, seg, st);
  } else {
    launch_one<LPL, MODE, P, kFitAny, 0, false>(a, lds, seg, st);
  }
}

// Prefetch depth (nodes in flight per stream) by labels per lane; the row
// sweeps have only H chains, so they need a deeper ring than the columns to
// keep enough bytes in flight.
#ifndef CCS_CRF_P_ROWS
#define CCS_CRF_P_ROWS 32
#endif
#ifndef CCS_CRF_P_COLS
#define CCS_CRF_P_COLS 16
#endif

// One sweep over all chains for LPL labels per lane.  Defined for LPL = 1, 2
// and 4 (up to 64, 128 and 256 labels), the row sweeps and the others each in a
// translation unit of their own (crf_sweeps_*.hip).
template <int LPL, int MODE>
int launch_labels(ChainArgs& a, bool seg, hipStream_t st) {
  const size_t lds = chain_lds(a.w2 != nullptr, a.n);
  constexpr int P = MODE == kColsMinorant ? CCS_CRF_P_COLS : CCS_CRF_P_ROWS;
  launch_lpl<MODE, LPL, LPL < 4 ? P : P / 2>(a, lds, seg, st);
  CCS_LAUNCH_CHECK();
  return CCS_OK;
}

}  // namespace ccs
