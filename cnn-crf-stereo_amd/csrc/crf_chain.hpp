// Interface between the SlackProp host code and the chain-sweep kernels.
#pragma once

#include "common.hpp"

namespace ccs {

constexpr float kGamma = 0.25f;
constexpr double kGammaD = 0.25;

enum ChainMode { kRowsMinorant = 0, kColsMinorant = 1, kRowsDecode = 2 };

struct ChainArgs {
  const float* cost;   // C (row and column sweeps)
  float* A;            // state: row unaries before a row sweep, column unaries C - A before a column sweep
  const float* A_in;   // where a row sweep reads the unaries (A, or cost for the first sweep)
  const float* w;      // edge weight of the edge (node i, node i+1), indexed by pixel (P1 with w2)
  const float* w2;     // per-edge penalties: P2 of the edge (then w holds P1); nullptr: w L1, w L2
  int wmul = 1;        // elements per pixel in the arrays of w / w2 (2: interleaved x, y)
  float* msg;          // backward messages, [chain][node][D]
  int* labels;         // decode output, indexed by pixel
  float* gap;          // decode: second best - best min-marginal (optional)
  double* lam;         // per chain: minimum chain energy
  double* kept;        // per chain: sum of kept constants
  int* nan_flags;      // row minorant (optional): per chain, 1 if a unary read was NaN, else 0
  long pcs, pns;       // pixel index = chain * pcs + node * pns
  int n_chains, n, D, delta;
  float L1, L2;
  bool stream = false;  // the costs are read without being kept in the caches (set by launch_chain)
};

// Column sweeps of large volumes keep the backward messages of every
// seg_len()-th node only; the forward pass recomputes a segment's messages from
// the checkpoint at its end, bit for bit (0: every message is stored and
// re-read).
#ifndef CCS_CRF_SEG
#define CCS_CRF_SEG 12
#endif
constexpr int kSeg = CCS_CRF_SEG;
// Segment length by labels per lane: a segment keeps two segments' unaries and
// costs and one segment's messages in registers, so four labels per lane take
// half the length (two waves per SIMD without spills).
constexpr int seg_length(int lpl) { return kSeg <= 0 ? 0 : lpl >= 4 ? (kSeg / 2 > 0 ? kSeg / 2 : 1) : kSeg; }

// Row sweeps with a message wave keep a ring of kRowRing segments' messages in LDS.
constexpr int kRowRing = 3;

constexpr size_t kLdsPerCu = 160 * 1024;

// LDS of one chain of k_chain: b (doubles), w, u, [w2].
constexpr size_t chain_lds(bool per_edge, int n) {
  return (sizeof(double) + (per_edge ? 3 : 2) * sizeof(float)) * (size_t)n;
}

// LDS of one row chain with the message wave: b, w, u, [w2], v floats rounded
// to 16 bytes, then the message ring.
constexpr size_t row_seg_lds(int lpl, bool per_edge, int n) {
  return sizeof(float) * ((((per_edge ? 6 : 5) * (size_t)n + 3) & ~(size_t)3) +
                          (size_t)kRowRing * seg_length(lpl) * 64 * lpl);
}

// One sweep of MODE for LPL (1, 2 or 4) labels per lane; seg: the checkpointed schemes.
template <int LPL, int MODE>
int launch_labels(ChainArgs& a, bool seg, hipStream_t st);

// Launches one sweep of `mode` over all chains of `a` on `st`.
int launch_chain(ChainMode mode, ChainArgs& a, hipStream_t st);

}  // namespace ccs
