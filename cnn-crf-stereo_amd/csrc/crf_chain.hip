// Chooses and launches the chain sweeps (crf_sweeps.hpp) of one half-step.
#include <cstdlib>

#include "crf_chain.hpp"

namespace ccs {

// Compute units of the current device (cached per device).
int cu_count() {
  static int cus[64] = {0};
  int dev = 0;
  (void)hipGetDevice(&dev);
  if (dev < 0 || dev >= 64) return 256;
  if (!cus[dev]) {
    int v = 0;
    if (hipDeviceGetAttribute(&v, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || v <= 0) v = 256;
    cus[dev] = v;
  }
  return cus[dev];
}

// Volumes from which the column sweeps recompute messages from checkpoints.
// Below it the sweep is latency-bound and the recomputation only adds steps;
// above it the sweep is HBM-bound and the recomputation removes two of the
// seven volume passes (measured: 0.304 -> 0.228 ms at 1242x375x128, 1.93 ->
// 1.55 ms at 1488x992x256; 0.056 -> 0.060 ms at 300x200x64).
constexpr long kSegMinBytes = 64l << 20;

// The threshold, overridable by the environment variable CCS_CRF_SEG_MIN_BYTES
// (read once per process; tests use it to run the checkpointed scheme on small
// volumes and compare it bit for bit with the store-everything one).
static long seg_min_bytes() {
  static const long v = [] {
    const char* e = getenv("CCS_CRF_SEG_MIN_BYTES");
    return e ? atol(e) : kSegMinBytes;
  }();
  return v;
}

template <int LPL>
static int launch_mode(ChainMode mode, ChainArgs& a, bool seg, hipStream_t st) {
  switch (mode) {
    case kRowsMinorant: return launch_labels<LPL, kRowsMinorant>(a, seg, st);
    case kColsMinorant: return launch_labels<LPL, kColsMinorant>(a, seg, st);
    case kRowsDecode: return launch_labels<LPL, kRowsDecode>(a, seg, st);
  }
  return fail(CCS_ERR_ARG, "unknown chain mode %d", (int)mode);
}

// The sweeps stream the costs where the cost and the state volume together are
// larger than the last-level cache: a sweep reads the costs once and the unaries
// twice, so keeping costs there only displaces unaries (measured, a row and a
// column sweep: 450 -> 432 us at 1242x375x128, 2763 -> 2710 us at 1488x992x256;
// where both fit, streaming costs 2-3 %: 185 -> 190 us at 320x240x256).
constexpr long kStreamMinBytes = 128l << 20;

int launch_chain(ChainMode mode, ChainArgs& a, hipStream_t st) {
  if (mode != kColsMinorant) {  // row chains are addressed with 32-bit byte offsets
    const long extent = ((long)(a.n - 1) * a.pns * a.D + a.D) * (long)sizeof(float);
    const long msg = (long)a.n * a.D * (long)sizeof(float);
    if (extent > 0x7fffffffL || msg > 0x7fffffffL)
      return fail(CCS_ERR_ARG, "row chain of %d nodes x %d labels exceeds 2 GiB", a.n, a.D);
  }
  bool seg = false;
  const long vol = (long)a.n_chains * a.n * a.D * (long)sizeof(float);
  a.stream = vol > kStreamMinBytes;
  if (mode == kColsMinorant && kSeg > 0) {
    // A segment's nodes are addressed with 32-bit byte offsets from its first node.
    const long span = ((long)(kSeg - 1) * a.pns * a.D + a.D) * (long)sizeof(float);
    seg = span <= 0x7fffffffL && vol >= seg_min_bytes();
  }
  // Row sweeps take the message wave at the same volumes (their chains are
  // addressed within the 2 GiB checked above).
  // The message wave also needs one chain's LDS to fit a CU.
  const bool pe = a.w2 != nullptr;
  const int lpl = a.D <= 64 ? 1 : a.D <= 128 ? 2 : 4;
  const size_t row_lds = row_seg_lds(lpl, pe, a.n);
  const bool row_seg = kSeg > 0 && vol >= seg_min_bytes() && row_lds <= kLdsPerCu;
  seg = mode == kColsMinorant ? seg : mode == kRowsMinorant && row_seg;
  if (a.D <= 64) return launch_mode<1>(mode, a, seg, st);
  if (a.D <= 128) return launch_mode<2>(mode, a, seg, st);
  return launch_mode<4>(mode, a, seg, st);
}

}  // namespace ccs
