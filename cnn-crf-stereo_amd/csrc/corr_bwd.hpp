// Correlation adjoint on the bf16 matrix cores (corr_bwd.hip).
#pragma once

#include "common.hpp"

namespace ccs {

struct CorrBwdArgs {
  const void* f0;
  const void* f1;
  const float* G;
  void* df0;
  void* df1;
  int H, W, Cs, D;
  int o0, ostep;  // o_k = o0 + k * ostep, ostep = 1 or -1
  int tiles;      // pixel tiles per row (set by the launch)
};

bool corr_bwd_split_supported(int Cs, int W, int D, int ostep);
void corr_bwd_split(const CorrBwdArgs& a, int precision, hipStream_t st);

}  // namespace ccs
