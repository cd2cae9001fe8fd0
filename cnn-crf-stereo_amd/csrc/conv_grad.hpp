// Weight gradient on the 16-bit matrix cores (conv_grad.hip).
#pragma once

#include "common.hpp"

namespace ccs {

struct DwArgs {
  const void* x;   // Hin x Win x Csx, the maps' type
  const void* dz;  // Ho rows of zpitch pixels x Csk
  float* part;     // nch x KH KW x 112 x 112
  int Win, Csx, zpitch, Ho, Wo, Csk;
  int nch, segs_per_row;
  long nseg, spc;  // segments in all and per chunk
};

// Layers whose input and dz have 72 to 112 channels (with padding).
bool dw_split_supported(int Csx, int Csk, int KW);
int dw_split_segment(int precision);  // output pixels per segment
void dw_split(const DwArgs& a, int precision, int KH, int KW, hipStream_t st);

}  // namespace ccs
