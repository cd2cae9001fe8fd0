// The column sweeps and the decode of up to 128 labels (2 per lane).
#include "crf_sweeps.hpp"

namespace ccs {
template int launch_labels<2, kColsMinorant>(ChainArgs& a, bool seg, hipStream_t st);
template int launch_labels<2, kRowsDecode>(ChainArgs& a, bool seg, hipStream_t st);
}  // namespace ccs
