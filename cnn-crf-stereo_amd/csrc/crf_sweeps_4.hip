// The column sweeps and the decode of up to 256 labels (4 per lane).
#include "crf_sweeps.hpp"

namespace ccs {
template int launch_labels<4, kColsMinorant>(ChainArgs& a, bool seg, hipStream_t st);
template int launch_labels<4, kRowsDecode>(ChainArgs& a, bool seg, hipStream_t st);
}  // namespace ccs
