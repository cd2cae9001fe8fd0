// The row sweeps of up to 256 labels (4 per lane).
#include "crf_sweeps.hpp"

namespace ccs {
template int launch_labels<4, kRowsMinorant>(ChainArgs& a, bool seg, hipStream_t st);
}  // namespace ccs
