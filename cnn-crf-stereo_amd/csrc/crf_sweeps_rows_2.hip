// The row sweeps of up to 128 labels (2 per lane).
#include "crf_sweeps.hpp"

namespace ccs {
template int launch_labels<2, kRowsMinorant>(ChainArgs& a, bool seg, hipStream_t st);
}  // namespace ccs
