// The row sweeps of up to 64 labels (1 per lane).
#include "crf_sweeps.hpp"

namespace ccs {
template int launch_labels<1, kRowsMinorant>(ChainArgs& a, bool seg, hipStream_t st);
}  // namespace ccs
