// The chain sweeps of up to 128 labels (2 per lane).
#include "crf_sweeps.hpp"

namespace ccs {
template int launch_labels<2>(ChainMode mode, ChainArgs& a, bool seg, hipStream_t st);
}  // namespace ccs
