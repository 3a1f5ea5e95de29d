// The plane-split forward kernel with two units per wavefront for fp32 tensors of head_dim 64.
#include "sa2_split_fwd_lone.h"

namespace sa2 {

int launch_split_fwd_lone_fp32(const Problem& p, int, bool, hipStream_t st) { return launch_split_fwd_lone<MemF32, 64, 3, EXACT>(p, st); }

}  // namespace sa2
