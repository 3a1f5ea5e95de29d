// The plane-split forward kernel with two units per wavefront for fp32 tensors of head_dim 16, 32 and 64.
#include "sa2_split_fwd_lone.h"

namespace sa2 {

int launch_split_fwd_lone_fp32(const Problem& p, int width, bool, hipStream_t st) {
    typedef MemF32 T;
    if (width == 64) return launch_split_fwd_lone<T, 64, 3, EXACT>(p, st);
    return p.D == 32 ? launch_split_fwd_lone<T, 32, 3, EXACT>(p, st) : launch_split_fwd_lone<T, 32, 3, PADDED>(p, st);
}

}  // namespace sa2
