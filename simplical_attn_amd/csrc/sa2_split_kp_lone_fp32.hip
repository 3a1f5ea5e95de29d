// The K'-side backward kernel with one wavefront per SIMD for fp32 tensors of head_dim 16, 32 and 64.
#include "sa2_split_kp_lone.h"

namespace sa2 {

int launch_split_kp_lone_fp32(const Problem& p, int width, bool, const SplitKpLaunch& l, hipStream_t st) {
    if (width == 64) return launch_split_kp_lone<MemF32, 64, 3, EXACT>(p, l, st);
    return p.D == 32 ? launch_split_kp_lone<MemF32, 32, 3, EXACT>(p, l, st) : launch_split_kp_lone<MemF32, 32, 3, PADDED>(p, l, st);
}

}  // namespace sa2
