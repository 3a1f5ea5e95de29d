// The K-side backward kernel with one wavefront per SIMD for fp32 tensors of head_dim 16, 32 and 64.
#include "sa2_split_kv_lone.h"

namespace sa2 {

int launch_split_kv_lone_fp32(const Problem& p, int width, bool, int nsplit, float* part, hipStream_t st) {
    if (width == 64) return launch_split_kv_lone<MemF32, 64, 3, EXACT>(p, nsplit, part, st);
    return p.D == 32 ? launch_split_kv_lone<MemF32, 32, 3, EXACT>(p, nsplit, part, st) : launch_split_kv_lone<MemF32, 32, 3, PADDED>(p, nsplit, part, st);
}

}  // namespace sa2
