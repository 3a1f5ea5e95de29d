// The K-side backward kernel with one wavefront per SIMD for fp16 tensors of the head dims in between.
#include "sa2_split_kv_lone.h"

namespace sa2 {

int launch_split_kv_lone_fp16(const Problem& p, int width, bool, int nsplit, float* part, hipStream_t st) {
    typedef Mem16<ElemF16> T;
    return width == 64 ? launch_split_kv_lone<T, 64, 3, PADDED>(p, nsplit, part, st) : launch_split_kv_lone<T, 96, 3, PADDED>(p, nsplit, part, st);
}

}  // namespace sa2
