// The K'-side backward kernel with one wavefront per SIMD for fp16 tensors of the head dims in between.
#include "sa2_split_kp_lone.h"

namespace sa2 {

int launch_split_kp_lone_fp16(const Problem& p, int width, bool, const SplitKpLaunch& l, hipStream_t st) {
    typedef Mem16<ElemF16> T;
    return width == 64 ? launch_split_kp_lone<T, 64, 3, PADDED>(p, l, st) : launch_split_kp_lone<T, 96, 3, PADDED>(p, l, st);
}

}  // namespace sa2
