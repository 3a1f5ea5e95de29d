// The plane-split forward kernel with two units per wavefront for fp16 tensors of the head dims in between.
#include "sa2_split_fwd_lone.h"

namespace sa2 {

int launch_split_fwd_lone_fp16(const Problem& p, int width, bool, hipStream_t st) {
    typedef Mem16<ElemF16> T;
    return width == 64 ? launch_split_fwd_lone<T, 64, 3, PADDED>(p, st) : launch_split_fwd_lone<T, 96, 3, PADDED>(p, st);
}

}  // namespace sa2
