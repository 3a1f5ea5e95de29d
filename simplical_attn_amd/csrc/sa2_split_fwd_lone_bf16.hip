// The plane-split forward kernel with two units per wavefront for bf16 tensors of the head dims in between.
#include "sa2_split_fwd_lone.h"

namespace sa2 {

int launch_split_fwd_lone_bf16(const Problem& p, int width, bool two_planes, hipStream_t st) {
    typedef Mem16<ElemBF16> T;
    auto of_width = [&](auto w) {
        constexpr int D = decltype(w)::value;
        return two_planes ? launch_split_fwd_lone<T, D, 2, PADDED>(p, st) : launch_split_fwd_lone<T, D, 3, PADDED>(p, st);
    };
    return width == 64 ? of_width(LONE_C(64)) : of_width(LONE_C(96));
}

}  // namespace sa2
