// The forward kernel with two units per wavefront, bf16 tensors.
#include "sa2_mfma_fwd_lone.h"

namespace sa2 {

int launch_mfma_fwd_lone_bf16(const FwdLoneArgs& args, hipStream_t st) { return launch_fwd_lone<ElemBF16>(args, st); }

}  // namespace sa2
