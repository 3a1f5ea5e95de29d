// The forward kernel with two units per wavefront, fp16 tensors.
#include "sa2_mfma_fwd_lone.h"

namespace sa2 {

int launch_mfma_fwd_lone_fp16(const FwdLoneArgs& args, hipStream_t st) { return launch_fwd_lone<ElemF16>(args, st); }

}  // namespace sa2
