// The K'-side backward kernel for wide K windows, bf16 tensors.
#include "sa2_mfma_bwd_kp_lone.h"

namespace sa2 {

int launch_mfma_bwd_kp_lone_bf16(const Problem& p, const KpLaunch& l, hipStream_t st) { return launch_kp_lone<ElemBF16>(p, l, st); }

}  // namespace sa2
