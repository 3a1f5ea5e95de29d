// The K-side backward kernel for fp16 tensors.
#include "sa2_mfma_bwd_kv.h"

namespace sa2 {

int launch_mfma_bwd_kv_fp16(const Problem& p, int kb, int nsplit, hipStream_t st, BwdSums* sums) { return launch_kv<ElemF16>(p, kb, nsplit, st, sums); }

}  // namespace sa2
