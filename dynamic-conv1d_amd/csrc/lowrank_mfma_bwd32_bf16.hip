// lr_bwd_t32 (lowrank_mfma_bwd32.h) in bf16.
#include "lowrank_mfma_bwd32.h"

namespace dc {
template hipError_t lr_bwd_t32_launch<bf16>(const LrBwdArgs&, int, int, bool, hipStream_t);
}  // namespace dc
