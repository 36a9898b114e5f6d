// lr_bwd_t32 (lowrank_mfma_bwd32.h) in fp16.
#include "lowrank_mfma_bwd32.h"

namespace dc {
template hipError_t lr_bwd_t32_launch<fp16>(const LrBwdArgs&, int, int, bool, hipStream_t);
}  // namespace dc
