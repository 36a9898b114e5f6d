// lr_fwd_t32 (lowrank_mfma_t32.h) in fp16.
#include "lowrank_mfma_fwd_t32.h"

namespace dc {
template hipError_t lr_fwd_t32_launch<fp16>(const LrArgs&, int, int, hipStream_t);
}  // namespace dc
