// The launch of lr_fwd_t32 (lowrank_mfma_t32.h), instantiated in
// lowrank_mfma_fwd_t32_{bf16,fp16}.hip.
#pragma once

#include "lowrank_mfma_t32.h"

namespace dc {

template <typename T, int W, int NC>
hipError_t lr_fwd_t32_one(const LrArgs& a, hipStream_t s) {
  constexpr int NT = 64 * t32_wg_waves(W, NC);
  if (a.zvec) {
    if (a.zrp > 0)
      lr_fwd_t32<T, W, NC, true, true><<<a.nblk, NT, 0, s>>>(a);
    else
      lr_fwd_t32<T, W, NC, true, false><<<a.nblk, NT, 0, s>>>(a);
  } else {
    if (a.zrp > 0)
      lr_fwd_t32<T, W, NC, false, true><<<a.nblk, NT, 0, s>>>(a);
    else
      lr_fwd_t32<T, W, NC, false, false><<<a.nblk, NT, 0, s>>>(a);
  }
  return hipGetLastError();
}

template <typename T>
hipError_t lr_fwd_t32_launch(const LrArgs& a, int W, int NC, hipStream_t s) {
#define DC_T32_CASE(WW, CC) \
  if (W == WW && NC == CC) return lr_fwd_t32_one<T, WW, CC>(a, s);
  DC_T32_CASE(1, 1) DC_T32_CASE(2, 1) DC_T32_CASE(3, 1) DC_T32_CASE(4, 1)
  DC_T32_CASE(5, 1) DC_T32_CASE(6, 1) DC_T32_CASE(7, 1) DC_T32_CASE(8, 1)
  DC_T32_CASE(1, 2) DC_T32_CASE(2, 2) DC_T32_CASE(3, 2) DC_T32_CASE(4, 2)
  DC_T32_CASE(5, 2) DC_T32_CASE(6, 2) DC_T32_CASE(7, 2) DC_T32_CASE(8, 2)
#undef DC_T32_CASE
  return hipErrorInvalidValue;
}

}  // namespace dc
