// Instances of the kV = 4 soft kernels (bcjr_soft16.h): HYB outside the column walk.
#include "bcjr_soft16.h"

namespace bcjr {

#define BCJR_SOFT16_KINDS(CODE_, V_, LPB_)                                                                    \
  if (kind == 0) return reinterpret_cast<const void*>(&bcjr_soft16_kernel<false, CODE_, V_, LPB_, false>);    \
  if (kind == 1) return reinterpret_cast<const void*>(&bcjr_soft16_kernel<true, CODE_, V_, LPB_, false>);     \
  return reinterpret_cast<const void*>(&bcjr_soft16_kernel<false, CODE_, V_, LPB_, true>);

const void* soft16_hyb_kernel_ptr(int kind, int lpb) {
  if (lpb == 4) {
    BCJR_SOFT16_KINDS(CODE_HYB, 2, 4)
  }
  BCJR_SOFT16_KINDS(CODE_HYB, 2, 16)
}

}  // namespace bcjr
