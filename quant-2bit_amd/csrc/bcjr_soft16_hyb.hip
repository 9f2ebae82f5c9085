// Instances of the kV = 4 soft kernels (bcjr_soft16.h): HYB outside the column walk.
#include "bcjr_soft16.h"

namespace bcjr {

const void* soft16_hyb_kernel_ptr(int kind, int lpb) {
  if (lpb == 4) {
    BCJR_SOFT16_KINDS(CODE_HYB, 2, 4)
  }
  BCJR_SOFT16_KINDS(CODE_HYB, 2, 16)
}

}  // namespace bcjr
