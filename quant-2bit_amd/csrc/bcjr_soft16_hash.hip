// Instances of the kV = 4 soft kernels (bcjr_soft16.h): 1MAD and 3INST.
#include "bcjr_soft16.h"

namespace bcjr {

const void* soft16_hash_kernel_ptr(int kind, int code, int lpb) {
  if (code == CODE_1MAD && lpb == 4) {
    BCJR_SOFT16_KINDS(CODE_1MAD, 1, 4)
  } else if (code == CODE_1MAD) {
    BCJR_SOFT16_KINDS(CODE_1MAD, 1, 16)
  } else if (lpb == 4) {
    BCJR_SOFT16_KINDS(CODE_3INST, 1, 4)
  }
  BCJR_SOFT16_KINDS(CODE_3INST, 1, 16)
}

}  // namespace bcjr
