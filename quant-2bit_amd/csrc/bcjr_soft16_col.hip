// Instances of the kV = 4 soft kernels (bcjr_soft16.h): the HYB column walk, and the dispatch over codes.
#include "bcjr_soft16.h"

namespace bcjr {

const void* soft16_col_kernel_ptr(int kind, int lpb) {
  if (lpb == 2) {
    BCJR_SOFT16_KINDS(CODE_HYB_COL, 2, 2)
  }
  BCJR_SOFT16_KINDS(CODE_HYB_COL, 2, 4)
}

const void* soft16_kernel_ptr(int kind, int V, int code, int lpb) {
  if (code == CODE_HYB_COL) return soft16_col_kernel_ptr(kind, lpb);
  if (code == CODE_HYB) return soft16_hyb_kernel_ptr(kind, lpb);
  if (code == CODE_TABLE) return soft16_table_kernel_ptr(kind, V, lpb);
  return soft16_hash_kernel_ptr(kind, code, lpb);
}

}  // namespace bcjr
