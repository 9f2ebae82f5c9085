// Instances of the two-halves soft kernels (bcjr_halves.h): forward.
#include "bcjr_halves.h"

namespace bcjr {

#define BCJR_HALVES_CASE(KV_, V_, CODE_, UPT_, LPB_)                                            \
  if (KV == KV_ && V == V_ && code == CODE_ && upt == UPT_ && lpb == LPB_)                      \
    return reinterpret_cast<const void*>(&bcjr_halves_kernel<KV_, V_, CODE_, UPT_, LPB_, false, false>);
#define BCJR_HALVES_ALL(V_, CODE_)         \
  BCJR_HALVES_CASE(2, V_, CODE_, 1, 1)     \
  BCJR_HALVES_CASE(2, V_, CODE_, 2, 1)     \
  BCJR_HALVES_CASE(2, V_, CODE_, 4, 1)     \
  BCJR_HALVES_CASE(2, V_, CODE_, 1, 4)

const void* halves_kernel_ptr(int kind, int KV, int V, int code, int upt, int lpb) {
  if (kind == 1) return halves_bwd_kernel_ptr(KV, V, code, upt, lpb);
  if (kind == 2) return halves_entropy_kernel_ptr(KV, V, code, upt, lpb);
  BCJR_HALVES_CASE(1, 1, CODE_TABLE, 1, 2)
  BCJR_HALVES_ALL(1, CODE_TABLE)
  BCJR_HALVES_ALL(1, CODE_1MAD)
  BCJR_HALVES_ALL(1, CODE_3INST)
  BCJR_HALVES_ALL(2, CODE_TABLE)
  BCJR_HALVES_ALL(2, CODE_HYB)
  return nullptr;
}

}  // namespace bcjr
