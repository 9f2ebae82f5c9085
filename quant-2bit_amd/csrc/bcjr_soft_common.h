// What the kV = 4 soft kernels (bcjr_soft16.h) and the two-halves kernels of kV <= 2
// (bcjr_halves.h) share.
#pragma once

#include <type_traits>

#include "bcjr_device.h"

namespace bcjr {

struct SoftMeet {
  double logZ2;  // log2 Z
  float EFg;     // E[F] - g_Z (GRAD)
};

// log2 Z = CD + LSE2(m~ + n~) where the sweeps meet (other = null: at the end, n~ = 0)
// and, GRAD, E[F] = sum_j P(j) (mu + nu)(j).  `own` and `other` hold the NT elements
// of the two vectors in one layout; wsum has 2 * kMaxWaves floats.  E[F] is taken off
// every path value of the marginal sweep, so its error enters all gradients of the
// sequence alike; it is summed in double, once per sequence, and rounded once (with
// float sums the gradients were 2-20 % further from 64 bits: 500 sequences of a table
// at L = 16 5.87e-6 against 5.71e-6, 8 tiles of the column walk 7.2e-6 against 6.5e-6,
// more the shorter the sequences).
template <bool GRAD>
__device__ __forceinline__ SoftMeet soft_meet(const float* own, const float* other, int NT, double CD, float gZ,
                                              float* wsum) {
  constexpr int ST = GRAD ? 2 : 1;
  const int tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63, wave = tid >> 6, nwaves = nthr >> 6;
  float mx = -INFINITY;
  for (int j = tid; j < NT; j += nthr) mx = fmaxf(mx, own[ST * j] + (other ? other[ST * j] : 0.0f));
  mx = wave_max(mx);
  if (lane == 0) wsum[wave] = mx;
  __syncthreads();
  float Mz = -INFINITY;
  for (int w = 0; w < nwaves; ++w) Mz = fmaxf(Mz, wsum[w]);
  using Sum = std::conditional_t<GRAD, double, float>;
  Sum ps = 0, pe = 0;
  for (int j = tid; j < NT; j += nthr) {
    const Sum e = fexp2(own[ST * j] + (other ? other[ST * j] : 0.0f) - Mz);
    ps += e;
    if constexpr (GRAD) pe = fma(e, (double)own[2 * j + 1] + (other ? (double)other[2 * j + 1] : 0.0), pe);
  }
  if constexpr (GRAD) {
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) {
      ps += __shfl_xor(ps, o, 64);
      pe += __shfl_xor(pe, o, 64);
    }
  } else {
    ps = wave_sum(ps);
  }
  __syncthreads();
  if (lane == 0) {
    wsum[wave] = (float)ps;
    if constexpr (GRAD) wsum[kMaxWaves + wave] = (float)pe;
  }
  __syncthreads();
  Sum Ssum = 0, Esum = 0;
  for (int w = 0; w < nwaves; ++w) {
    Ssum += wsum[w];
    if constexpr (GRAD) Esum += wsum[kMaxWaves + w];
  }
  __syncthreads();
  return {CD + (double)Mz + (double)flog2((float)Ssum), GRAD ? (float)(Esum / Ssum - gZ) : 0.0f};
}

}  // namespace bcjr
