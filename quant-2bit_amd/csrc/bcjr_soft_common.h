// What the kV = 4 soft kernels (bcjr_soft16.h) and the two-halves kernels of kV <= 2
// (bcjr_halves.h) share.
#pragma once

#include <type_traits>

#include "bcjr_device.h"

namespace bcjr {

// Reads a sequence's inputs into LDS and checks them: T must be finite and > 0, the
// weights and upstream gradients finite.  bflag is the workgroup's flag word; when it
// is set the sequence's outputs are NaN (soft_fill_nan).  Uniform result.
template <bool GRAD>
__device__ __forceinline__ bool soft_inputs(const float* seq, const float* g_soft, int n, float T, float gZ, float* wbuf,
                                            float* gbuf, int* bflag) {
  const int tid = threadIdx.x, nthr = blockDim.x;
  if (tid == 0) *bflag = 0;
  __syncthreads();
  int bad = !(T > 0.0f && T < INFINITY) || !__builtin_isfinite(gZ);
  for (int i = tid; i < n; i += nthr) {
    const float w = seq[i];
    wbuf[i] = w;
    bad |= !__builtin_isfinite(w);
    if constexpr (GRAD) {
      const float gg = g_soft[i];
      gbuf[i] = gg;
      bad |= !__builtin_isfinite(gg);
    }
  }
  if (bad) *bflag = 1;
  __syncthreads();
  return *bflag == 0;  // every thread reads the flag after the barrier
}

// The outputs of sequence b whose inputs are not finite.
template <bool GRAD, bool ENT>
__device__ __forceinline__ void soft_fill_nan(const Soft16Params& P, long long b, float* out, int n) {
  const int tid = threadIdx.x, nthr = blockDim.x;
  for (int i = tid; i < n; i += nthr) out[i] = NAN;
  if (tid == 0 && !GRAD && P.logZ) P.logZ[b] = NAN;
  if constexpr (ENT)
    for (int i = tid; i < P.N; i += nthr) P.H_out[(size_t)b * P.N + i] = NAN;
}

// Outputs of one step from its per-wave partials sp (wave 0): GRAD d seq of the step
// (w its weights), else the soft codeword and, ENT, the entropy into *H.
template <bool GRAD, bool ENT, int V>
__device__ __forceinline__ void soft_step_out(const float* sp, int nwaves, const float* w, float twoT, float* out,
                                              float* H) {
  constexpr int NS = V + (GRAD || ENT ? 1 : 0);
  const int lane = threadIdx.x & 63;
  if constexpr (GRAD) {
    const float a0 = sum_of_waves(sp, nwaves, NS);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const float a1 = sum_of_waves(sp + 1 + v, nwaves, NS);
      if (lane == 0) out[v] = twoT * (a1 - w[v] * a0);
    }
  } else {
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const float a = sum_of_waves(sp + v, nwaves, NS);
      if (lane == 0) out[v] = a;
    }
    if constexpr (ENT) {
      const float h = sum_of_waves(sp + V, nwaves, NS);
      if (lane == 0) *H = -h * (float)kLn2;
    }
  }
}

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
