// Instances of the kV = 4 soft kernels (bcjr_soft16.h): codebook tables, and their transposed copy.
#include "bcjr_soft16.h"

namespace bcjr {

namespace {

// out[(p * 16 + c) * NB + u] = table[p * NT + 16 u + c] (V floats each): states of
// one (p, c) on consecutive addresses.  512 KiB at L = 16, V = 2: a few
// microseconds, written once per call.
template <int V>
__global__ __launch_bounds__(256) void transpose16_kernel(const float* __restrict__ table, float* __restrict__ out,
                                                          int L) {
  const uint32_t NB = 1u << (L - 8), NT = NB << 4, i = blockIdx.x * 256u + threadIdx.x;
  if (i >= (1u << L)) return;
  const uint32_t u = i & (NB - 1), c = (i >> (L - 8)) & 15u, p = i >> (L - 4);
  const uint32_t s = p * NT + 16u * u + c;
#pragma unroll
  for (int v = 0; v < V; ++v) out[(size_t)V * i + v] = table[(size_t)V * s + v];
}

}  // namespace

hipError_t launch_transpose16(const float* table, float* out, int L, int V, hipStream_t stream) {
  const unsigned grid = ((1u << L) + 255u) / 256u;
  if (V == 2) hipLaunchKernelGGL(transpose16_kernel<2>, dim3(grid), dim3(256), 0, stream, table, out, L);
  else hipLaunchKernelGGL(transpose16_kernel<1>, dim3(grid), dim3(256), 0, stream, table, out, L);
  return hipGetLastError();
}

const void* soft16_table_kernel_ptr(int kind, int V, int lpb) {
  if (V == 1 && lpb == 4) {
    BCJR_SOFT16_KINDS(CODE_TABLE, 1, 4)
  } else if (V == 1) {
    BCJR_SOFT16_KINDS(CODE_TABLE, 1, 16)
  } else if (lpb == 4) {
    BCJR_SOFT16_KINDS(CODE_TABLE, 2, 4)
  }
  BCJR_SOFT16_KINDS(CODE_TABLE, 2, 16)
}

}  // namespace bcjr
