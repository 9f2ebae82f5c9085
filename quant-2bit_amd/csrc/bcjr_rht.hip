// Fast Walsh-Hadamard transforms for the random Hadamard transform (RHT) that
// wraps the BCJR quantizer:
//   RHT(W)     = s * H_m diag(sl) W diag(sr) H_n            (src/rht/transform.py:65-96)
//   RHT^-1(W~) = s * diag(sl) H_m W~ H_n diag(sr)           (src/rht/transform.py:99-126)
// with s = 1/sqrt(m*n) and H unscaled Sylvester-ordered Hadamard matrices.  The
// butterflies run in the reference's order (fwht_numpy, transform.py:26-42: h = 1,
// 2, 4, ..., x[i] = a + b, x[i+h] = a - b), so for each element the sequence of
// float32 additions is the reference's and the results agree bit for bit (the
// final scale is a multiply by s, exact whenever m*n is an even power of two).
//
// A batch of matrices (E, m, n) with per-matrix sign vectors (E, m), (E, n) runs
// in the same launches (expert-batched dispatch).
//
// Rows (last axis, contiguous): one workgroup per row, staged in LDS (n <= 16384).
// Columns (first axis, stride n): m = a*b with b = min(m, 128); a first pass does
// the stages h < b on tiles of b consecutive rows x 64 consecutive columns, a
// second the stages h >= b on tiles of a rows spaced b apart; every global access
// reads or writes 256 contiguous bytes of a row (4n bytes when n < 64).  No
// transposes.
#include <hip/hip_runtime.h>

#include <stdint.h>

#include <algorithm>
#include <atomic>
#include <type_traits>

#include "bcjr_kernels.h"

namespace bcjr {

namespace {

constexpr int kRowThreads = 256;
constexpr int kColTile = 64;  // columns per column-pass tile (fewer when n < 64)
constexpr int kColThreads = 256;

// One butterfly stage of span h on n values in LDS: pairs (i, i + h) with
// i = 2h * (j / h) + j % h for j < n/2.
__device__ __forceinline__ void stage(float* v, int n, int h, int tid, int nthr) {
  for (int j = tid; j < (n >> 1); j += nthr) {
    const int i = ((j & ~(h - 1)) << 1) | (j & (h - 1));
    const float a = v[i], b = v[i + h];
    v[i] = a + b;
    v[i + h] = a - b;
  }
}

struct RowsParams {
  const float* x;
  float* out;
  long long rows;
  int n;
  const float* pre;       // (rows / vec_rows, n) multiplies x before the transform, or null
  const float* post;      // (rows / vec_rows, n) multiplies the result, or null
  long long vec_rows;     // consecutive rows sharing one pre/post vector (m of a batch)
  const float* row_sign;  // (rows) multiplies row r of the result, or null
  float scale;
};

__global__ __launch_bounds__(kRowThreads) void fwht_rows_kernel(RowsParams P) {
  extern __shared__ __align__(16) float v[];
  const int n = P.n, tid = threadIdx.x, nthr = blockDim.x;
  for (long long r = blockIdx.x; r < P.rows; r += gridDim.x) {
    const float* xr = P.x + (size_t)r * n;
    const size_t vo = (size_t)(r / P.vec_rows) * n;
    for (int i = tid; i < n; i += nthr) v[i] = P.pre ? xr[i] * P.pre[vo + i] : xr[i];
    __syncthreads();
    for (int h = 1; h < n; h <<= 1) {
      stage(v, n, h, tid, nthr);
      __syncthreads();
    }
    const float rs = P.row_sign ? P.row_sign[r] : 1.0f;
    float* orow = P.out + (size_t)r * n;
    for (int i = tid; i < n; i += nthr) {
      float y = v[i];
      if (P.post) y *= P.post[vo + i];
      orow[i] = (y * rs) * P.scale;
    }
    __syncthreads();
  }
}

struct ColsParams {
  float* x;               // (batch, m, n) transformed in place
  long long mat_stride;   // m * n
  int m;                  // rows per matrix (row_sign offset of matrix e is e * m)
  int n;
  int C;                  // tile width: min(kColTile, n), a power of two dividing n
  int len;                // transform length along the column (tile rows)
  long long step;         // floats between consecutive tile rows
  long long outer_stride; // floats between tiles of consecutive outer index
  int outer;              // outer index count
  int batch;              // matrices
  const float* row_sign;  // (batch, m) multiplies row o*row_o + p*row_p of the result, or null
  int row_o, row_p;
  float scale;
};

__global__ __launch_bounds__(kColThreads) void fwht_cols_kernel(ColsParams P) {
  extern __shared__ __align__(16) float t[];  // len x C
  const int tid = threadIdx.x, nthr = blockDim.x;
  const int C = P.C;
  const int ncb = P.n / C;
  const long long per_mat = (long long)P.outer * ncb;
  const long long tiles = per_mat * P.batch;
  for (long long g = blockIdx.x; g < tiles; g += gridDim.x) {
    const long long e = g / per_mat, gm = g - e * per_mat;
    const int o = (int)(gm / ncb), cb = (int)(gm % ncb);
    float* base = P.x + (size_t)e * P.mat_stride + (size_t)o * P.outer_stride + (size_t)cb * C;
    const float* rsgn = P.row_sign ? P.row_sign + (size_t)e * P.m : nullptr;
    for (int e = tid; e < P.len * C; e += nthr) {
      const int p = e / C, c = e % C;
      t[e] = base[(size_t)p * P.step + c];
    }
    __syncthreads();
    // Stage h along the tile rows for every column: butterfly (p, p + h) of
    // column c is item j = q * C + c, q < len/2.
    for (int h = 1; h < P.len; h <<= 1) {
      for (int j = tid; j < (P.len >> 1) * C; j += nthr) {
        const int q = j / C, c = j % C;
        const int p = ((q & ~(h - 1)) << 1) | (q & (h - 1));
        const float a = t[p * C + c], b = t[(p + h) * C + c];
        t[p * C + c] = a + b;
        t[(p + h) * C + c] = a - b;
      }
      __syncthreads();
    }
    for (int e = tid; e < P.len * C; e += nthr) {
      const int p = e / C, c = e % C;
      float y = t[e];
      if (rsgn) y *= rsgn[o * P.row_o + p * P.row_p];
      base[(size_t)p * P.step + c] = y * P.scale;
    }
    __syncthreads();
  }
}

int grid_for(long long items, int max_blocks) {
  return (int)(items < max_blocks ? items : max_blocks);
}

// ---------------------------------------------------------------------------
// Tiled FWHT for n >= 64.  Stage h acts on index bit log2(h); on a tile of whole
// rows, laid out contiguously, the row transform is the stages on bits [0, log2 n)
// and the column transform within the tile the stages on the row bits above.
// Every element sees the additions of fwht_numpy in the same order, so results are
// bit-identical to the per-stage kernels.  Both passes are bound by HBM: what they
// need is every access coalesced, few barriers and several workgroups per CU.
//
//   pass 1 (fwht_tile_kernel): tiles of up to 2^14 floats, 32 per thread.  A wave
//     owns 2^11 consecutive floats and does bits 0-10 in registers: bits 0, 1 lie
//     in a float4, bits 2-5 in lane bits 0-3 (DPP), bits 6-10 in lane bits 4, 5 and
//     the register index (v_permlane16/32_swap turn a lane bit into a register
//     bit).  Bits 11-13 take one exchange through LDS, after which a thread holds
//     the float4s 2^11 floats apart.
//   pass 2 (fwht_cols2_kernel): column stages h0 <= h < h0 * len, 64 <= len <= 1024,
//     on tiles of len rows spaced h0 apart x 32 columns (128 contiguous bytes of a
//     row): half of the row bits in registers, one exchange through LDS, the other
//     half.  len <= 32 needs no exchange (fwht_cols1_kernel).
//
// 8192 x 2048: 25.5 and 25.3 us, 5.3 TB/s of HBM traffic each, the rate of a
// device-to-device copy; the whole transform 71 -> 51 us.  Before, a thread read 32
// consecutive floats (64 cache lines an instruction) and each pass ran radix-8 steps
// with four exchanges and one 1,024-thread workgroup per CU in pass 2: 36 us a pass.
// 2048 x 2048: 11 and 7 us; 512 x 2048: 6.5 and 4.3 us.
// ---------------------------------------------------------------------------
constexpr int kWaveBits = 11;  // floats of a wave's block in pass 1
constexpr int kTileBits = 14;  // largest pass-1 tile: 64 KiB of LDS, two workgroups per CU
constexpr int kColBits = 5;    // pass-2 tile width: 32 columns
constexpr int kColLenBits = 10;
constexpr int kFlatThreads = 256;
constexpr int kMaxGrid = 1 << 20;  // workgroups of a launch; the kernels' loops take the rest

// Butterflies of register bits [K0, K1) of v[0..E).
template <int K0, int K1, int E>
__device__ __forceinline__ void slot_stages(float (&v)[E]) {
#pragma unroll
  for (int hs = 1 << K0; hs < (1 << K1); hs <<= 1) {
#pragma unroll
    for (int s = 0; s < E; ++s) {
      if (!(s & hs)) {
        const float a = v[s], b = v[s + hs];
        v[s] = a + b;
        v[s + hs] = a - b;
      }
    }
  }
}

template <int CTRL>
__device__ __forceinline__ float dpp(float x) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true));
}

// The partner of lane l: l ^ (1 << K).
template <int K>
__device__ __forceinline__ float lane_partner(float x) {
  if constexpr (K == 0) return dpp<0xB1>(x);              // quad_perm 1,0,3,2
  else if constexpr (K == 1) return dpp<0x4E>(x);         // quad_perm 2,3,0,1
  else if constexpr (K == 2) return dpp<0x1B>(dpp<0x141>(x));  // half-row mirror (l ^ 7), quad_perm 3,2,1,0 (l ^ 3)
  else return dpp<0x128>(x);                              // row rotate by 8
}

// One butterfly stage on lane bit K (0-3): the lower lane's a + b, the upper's
// a - b, as partner + (+-own); the product with +-1 is exact, so the sum rounds as
// the plain addition.
template <int K, int E>
__device__ __forceinline__ void lane_stage(float (&v)[E], int lane) {
  const float sgn = (lane >> K) & 1 ? -1.0f : 1.0f;
#pragma unroll
  for (int s = 0; s < E; ++s) v[s] = __builtin_fmaf(v[s], sgn, lane_partner<K>(v[s]));
}

// Exchanges lane bit 4 (HALF = false) or 5 with register bit B of v.
template <bool HALF, int B, int E>
__device__ __forceinline__ void swap_lane_reg(float (&v)[E]) {
#pragma unroll
  for (int s = 0; s < E; ++s) {
    if (!(s & (1 << B))) {
      const uint32_t x = __builtin_bit_cast(uint32_t, v[s]), y = __builtin_bit_cast(uint32_t, v[s + (1 << B)]);
      const auto r = HALF ? __builtin_amdgcn_permlane32_swap(x, y, false, false)
                          : __builtin_amdgcn_permlane16_swap(x, y, false, false);
      v[s] = __builtin_bit_cast(float, (uint32_t)r[0]);
      v[s + (1 << B)] = __builtin_bit_cast(float, (uint32_t)r[1]);
    }
  }
}

// p[i] by a 32-bit byte offset from a uniform pointer (one address register).
template <typename V, typename F>
__device__ __forceinline__ V* at32(F* p, uint32_t i) {
  using B = std::conditional_t<std::is_const_v<F>, const char, char>;
  return reinterpret_cast<V*>(reinterpret_cast<B*>(p) + (i << 2));
}

struct TileParams {
  const float* x;
  float* out;
  int batch;
  int m;                  // rows per matrix
  int n;                  // row length, 64 <= n <= 16384, power of two
  int rb;                 // rows per tile (power of two, rb * n <= 2^14, rb | m)
  int end_bit;            // stages on tile bits [0, end_bit)
  const float* pre_col;   // (batch, n) and
  const float* pre_row;   // (batch, m) multiply the input (PRE)
  const float* post_col;  // (batch, n) multiplies the result (POST), as does
  const float* post_row;  // (batch, m), unless null (a later pass applies it)
  float scale;            // multiplies every element at the store
};

// Column signs commute with the column transform, and row signs with the row
// transform, exactly, so the signs between the two apply at the load (forward,
// PRE) or at the store (inverse, POST).  Their loads are issued beside the data's
// and before the barrier: a tile waits for memory once on each side.
// VEC: out is 16-byte aligned (decided at run time, the two kinds of store were
// merged into scalar ones).
template <bool PRE, bool POST, bool VEC>
__global__ __launch_bounds__(1 << (kTileBits - 5), 4) void fwht_tile_kernel(TileParams P) {
  extern __shared__ __align__(16) float t[];
  const uint32_t n = (uint32_t)P.n, rb = (uint32_t)P.rb;
  const uint32_t nb = (uint32_t)__builtin_ctz(n);
  const uint32_t T = rb * n;  // a multiple of 64
  const int end = P.end_bit;
  const uint32_t tiles_per_mat = (uint32_t)P.m / rb;
  const long long tiles = (long long)P.batch * tiles_per_mat;
  for (long long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint32_t e = (uint32_t)(tile / tiles_per_mat);
    const uint32_t r0 = (uint32_t)(tile - (long long)e * tiles_per_mat) * rb;
    const size_t row0 = (size_t)e * P.m + r0, off = row0 * n;  // the tile is rb consecutive rows
    const float* src = P.x + off;
    float* dst = P.out + off;
    // formed again for every tile: indices held over the loop spilled 43 registers
    uint32_t tid = threadIdx.x;
    asm("" : "+v"(tid) : "s"(r0));
    const int lane = tid & 63;
    const uint32_t w0 = (tid >> 6) << kWaveBits;  // the wave's block of the tile

    auto col4 = [&](const float* p, uint32_t i) {  // the column factors of tile index i
      return *at32<const float4>(p + (size_t)e * n, i & (n - 1));
    };
    // row factors of tile indices i0 + step s, s < F (past a short tile: index 0's)
    auto end_rows = [&](auto& f, uint32_t i0, uint32_t step) {
      constexpr int F = sizeof(f) / sizeof(float);
#pragma unroll
      for (int s = 0; s < F; ++s) f[s] = 1.0f;
      if (POST && P.post_row) {
#pragma unroll
        for (int s = 0; s < F; ++s) {
          const uint32_t i = i0 + step * s;
          f[s] = *at32<const float>(P.post_row + row0, (i < T ? i : 0) >> nb);
        }
      }
#pragma unroll
      for (int s = 0; s < F; ++s) f[s] *= P.scale;
    };
    auto store4 = [&](uint32_t i, float4 q, float f, float4 p) {
      q.x *= f; q.y *= f; q.z *= f; q.w *= f;
      if constexpr (POST) {
        q.x *= p.x; q.y *= p.y; q.z *= p.z; q.w *= p.w;
      }
      if constexpr (VEC) {
        *at32<float4>(dst, i) = q;
      } else {
        float* d = at32<float>(dst, i);
        d[0] = q.x; d[1] = q.y; d[2] = q.z; d[3] = q.w;
      }
    };

    // float4 j of a lane: tile index w0 + 256 j + 4 lane; register 4 j + (bits 0, 1)
    float v[32];
    {
      float4 q[8], pc[PRE ? 8 : 1];
      float pr[PRE ? 8 : 1];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        const uint32_t i = w0 + 256u * j + 4u * lane;
        const uint32_t il = i < T ? i : 0;  // past a short tile: read again, not stored
        q[j] = *at32<const float4>(src, il);
        if constexpr (PRE) {
          pc[j] = col4(P.pre_col, il);
          pr[j] = *at32<const float>(P.pre_row + row0, il >> nb);
        }
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        float4 a = q[j];
        if constexpr (PRE) {
          a.x *= pc[j].x * pr[j]; a.y *= pc[j].y * pr[j]; a.z *= pc[j].z * pr[j]; a.w *= pc[j].w * pr[j];
        }
        v[4 * j] = a.x; v[4 * j + 1] = a.y; v[4 * j + 2] = a.z; v[4 * j + 3] = a.w;
      }
    }
    slot_stages<0, 2>(v);  // bits 0, 1
    __builtin_amdgcn_sched_barrier(0);
    lane_stage<0>(v, lane);
    lane_stage<1>(v, lane);
    lane_stage<2>(v, lane);
    lane_stage<3>(v, lane);  // bits 2-5 (n >= 64: row bits)
    __builtin_amdgcn_sched_barrier(0);
    // bits 6, 7, 8 pass through register bit 2; end is uniform
    swap_lane_reg<false, 2>(v);
    if (end > 6) slot_stages<2, 3>(v);
    swap_lane_reg<true, 2>(v);
    if (end > 7) slot_stages<2, 3>(v);
    swap_lane_reg<false, 2>(v);
    if (end > 8) slot_stages<2, 3>(v);
    if (end > 9) slot_stages<3, 4>(v);
    if (end > 10) slot_stages<4, 5>(v);
    __builtin_amdgcn_sched_barrier(0);
    // now lane bits 0-3, 4, 5 hold tile bits 2-5, 7, 6
    const uint32_t i0 = w0 + 4u * (lane & 15) + 128u * ((lane >> 4) & 1) + 64u * (lane >> 5);
    if (end <= kWaveBits) {
#pragma unroll
      for (int h = 0; h < 8; h += 4) {
        float f[4];
        float4 p[4] = {};
        end_rows(f, i0 + 256u * h, 256u);
        if constexpr (POST) {
#pragma unroll
          for (int j = 0; j < 4; ++j) p[j] = col4(P.post_col, i0 + 256u * (h + j));
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const uint32_t i = i0 + 256u * (h + j);
          const int k = 4 * (h + j);
          if (i < T) store4(i, make_float4(v[k], v[k + 1], v[k + 2], v[k + 3]), f[j], p[j]);
        }
      }
      continue;
    }
    // bits 11 .. end - 1 (T >= 2^12, whole blocks): float4s 2^11 floats apart
#pragma unroll
    for (int j = 0; j < 8; ++j)
      *reinterpret_cast<float4*>(t + i0 + 256u * j) = make_float4(v[4 * j], v[4 * j + 1], v[4 * j + 2], v[4 * j + 3]);
    auto exchange = [&](auto kc) {
      constexpr int K = decltype(kc)::value, E = 1 << K;
#pragma unroll 1
      for (int r = 0; r < 8 / E; ++r) {  // T / 32 threads, T / (4 E) groups
        const uint32_t g = tid + r * blockDim.x;
        const uint32_t i = ((g & 511u) << 2) | ((g >> 9) << (kWaveBits + K));
        float f[E];
        float4 p[E] = {};
        end_rows(f, i, 1u << kWaveBits);
        if constexpr (POST) {
          if (n <= 1u << kWaveBits) {  // the same columns in every row
            p[0] = col4(P.post_col, i);
#pragma unroll
            for (int s = 1; s < E; ++s) p[s] = p[0];
          } else {
#pragma unroll
            for (int s = 0; s < E; ++s) p[s] = col4(P.post_col, i + ((uint32_t)s << kWaveBits));
          }
        }
        if (r == 0) __syncthreads();
        float u[4][E];
#pragma unroll
        for (int s = 0; s < E; ++s) {
          const float4 q = *reinterpret_cast<const float4*>(t + i + ((uint32_t)s << kWaveBits));
          u[0][s] = q.x; u[1][s] = q.y; u[2][s] = q.z; u[3][s] = q.w;
        }
#pragma unroll
        for (int c = 0; c < 4; ++c) slot_stages<0, K>(u[c]);
#pragma unroll
        for (int s = 0; s < E; ++s)
          store4(i + ((uint32_t)s << kWaveBits), make_float4(u[0][s], u[1][s], u[2][s], u[3][s]), f[s], p[s]);
      }
    };
    if (end == kWaveBits + 3) exchange(std::integral_constant<int, 3>());
    else if (end == kWaveBits + 2) exchange(std::integral_constant<int, 2>());
    else exchange(std::integral_constant<int, 1>());
    __syncthreads();
  }
}

struct ColPassParams {
  float* x;               // (batch, m, n) transformed in place
  int batch, m, n;
  int h0;                 // first stage span of the pass
  int len;                // rows per group (power of two <= 1024): stages h0 .. h0 * len / 2
  const float* row_end;   // (batch, m) multiplies row r at the store, or null
  float scale;            // multiplies every element at the store
};

// m, n, h0 and len are powers of two.  Group o of a matrix holds the rows (o / h0) h0 len + o mod h0 + p h0, p < len.
__device__ __forceinline__ uint32_t group_row(const ColPassParams& P, uint32_t o) {
  const uint32_t h0 = (uint32_t)P.h0;
  return (o & ~(h0 - 1u)) * (uint32_t)P.len + (o & (h0 - 1u));
}

// len = 2^LA <= 32: a thread holds a column of a group.
template <int LA>
__global__ __launch_bounds__(kFlatThreads) void fwht_cols1_kernel(ColPassParams P) {
  constexpr int E = 1 << LA;
  const uint32_t n = (uint32_t)P.n, per_mat = (uint32_t)P.m >> LA;
  const size_t rstride = (size_t)P.h0 * n;
  const long long total = (long long)P.batch * per_mat * n;  // a multiple of 64
  for (long long g = (long long)blockIdx.x * kFlatThreads + threadIdx.x; g < total;
       g += (long long)gridDim.x * kFlatThreads) {
    const uint32_t c = (uint32_t)g & (n - 1u);
    const long long eo = g >> __builtin_ctz(n);
    const uint32_t e = (uint32_t)(eo >> __builtin_ctz(per_mat)), o = (uint32_t)eo & (per_mat - 1u);
    const size_t row = (size_t)e * P.m + group_row(P, o);
    float* base = P.x + row * n + c;
    float v[E];
#pragma unroll
    for (int s = 0; s < E; ++s) v[s] = base[s * rstride];
    slot_stages<0, LA>(v);
#pragma unroll
    for (int s = 0; s < E; ++s) {
      const float f = P.row_end ? P.row_end[row + (size_t)s * P.h0] * P.scale : P.scale;
      base[s * rstride] = v[s] * f;
    }
  }
}

// len = 2^(LA + LB): row bits [0, LA) of a group in registers, one exchange through
// LDS, row bits [LA, LA + LB).  A wave holds 32 columns of two rows; the exchange
// flips a row's lowest bit by bit LA, so the two fall in different LDS banks.
template <int LA, int LB>
__global__ __launch_bounds__(32 << LB) void fwht_cols2_kernel(ColPassParams P) {
  static_assert(LA >= LB && LB > 0, "a thread holds one group of the first half");
  extern __shared__ __align__(16) float t[];
  constexpr uint32_t C = 1u << kColBits, LEN = 1u << (LA + LB);
  constexpr int EA = 1 << LA, EB = 1 << LB;
  const uint32_t n = (uint32_t)P.n, h0 = (uint32_t)P.h0;
  const uint32_t per_mat = (uint32_t)P.m / LEN, ncb = n / C;
  float* f_end = t + LEN * C;  // LEN row factors (times scale)
  const long long tiles = (long long)P.batch * per_mat * ncb;
  const uint32_t c = threadIdx.x & (C - 1u), q = threadIdx.x >> kColBits;  // q < EB
  const size_t rbytes = (size_t)h0 * n * sizeof(float);  // from tile row to tile row
  for (long long tile = blockIdx.x; tile < tiles; tile += gridDim.x) {
    const uint32_t e = (uint32_t)(tile / ((long long)per_mat * ncb));
    const uint32_t rest = (uint32_t)(tile - (long long)e * per_mat * ncb);
    const uint32_t o = rest / ncb, cb = rest - o * ncb;
    const size_t row = (size_t)e * P.m + group_row(P, o);
    char* base = reinterpret_cast<char*>(P.x + row * n + (size_t)cb * C);
    {
      // uniform row base + 32-bit lane offset (a matrix has at most 1 GiB)
      const uint32_t vo = ((q << LA) * h0 * n + c) * 4u;
      float v[EA];
#pragma unroll
      for (int s = 0; s < EA; ++s) v[s] = *reinterpret_cast<const float*>(base + s * rbytes + vo);
      for (uint32_t p = threadIdx.x; p < LEN; p += blockDim.x)
        f_end[p] = P.row_end ? P.row_end[row + (size_t)p * h0] * P.scale : P.scale;
      slot_stages<0, LA>(v);
#pragma unroll
      for (int s = 0; s < EA; ++s) t[((((q << LA) + s) ^ (q & 1u)) << kColBits) + c] = v[s];
    }
    __syncthreads();
#pragma unroll
    for (int k = 0; k < EA / EB; ++k) {
      const uint32_t lo = q + (uint32_t)(k * EB);  // < EA
      const uint32_t vo = (lo * h0 * n + c) * 4u;
      float v[EB];
#pragma unroll
      for (int s = 0; s < EB; ++s) v[s] = t[(((lo + ((uint32_t)s << LA)) ^ (s & 1u)) << kColBits) + c];
      slot_stages<0, LB>(v);
#pragma unroll
      for (int s = 0; s < EB; ++s)
        *reinterpret_cast<float*>(base + ((size_t)s << LA) * rbytes + vo) = v[s] * f_end[lo + ((uint32_t)s << LA)];
    }
    __syncthreads();
  }
}

template <bool PRE, bool POST>
const void* tile_kernel_ptr(bool vec) {
  return vec ? reinterpret_cast<const void*>(&fwht_tile_kernel<PRE, POST, true>)
             : reinterpret_cast<const void*>(&fwht_tile_kernel<PRE, POST, false>);
}

const void* cols1_kernel_ptr(int bits) {
  switch (bits) {
    case 1: return reinterpret_cast<const void*>(&fwht_cols1_kernel<1>);
    case 2: return reinterpret_cast<const void*>(&fwht_cols1_kernel<2>);
    case 3: return reinterpret_cast<const void*>(&fwht_cols1_kernel<3>);
    case 4: return reinterpret_cast<const void*>(&fwht_cols1_kernel<4>);
    default: return reinterpret_cast<const void*>(&fwht_cols1_kernel<5>);
  }
}

const void* cols2_kernel_ptr(int bits) {
  switch (bits) {
    case 6: return reinterpret_cast<const void*>(&fwht_cols2_kernel<3, 3>);
    case 7: return reinterpret_cast<const void*>(&fwht_cols2_kernel<4, 3>);
    case 8: return reinterpret_cast<const void*>(&fwht_cols2_kernel<4, 4>);
    case 9: return reinterpret_cast<const void*>(&fwht_cols2_kernel<5, 4>);
    default: return reinterpret_cast<const void*>(&fwht_cols2_kernel<5, 5>);
  }
}

size_t cols2_lds(int bits) { return ((size_t)(1u << bits) * ((1u << kColBits) + 1)) * sizeof(float); }

}  // namespace

// Host launchers used by the C ABI.  Shapes are validated by the caller.
hipError_t launch_fwht_rows(const float* x, float* out, long long rows, int n, const float* pre,
                            const float* post, long long vec_rows, const float* row_sign, float scale,
                            int max_blocks, hipStream_t stream) {
  if (rows == 0) return hipSuccess;
  RowsParams P = {x, out, rows, n, pre, post, vec_rows > 0 ? vec_rows : rows, row_sign, scale};
  const size_t lds = (size_t)n * sizeof(float);  // n <= 16384: at most 64 KiB
  hipLaunchKernelGGL(fwht_rows_kernel, dim3(grid_for(rows, max_blocks)), dim3(kRowThreads), lds, stream, P);
  return hipGetLastError();
}

// Tiled RHT / row transform for n >= 64 (see fwht_tile_kernel).  Forward:
// pre_col = sign_r, pre_row = sign_l; inverse: post_col = sign_r, post_row = sign_l.
// col = false transforms rows only (m = row count, any value; no factors).
hipError_t launch_fwht_tiled(const float* x, float* out, int batch, int m, int n, bool col, const float* pre_col,
                             const float* pre_row, const float* post_col, const float* post_row, float scale,
                             hipStream_t stream) {
  if (batch == 0 || m == 0) return hipSuccess;
  static std::atomic<bool> attr_set[64];  // per device: opt-in to > 64 KiB of dynamic LDS
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= 64 || !attr_set[dev].load(std::memory_order_acquire)) {
    for (int bits = 9; bits <= kColLenBits; ++bits) {
      e = hipFuncSetAttribute(cols2_kernel_ptr(bits), hipFuncAttributeMaxDynamicSharedMemorySize,
                              (int)cols2_lds(bits));
      if (e != hipSuccess) return e;
    }
    if (dev >= 0 && dev < 64) attr_set[dev].store(true, std::memory_order_release);
  }
  const int nb = __builtin_ctz((unsigned)n);
  int tb = kTileBits;
  if (col) {
    // One pass where a matrix fits a tile.  Else a tile of 2^tb floats gives m n / 2^tb
    // workgroups in pass 1 and 2^tb / 32 in pass 2, so small matrices take the tb that
    // fills both alike: about half of log2(32 m n).
    const int lg = nb + __builtin_ctz((unsigned)m);
    if (lg <= kTileBits) tb = lg;
    else tb = std::max(nb, std::min(kTileBits, std::max(kWaveBits, (lg + kColBits + 1) / 2)));
  }
  int rb = 1 << (tb - nb);
  while (m % rb) rb >>= 1;  // rows only: the largest power of two that divides the row count
  const bool single = !col || rb == m;
  const int T = rb * n, end = col ? __builtin_ctz((unsigned)T) : nb;
  TileParams P1 = {x, out, batch, m, n, rb, end, pre_col, pre_row,
                   post_col, single ? post_row : nullptr, single ? scale : 1.0f};
  const long long tiles1 = (long long)batch * (m / rb);
  const int threads = std::max(64, T >> 5);
  void* args1[] = {&P1};
  const bool vec = (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  e = hipLaunchKernel(pre_col    ? tile_kernel_ptr<true, false>(vec)
                      : post_col ? tile_kernel_ptr<false, true>(vec)
                                 : tile_kernel_ptr<false, false>(vec),
                      dim3(grid_for(tiles1, kMaxGrid)), dim3(threads), args1,
                      end > kWaveBits ? (size_t)T * sizeof(float) : 0, stream);
  if (e != hipSuccess || single) return e;
  for (int h0 = rb; h0 < m;) {
    const int bits = std::min(__builtin_ctz((unsigned)(m / h0)), kColLenBits);
    const int len = 1 << bits;
    const bool fin = h0 * len == m;
    ColPassParams P2 = {out, batch, m, n, h0, len, fin ? post_row : nullptr, fin ? scale : 1.0f};
    void* args[] = {&P2};
    if (bits <= 5) {
      const long long blocks = ((long long)batch * (m >> bits) * n + kFlatThreads - 1) / kFlatThreads;
      e = hipLaunchKernel(cols1_kernel_ptr(bits), dim3(grid_for(blocks, kMaxGrid)), dim3(kFlatThreads), args, 0,
                          stream);
    } else {
      const long long tiles2 = (long long)batch * (m >> bits) * (n >> kColBits);
      e = hipLaunchKernel(cols2_kernel_ptr(bits), dim3(grid_for(tiles2, kMaxGrid)), dim3(32 << (bits / 2)), args,
                          cols2_lds(bits), stream);
    }
    if (e != hipSuccess) return e;
    h0 *= len;
  }
  return hipSuccess;
}

// H_m applied to every column of each (m, n) matrix of x (batch of them), in
// place; the result is multiplied by row_sign (batch, m) (after the transform)
// and scale.  m, n powers of two.
hipError_t launch_fwht_cols(float* x, int batch, int m, int n, const float* row_sign, float scale,
                            int max_blocks, hipStream_t stream) {
  if (batch == 0) return hipSuccess;
  const long long ms = (long long)m * n;
  const int b = m < 128 ? m : 128;
  const int a = m / b;
  const int C = n < kColTile ? n : kColTile;
  // pass 1: stages h < b, tiles of b consecutive rows
  ColsParams P1 = {x, ms, m, n, C, b, n, (long long)b * n, a, batch, nullptr, 0, 0, 1.0f};
  if (a == 1) {  // the only pass: signs and scale here
    P1.row_sign = row_sign;
    P1.row_o = 0;
    P1.row_p = 1;
    P1.scale = scale;
  }
  hipLaunchKernelGGL(fwht_cols_kernel, dim3(grid_for((long long)batch * a * (n / C), max_blocks)),
                     dim3(kColThreads), (size_t)b * C * sizeof(float), stream, P1);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || a == 1) return e;
  // pass 2: stages h >= b, tiles of a rows spaced b apart (row = ia*b + ib)
  ColsParams P2 = {x, ms, m, n, C, a, (long long)b * n, n, b, batch, row_sign, 1, b, scale};
  hipLaunchKernelGGL(fwht_cols_kernel, dim3(grid_for((long long)batch * b * (n / C), max_blocks)),
                     dim3(kColThreads), (size_t)a * C * sizeof(float), stream, P2);
  return hipGetLastError();
}

}  // namespace bcjr
