// Soft forward and backward of the BCJR node in two halves, for kV <= 2 and
// batches that leave half of the chip idle in one launch per sequence.
//
// The recursions, outputs and two-halves scheme of bcjr_soft16.h: the first
// launch runs alpha over steps 0..h-1 and beta over N-1..h on a workgroup each,
// both storing their raw inputs at [t][u] of the sequence's slot; the second goes
// on with alpha over h..N-1 and beta over h-1..0, each forming the marginals of
// its steps from what the other one stored.  log Z and E[F] come from the two
// state vectors where the sweeps meet.  N steps in sequence in place of 2N; the
// launch boundary is the only synchronisation.
//
// A workgroup has its CU to itself here, so it takes up to 1,024 threads (four
// waves per SIMD): kV = 2 whole butterflies, UPT = 2^(L-14) per thread, from
// L = 12 on (LPB = 1), and below that a lane per output (LPB = R, the R lanes of
// a butterfly in one wave); a step is bound by the latency of its chain of
// exponentials, sums, reductions and the barrier.  The state vector (GRAD: (m~, mu)
// pairs) is double-buffered in natural order, or, where two of them exceed the LDS
// (GRAD, L = 16), updated in place (Swizzle).  What the opposite sweep stored comes
// back two butterflies ahead of its use, except at UPT = 4, where the waves' other
// butterflies cover the latency and the registers are short.
//
// Measured, one launch -> two halves, N = 256, T = 0.1, forward and backward: L = 12,
// 1MAD, 128 sequences 0.36 -> 0.23 and 0.57 -> 0.30 ms; L = 14, 3INST, 128 sequences
// 0.74 -> 0.42 and 1.15 -> 0.67 ms; L = 16, 8 sequences 1.91 -> 1.07 and 3.48 ->
// 1.80 ms, 128 sequences 2.00 -> 1.28 and 3.56 -> 2.22 ms (T = 0.06: 2.54 -> 1.57
// and 3.63 -> 2.37 ms); HYB k = 1 at L = 16, 64 sequences 2.29 -> 1.20 and 3.16 ->
// 1.67 ms.
#pragma once

#include "bcjr_device.h"
#include "bcjr_kernels.h"
#include "bcjr_soft_common.h"

namespace bcjr {

// Codewords of a lane kept in VGPRs over a sweep: all of them up to 64 values,
// except in the backward's gradient-forming sweep past 16 and in the computed
// codes' low-temperature variant past 16, whose working sets need the registers.
// A table's variant holds them there too, and unrolls its units where it does not,
// so that their reads overlap: read one unit after the other, they cost more than
// the halves save (T = 0.06, N = 96, 8 sequences, forward, backward, entropy:
// L = 15 0.78, 0.83, 0.79 -> 0.26, 0.57, 0.28 ms, in one launch 0.56, 0.71, 0.52;
// L = 16 1.46, 1.58, 1.46 -> 0.45, 1.03, 0.49, in one launch 1.03, 1.48, 1.55).
constexpr bool halves_cached(int values, bool grad_marg, bool exact_computed) {
  return values <= ((grad_marg || exact_computed) ? 16 : 64);
}

template <int KV, int V, int CODE, int UPT, int LPB, bool GRAD, bool ENT>
__global__ __launch_bounds__(1024, 4) void bcjr_halves_kernel(Soft16Params P) {
  constexpr int R = 1 << KV, RO = R / LPB, UW = 64 / LPB;
  constexpr int ST = GRAD ? 2 : 1;               // floats of a state element
  constexpr int NS = V + (GRAD || ENT ? 1 : 0);  // sums of a marginal-forming step
  constexpr bool INPLACE = halves_in_place(GRAD, UPT, LPB);
  using CT = CodeTraits<CODE>;
  static_assert(KV <= 2 && (LPB == 1 || LPB == R), "whole butterflies, or a lane per output");
  static_assert(!(GRAD && ENT), "the entropy is an output of the forward");

  extern __shared__ __align__(16) unsigned char smem[];
  const int L = P.L, N = P.N, nb = L - KV;
  const int NT = 1 << nb, NB = NT >> KV;
  const int tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63, wave = tid >> 6, nwaves = nthr >> 6;
  const int part = lane / UW;                    // output of the lane (LPB = R)
  const int uq = wave * UW + (lane & (UW - 1));  // its first butterfly; the others US apart
  const int US = NB / UPT;
  const bool live = uq < US;
  const int u0 = min(uq, US - 1);
  const int b = blockIdx.x >> 1, role = blockIdx.x & 1;  // role 0: alpha, 1: beta

  const uint32_t state0 = CODE == CODE_HYB ? 16u << P.Q : 0u;  // behind the signed LUT
  float* stv = reinterpret_cast<float*>(smem + state0);           // ST * NT, twice unless in place
  double* ovec = reinterpret_cast<double*>(stv + (INPLACE ? 1 : 2) * ST * NT);  // N  offsets of the stored inputs
  float* wmax = reinterpret_cast<float*>(ovec + ((N + 1) & ~1));    // 2 * kMaxWaves
  float* apart = wmax + 2 * kMaxWaves;                             // max(2 * nwaves * NS, 2 * kMaxWaves + 4)
  const int napart = max(2 * nwaves * NS, 2 * kMaxWaves + 4);
  float* wsum = apart;                                             // 2 * kMaxWaves, before the sweep
  int* bflag = reinterpret_cast<int*>(apart + 2 * kMaxWaves);      // input flag
  float* wbuf = apart + napart;                                    // N * V
  float* gbuf = wbuf + N * V;                                      // GRAD: N * V
  float* lut = reinterpret_cast<float*>(smem);

  if constexpr (CODE == CODE_HYB) stage_hyb_signed(reinterpret_cast<float2*>(lut), P.table, P.Q, tid, nthr);
  const uint32_t ANT = opaque_uniform(CT::A * (uint32_t)NT);
  const Swizzle swz = P.swz;
  constexpr int LGB = GRAD ? 3 : 2;
  auto el_off = [&](uint32_t x, int rho) -> uint32_t { return swizzle(rotr_bits(x, rho, nb), swz) << LGB; };

  float* slot = P.ws + (size_t)b * P.slot_floats;
  const float Tb = P.T[P.t_per_seq ? b : 0];
  const float sk = sqrtf(kLog2e / Tb);
  const float ssk = CT::kSigma * sk;
  const float gZ = GRAD && P.g_logZ ? P.g_logZ[b] : 0.0f;
  const float twoT = 2.0f / Tb;
  const float* seqb = P.seq + (size_t)b * N * V;
  float* outb = P.out + (size_t)b * N * V;

  for (int i = tid; i < 2 * kMaxWaves; i += nthr) wmax[i] = -INFINITY;  // waves that do not exist
  if (!soft_inputs<GRAD>(seqb, P.g_soft + (GRAD ? (size_t)b * N * V : 0), N * V, Tb, gZ, wbuf, gbuf, bflag)) {
    if (role == 0 && P.mode == SOFT_SECOND) soft_fill_nan<GRAD, ENT>(P, b, outb, N * V);
    return;
  }
  __syncthreads();  // the flag's words serve as wsum below

  double logZ2 = 0.0;
  float EFg = 0.0f;  // E[F] - g_Z

  // Result of step t from the per-wave partials in buffer par (wave 0).
  auto step_out = [&](int t, int par) __attribute__((always_inline)) {
    soft_step_out<GRAD, ENT, V>(apart + par * nwaves * NS, nwaves, wbuf + t * V, twoT, outb + t * V,
                                ENT ? P.H_out + (size_t)b * N + t : nullptr);
  };

  // One sweep over steps t0, t0 + dt, ... (n of them), dt = +1 (alpha) or -1
  // (beta), from the state vector in (the first buffer of) LDS with running offset
  // `off`; O0 is the first step's offset.  Returns the offset after it.
  auto sweep = [&](auto beta_tag, auto marg_tag, auto exact_tag, int t0, int n, double off,
                   float O0) __attribute__((always_inline)) -> double {
    constexpr bool BETA = decltype(beta_tag)::value, MARG = decltype(marg_tag)::value;
    constexpr bool EXACT = decltype(exact_tag)::value;
    constexpr bool CACHE = V == 1 && halves_cached(UPT * R * RO, GRAD && MARG, EXACT && CODE != CODE_TABLE);
    constexpr int dt = BETA ? -1 : 1;
    const int o_lane = LPB == 1 ? 0 : part;
    // Codeword of output j + o_lane, input i of unit q: state p*NT + R*u + c with
    // (p, c) = (i, o) in the alpha direction and (o, i) in the beta direction.
    const uint32_t sl = (uint32_t)(R * u0) + (BETA ? (uint32_t)o_lane << nb : (uint32_t)o_lane);
    auto codeword_of = [&](uint32_t sl_s, int q, int j, int i, float (&h)[V]) {
      const uint32_t p = (uint32_t)(BETA ? j : i), c = (uint32_t)(BETA ? i : j);
      if constexpr (CODE == CODE_1MAD || CODE == CODE_3INST) {
        h[0] = raw_from_hash<CODE>(sl_s + CT::A * (uint32_t)R * (uint32_t)(q * US) + p * ANT + CT::A * c);
      } else {
        raw_codeword<CODE, V>(0u, 0u, sl_s + (uint32_t)(R * q * US) + (p << nb) + c, P.table, lut, P.Q, h);
      }
    };
    const uint32_t base = CODE == CODE_1MAD || CODE == CODE_3INST ? CT::A * sl + CT::B : sl;
    float hc[CACHE ? UPT : 1][CACHE ? RO : 1][CACHE ? R : 1];
    if constexpr (CACHE) {
      const uint32_t b0 = (uint32_t)opaque((int)base);
#pragma unroll
      for (int q = 0; q < UPT; ++q)
#pragma unroll
        for (int j = 0; j < RO; ++j)
#pragma unroll
          for (int i = 0; i < R; ++i) {
            float h[V];
            codeword_of(b0, q, j, i, h);
            hc[q][j][i] = h[0];
          }
    }

    // What the opposite sweep stored for the lane's outputs, two units ahead.
    constexpr bool AHEAD = MARG && UPT <= 2;
    auto stored = [&](int t, int q) -> float* {
      return slot + ((size_t)t * NB + u0 + q * US) * (R * ST) + (size_t)(o_lane * ST);
    };
    float pa[AHEAD ? RO * ST : 1], pb[AHEAD ? RO * ST : 1];
    if constexpr (AHEAD) {
      load_vec<RO * ST>(stored(t0, 0), pa);
      if (UPT > 1 || n > 1) load_vec<RO * ST>(stored(UPT > 1 ? t0 : t0 + dt, UPT > 1 ? 1 : 0), pb);
    }
    int rho = (int)(((long long)KV * (t0 - 1) % nb + nb) % nb);
    for (int st = 0; st < n; ++st) {
      const int t = t0 + dt * st;
      float O = O0;
      if (st > 0) {
        O = block_max(wmax + ((st + 1) & 1) * kMaxWaves);
        if (MARG && wave == 0) step_out(t - dt, (st + 1) & 1);
      }
      // alpha: the inputs' offset is C_{t-1}; beta: D_t
      const float Kt = MARG ? (float)(ovec[t] + off - logZ2) : 0.0f;
      if (!MARG && tid == 0) ovec[t] = off;
      off += (double)O;
      float nw[V], sg[V];
#pragma unroll
      for (int v = 0; v < V; ++v) {
        nw[v] = -wbuf[t * V + v] * sk;
        sg[v] = GRAD ? CT::kSigma * gbuf[t * V + v] : 0.0f;
      }
      const uint32_t yu = INPLACE ? el_off((uint32_t)u0, rho) : 0u;
      const uint32_t K1 = INPLACE ? el_off((uint32_t)NB, rho) : 0u, K2 = INPLACE ? el_off((uint32_t)NB << 1, rho) : 0u;
      auto koff = [&](int q) -> uint32_t { return ((q & 1) ? K1 : 0u) ^ ((q & 2) ? K2 : 0u); };
      const float* prev = stv + (st & 1) * ST * NT;
      float* cur = stv + ((st + 1) & 1) * ST * NT;
      float tmax = -INFINITY, acc[NS];
#pragma unroll
      for (int v = 0; v < NS; ++v) acc[v] = 0.0f;
      if (live) {
        // One unit: unrolled, or in the low-temperature variant of the codes it computes,
        // a loop, so that one unit's registers serve all.
        auto unit = [&](int q) __attribute__((always_inline)) {
          __builtin_amdgcn_sched_barrier(0);
          // (also keeps the hashes inside the step)
          const uint32_t base_s = CACHE ? base : (uint32_t)opaque((int)base);
          const uint32_t yi = yu ^ (INPLACE && q ? el_off((uint32_t)(q * US), rho) : 0u);
          const int u = u0 + q * US;
          float m[R], mu[GRAD ? R : 1], po[MARG ? RO * ST : 1];
          if constexpr (MARG && !AHEAD) load_vec<RO * ST>(stored(t, q), po);
          if constexpr (AHEAD) {
#pragma unroll
            for (int i = 0; i < RO * ST; ++i) {
              po[i] = pa[i];
              pa[i] = pb[i];
            }
            const int ahead = q + 2, tt = st + ahead / UPT;
            if (tt < n) load_vec<RO * ST>(stored(t0 + dt * tt, ahead % UPT), pb);
          }
          if constexpr (INPLACE) {
#pragma unroll
            for (int i = 0; i < R; ++i) {
              const float2 v2 = *reinterpret_cast<const float2*>(smem + state0 + (yi ^ koff(i)));
              m[i] = v2.x;
              mu[i] = v2.y;
            }
          } else {  // alpha reads elements i*NB + u, beta R*u + i
            float in[R * ST];
            if constexpr (BETA) {
              load_vec<R * ST>(prev + R * ST * u, in);
            } else {
#pragma unroll
              for (int i = 0; i < R; ++i) load_vec<ST>(prev + ST * (i * NB + u), in + ST * i);
            }
#pragma unroll
            for (int i = 0; i < R; ++i) {
              m[i] = in[ST * i];
              if constexpr (GRAD) mu[i] = in[2 * i + 1];
            }
          }
          if constexpr (!MARG) {  // the lane's share of the raw inputs: those of its output positions
            float own[RO * ST];
            if constexpr (LPB == 1) {
#pragma unroll
              for (int j = 0; j < RO; ++j) {
                own[ST * j] = m[j];
                if constexpr (GRAD) own[2 * j + 1] = mu[j];
              }
            } else {
              load_vec<ST>(prev + ST * (BETA ? R * u + o_lane : o_lane * NB + u), own);
            }
            store_vec<RO * ST>(stored(t, q), own);
          }
          const float M = max_of_inputs(m);
#pragma unroll
          for (int i = 0; i < R; ++i) m[i] -= M;
          const float oout = O - M, kts = Kt + M;
          float no[RO], nuo[RO], g[NS], smin = INFINITY;

          // The unit's outputs; SHIFT: against each group's maximum.
          auto outputs = [&](auto shift_tag) __attribute__((always_inline)) {
            constexpr bool SHIFT = decltype(shift_tag)::value;
#pragma unroll
            for (int v = 0; v < NS; ++v) g[v] = 0.0f;
#pragma unroll
            for (int j = 0; j < RO; ++j) {
              float y[R], z[R], h[R][V], Mo = 0.0f;
#pragma unroll
              for (int i = 0; i < R; ++i) {
                if constexpr (CACHE) {
                  h[i][0] = hc[q][j][i];
                } else {
                  codeword_of(base_s, q, j, i, h[i]);
                }
                y[i] = m[i];
                if constexpr (GRAD) z[i] = mu[i];
#pragma unroll
                for (int v = 0; v < V; ++v) {
                  const float d = fmaf(h[i][v], ssk, nw[v]);
                  y[i] = fmaf(-d, d, y[i]);
                  if constexpr (GRAD) z[i] = fmaf(sg[v], h[i][v], z[i]);
                }
              }
              if constexpr (SHIFT) Mo = max_of_inputs(y);
              const float D = MARG && GRAD ? po[MARG && GRAD ? 2 * j + 1 : 0] - EFg : 0.0f;
              float s = 0.0f, w = 0.0f, x[V], ey = 0.0f;
#pragma unroll
              for (int i = 0; i < R; ++i) {
                const float e = fexp2(SHIFT ? y[i] - Mo : y[i]);
                s = i ? s + e : e;
                float wgt = e;
                if constexpr (GRAD) {
                  const float ez = e * z[i];
                  w = i ? w + ez : ez;
                  wgt = fmaf(e, D, ez);  // e (z + D)
                }
                if constexpr (MARG) {
#pragma unroll
                  for (int v = 0; v < V; ++v) x[v] = i ? fmaf(wgt, h[i][v], x[v]) : wgt * h[i][v];
                  if constexpr (ENT) ey = fmaf(e, y[i], ey);
                }
              }
              smin = fminf(smin, s);
              no[j] = flog2(s) + (Mo - oout);
              if constexpr (GRAD) nuo[j] = w * frcp(s);
              if constexpr (MARG) {
                const float pms = po[MARG ? ST * j : 0] + kts;
                const float G = fexp2(SHIFT ? pms + Mo : pms);
                // GRAD: sum_s dll_t(s) is accumulated, not assumed to be g_Z: its
                // computed value cancels the common-mode rounding in the gradient
                if constexpr (GRAD) g[0] = fmaf(G, fmaf(D, s, w), g[0]);
#pragma unroll
                for (int v = 0; v < V; ++v) g[v + (GRAD ? 1 : 0)] = fmaf(G, x[v], g[v + (GRAD ? 1 : 0)]);
                if constexpr (ENT) g[V] = fmaf(G, fmaf(pms, s, ey), g[V]);
              }
            }
          };
          outputs(std::integral_constant<bool, EXACT>{});
          if constexpr (!EXACT) {
            if (smin < kUnderflow) outputs(std::true_type{});  // a group underflowed: redo the unit's outputs
          }
          float out[RO * ST];
#pragma unroll
          for (int j = 0; j < RO; ++j) {
            out[ST * j] = no[j];
            if constexpr (GRAD) out[2 * j + 1] = nuo[j];
          }
          if constexpr (INPLACE) {
#pragma unroll
            for (int j = 0; j < RO; ++j)
              *reinterpret_cast<float2*>(smem + state0 + (yi ^ koff(j))) = make_float2(out[2 * j], out[2 * j + 1]);
          } else if constexpr (BETA) {  // outputs at o*NB + u
#pragma unroll
            for (int j = 0; j < RO; ++j) store_vec<ST>(cur + ST * ((o_lane + j) * NB + u), out + ST * j);
          } else {  // at R*u + o
            store_vec<RO * ST>(cur + ST * (R * u + o_lane), out);
          }
          tmax = max_with(tmax, no);
#pragma unroll
          for (int v = 0; v < NS; ++v) acc[v] += g[v];
        };
        if constexpr (CACHE || !EXACT || (CODE == CODE_TABLE && V == 1)) {
#pragma unroll
          for (int q = 0; q < UPT; ++q) unit(q);
        } else {
#pragma unroll 1
          for (int q = 0; q < UPT; ++q) unit(q);
        }
      }
      if constexpr (MARG) {
#pragma unroll
        for (int v = 0; v < NS; ++v) {
          const bool plain = GRAD ? v == 0 : v == V;  // sum dll, entropy: not scaled by kSigma
          const float s = wave_sum(acc[v]);
          if (lane == 0) apart[((st & 1) * nwaves + wave) * NS + v] = plain ? s : s * CT::kSigma;
        }
      }
      tmax = wave_max(tmax);
      if (lane == 0) wmax[(st & 1) * kMaxWaves + wave] = tmax;
      if constexpr (INPLACE) {
        rho += dt * KV;
        rho = rho >= nb ? rho - nb : rho < 0 ? rho + nb : rho;
      }
      __syncthreads();
    }
    if (MARG && wave == 0) step_out(t0 + dt * (n - 1), (n - 1) & 1);
    return off;
  };

  auto run = [&](auto exact) __attribute__((always_inline)) {
    using F = std::false_type;
    using Y = std::true_type;
    const int h = N / 2;
    float* mid = P.mid + (size_t)b * 2 * ST * NT;
    double* moff = P.moff + (size_t)b * (N + 2);
    if (P.mode == SOFT_FIRST) {
      const float init = role ? 0.0f : (float)KV;  // m~_{-1} = log2(R), n~_{N-1} = 0
      for (int j = tid; j < NT; j += nthr) {
        stv[ST * j] = init;
        if constexpr (GRAD) stv[2 * j + 1] = 0.0f;
      }
      __syncthreads();
      double off;
      if (role == 0) off = sweep(F{}, F{}, exact, 0, h, 0.0, (float)KV);
      else off = sweep(Y{}, F{}, exact, N - 1, N - h, 0.0, 0.0f);
      const float* fin = stv + (INPLACE ? 0 : ((role ? N - h : h) & 1) * ST * NT);
      for (int j = tid; j < ST * NT; j += nthr) mid[(size_t)role * ST * NT + j] = fin[j];
      const int lo = role ? h : 0, hi = role ? N : h;
      for (int i = lo + tid; i < hi; i += nthr) moff[i] = ovec[i];
      if (tid == 0) moff[N + role] = off;
      return;
    }
    // second halves: this side's vector and offset, the other side's offsets
    for (int j = tid; j < ST * NT; j += nthr) stv[j] = mid[(size_t)role * ST * NT + j];
    const int lo = role ? 0 : h, hi = role ? h : N;
    for (int i = lo + tid; i < hi; i += nthr) ovec[i] = moff[i];
    __syncthreads();
    const SoftMeet z = soft_meet<GRAD>(stv, mid + (size_t)(1 - role) * ST * NT, NT, moff[N] + moff[N + 1], gZ, wsum);
    logZ2 = z.logZ2;
    EFg = z.EFg;
    if (role == 0) sweep(F{}, Y{}, exact, h, N - h, moff[N], 0.0f);
    else sweep(Y{}, Y{}, exact, h - 1, h, moff[N + 1], 0.0f);
    if (!GRAD && role == 0 && tid == 0 && P.logZ) P.logZ[b] = (float)(logZ2 * kLn2);
  };
  if (Tb < kExactBelowT) {
    run(std::true_type{});
  } else {
    run(std::false_type{});
  }
}

}  // namespace bcjr
