// Soft forward and backward of the BCJR node for 4-bit steps (kV = 4: 16-input,
// 16-output butterflies), L = 8..16, every code.
//
// Same recursions, offsets, underflow handling and outputs as the other soft
// kernels (bcjr_fwd.hip, bcjr_bwd.hip; replaces the compute of
// src/bcjr/forward_backward.py:190-232 and src/bcjr/bcjr_monolithic.py:192-243).
//
// Work split.  LPB lanes of one wave share a butterfly: each reads all 16
// inputs and forms RO = 16 / LPB of the outputs, so no partial sum crosses
// lanes, and NB * LPB lanes work at every step (1,024 for L = 16 at LPB = 4;
// one lane per butterfly left a 1,024-state trellis 4 lanes of a wave).  The
// state vector (GRAD: of (m~, mu) pairs) is updated in place in LDS: at rotation
// rho_t = 4 (t - 1) mod nb a butterfly's outputs land on its inputs' elements,
// and because its lanes belong to one wave, their reads come before their
// writes without a barrier.
//
// Sweeps.  One body serves both directions: the cell of input i and output o is
// trellis state (p, c) = (i, o) in the alpha direction and (o, i) in the beta
// direction.  A sweep either stores its raw inputs to the sequence's slot at
// [t][u] (16 values, GRAD: pairs) or, as the marginal-forming sweep, reads there
// what the opposite sweep of the same step stored and accumulates the soft
// codeword (GRAD: the gradient sums).
//   whole sequence:  alpha over 0..N-1 stores, beta over N-1..0 forms marginals.
//   two halves (one workgroup each, two launches): first, alpha over 0..h-1 and
//     beta over N-1..h store and leave their state vectors in `mid`; then alpha
//     goes on over h..N-1 and beta over h-1..0, both forming marginals from what
//     the other one stored.  log Z (and E[F]) come from the two vectors where
//     they meet.  The steps in sequence are halved, which is what a batch too
//     small to fill the chip waits for; the launch boundary is the only
//     synchronisation.
//
// Codewords.  CODE_HYB_COL (L = 16, 3 <= Q <= 9) reads per-step LDS tables over
// the LUT's entries (below).  CODE_TABLE reads c(s) at p SP + c SC + u SU floats
// times V: with the transposed copy the host makes in the workspace (SC = NB, SU = 1)
// a wave's lanes, which hold consecutive u, read consecutive addresses; in the
// natural order (SC = 1, SU = 16) each lane reads a cache line of its own (500
// sequences of 128 steps at L = 16, V = 2: forward 4.87 against 23.2 ms, backward
// 5.06 against 17.3 ms).  The other codes hash each state, HYB through the LUT in
// LDS.
//
// Bounds.  Large batches: VALU issue (column walk, L = 16, T = 0.1: 11.8 VALU
// instructions per cell forward, 2.3 of them transcendental, and 20.5 backward),
// LDS latency and the tables' barrier; small ones: the latency of a step, N/2 of
// them each way.  Measured against one 256-thread workgroup per
// sequence with a butterfly per lane, at N = 128, HYB Q = 9: 8 sequences forward
// 1.61 -> 0.62 ms, backward 2.67 -> 0.85 ms; 4,096 sequences 15.4 -> 14.1-14.3 ms
// and 24.5 -> 24.0-24.6 ms; L = 12, 128 sequences (16 butterflies) 2.71 -> 0.21 ms and
// 3.62 -> 0.24 ms; a table at L = 16, 500 sequences 24.7 -> 4.9 and 24.0 -> 5.1 ms.
#pragma once

#include "bcjr_device.h"
#include "bcjr_kernels.h"
#include "bcjr_soft_common.h"

namespace bcjr {

// Threads of a workgroup and waves per SIMD the instance is built for.
template <int CODE, int LPB>
struct Soft16Shape {
  static constexpr bool kCol = CODE == CODE_HYB_COL;
  static constexpr int threads = LPB == 2 || LPB == 16 ? 512 : 1024;
  static constexpr int waves = !kCol ? (LPB == 4 ? 4 : 2) : 4;
};

template <bool GRAD, int CODE, int V, int LPB, bool ENT>
__global__ __launch_bounds__((Soft16Shape<CODE, LPB>::threads), (Soft16Shape<CODE, LPB>::waves)) void bcjr_soft16_kernel(Soft16Params P) {
  constexpr int KV = 4, R = 16, RO = R / LPB, UW = 64 / LPB;
  constexpr bool kCol = CODE == CODE_HYB_COL;
  constexpr int ST = GRAD ? 2 : 1;      // floats of a state element
  constexpr int GRP = 4;  // column-walk table entries in flight: more spill
  // Low temperature, column walk: a group's exponents are held from its maximum
  // to its sums (KEEP), or GRAD, which has no registers for them, formed again.
  constexpr bool KEEP = !GRAD;
  constexpr int NS = V + (GRAD || ENT ? 1 : 0);  // sums of a marginal-forming step
  using CT = CodeTraits<CODE>;
  static_assert(!(GRAD && ENT), "the entropy is an output of the forward");

  extern __shared__ __align__(16) unsigned char smem[];
  const int L = P.L, N = P.N, nb = L - KV;
  const int NT = 1 << nb, NB = NT >> KV;
  const int tid = threadIdx.x, nthr = blockDim.x, lane = tid & 63, wave = tid >> 6, nwaves = nthr >> 6;
  const int part = lane / UW;                     // which outputs of the butterfly
  const int uq = wave * UW + (lane & (UW - 1));   // butterfly slot of the lane
  const bool live = uq < NB;
  const int u = kCol ? (int)col_walk_unit((uint32_t)uq) : min(uq, NB - 1);

  // LDS: tables (column walk, 24 KiB) or LUT, state, offsets, per-wave entries.
  const uint32_t state0 = kCol ? 24576u : CODE == CODE_HYB ? 8u << P.Q : 0u;
  float* stv = reinterpret_cast<float*>(smem + state0);         // ST * NT
  double* ovec = reinterpret_cast<double*>(stv + ST * NT);       // N  offsets of the stored inputs
  float* wmax = reinterpret_cast<float*>(ovec + ((N + 1) & ~1));  // 2 * kMaxWaves
  float* apart = wmax + 2 * kMaxWaves;                           // max(2 * nwaves * NS, 2 * kMaxWaves + 4)
  const int napart = max(2 * nwaves * NS, 2 * kMaxWaves + 4);
  float* wsum = apart;                                           // 2 * kMaxWaves, outside the marginal sweeps
  int* bflag = reinterpret_cast<int*>(apart + 2 * kMaxWaves);    // input flag, at a sequence's start
  float* wbuf = apart + napart;                                  // N * V
  float* gbuf = wbuf + N * V;                                    // GRAD: N * V
  float* lut = reinterpret_cast<float*>(smem);

  if constexpr (CODE == CODE_HYB) {
    for (int i = tid; i < 2 << P.Q; i += nthr) lut[i] = P.table[i];
  }
  // Column walk: LUT entry tid (rows 0..7 of 64 columns), whose emissions this
  // thread forms each step for its rows tid >> 6 + {0, 8, 16} of the 24.  Rows 8
  // apart hold the same entry with the sign of its second component flipped.
  float2 ce = make_float2(0.0f, 0.0f);
  if constexpr (kCol) {
    const int ncol = 1 << (P.Q - 3), mask = (1 << P.Q) - 1, col = tid & 63;
    if (tid < 512 && col < ncol) {
      const int e = (col + ncol * (tid >> 6)) & mask;
      ce = make_float2(P.table[2 * e], P.table[2 * e + 1]);
    }
  }
  const uint32_t ANT = opaque_uniform(CT::A * (uint32_t)NT);
  // Byte address of element k of the lane's butterfly at rotation rho:
  // state0 + 4 ST S(rotr(u + k NB, rho)) (disjoint bits, so XOR).
  const Swizzle swz = P.swz;
  constexpr int LGB = GRAD ? 3 : 2;
  auto el_off = [&](uint32_t x, int rho) -> uint32_t {
    const uint32_t y = rotr_bits(x, rho, nb);
    return (kCol && !GRAD ? col_walk_state_el(y) : swizzle(y, swz)) << LGB;
  };

  for (long long b = P.mode == SOFT_WHOLE ? blockIdx.x : blockIdx.x >> 1; b < P.B;
       b += P.mode == SOFT_WHOLE ? gridDim.x : (P.B + 1)) {
    const size_t slot_id = P.mode == SOFT_WHOLE ? (size_t)blockIdx.x : (size_t)b;
    float* slot = P.ws + slot_id * P.slot_floats;
    const float Tb = P.T[P.t_per_seq ? b : 0];
    const float sk = sqrtf(kLog2e / Tb);
    const float ssk = CT::kSigma * sk;
    const float gZ = GRAD && P.g_logZ ? P.g_logZ[b] : 0.0f;
    const float twoT = 2.0f / Tb;
    const float* seqb = P.seq + (size_t)b * N * V;
    float* outb = P.out + (size_t)b * N * V;
    const int role = P.mode == SOFT_WHOLE ? 0 : (int)(blockIdx.x & 1);  // two halves: 0 alpha, 1 beta

    if (!soft_inputs<GRAD>(seqb, P.g_soft + (GRAD ? (size_t)b * N * V : 0), N * V, Tb, gZ, wbuf, gbuf, bflag)) {
      if (role == 0 && P.mode != SOFT_FIRST) soft_fill_nan<GRAD, ENT>(P, b, outb, N * V);
      __syncthreads();
      continue;
    }

    double logZ2 = 0.0;
    float EFg = 0.0f;  // E[F] - g_Z
    int k = 0;         // steps done: parity of the wmax and partial-sum buffers

    // Result of step t from the per-wave partials in buffer par (wave 0).
    auto step_out = [&](int t, int par) __attribute__((always_inline)) {
      soft_step_out<GRAD, ENT, V>(apart + par * nwaves * NS, nwaves, wbuf + t * V, twoT, outb + t * V,
                                  ENT ? P.H_out + (size_t)b * N + t : nullptr);
    };

    // One sweep over steps t0, t0 + dt, ... (n of them), dt = +1 (alpha) or -1
    // (beta), from the state vector in LDS with running offset `off`; first
    // says that the state is the trellis' free end.  Returns the offset after it.
    auto sweep = [&](auto beta_tag, auto marg_tag, auto exact_tag, int t0, int n, double off,
                     float O0) __attribute__((always_inline)) -> double {
      constexpr bool BETA = decltype(beta_tag)::value, MARG = decltype(marg_tag)::value;
      constexpr bool EXACT = decltype(exact_tag)::value;
      constexpr int dt = BETA ? -1 : 1;
      // The column walk's lanes take outputs in pairs p, p + 8 in the beta direction
      // (one table entry serves both): o(j) = (j mod H) + H part + 8 (j / H).
      // Elsewhere o(j) = j + RO part.
      constexpr int H = RO / 2;
      constexpr bool PAIRS = kCol && BETA;
      auto o_uni = [](int j) -> int { return PAIRS ? (j % (H > 0 ? H : 1)) + 8 * (j / (H > 0 ? H : 1)) : j; };
      const int o_lane = PAIRS ? H * part : RO * part;
      const int ul = opaque(u);

      // Column-walk bases, as byte offsets of 16-byte entries (entry row * 64 +
      // col): alpha, of the state 16u + o of the lane's outputs, for even and (LPB
      // = 4: 8 rows on for odd parts) odd p; beta, of the states 16u + c, moved on
      // by the lane's first output.
      constexpr int NCB = !kCol ? 1 : BETA ? R : LPB == 4 ? 2 * RO : RO;
      uint32_t cb[NCB];
      if constexpr (kCol) {
#pragma unroll
        for (int q = 0; q < NCB; ++q) {
          const int c = BETA ? q : (q % RO) + o_lane;
          const uint32_t e = hyb_col_base((uint32_t)(R * ul + c), P.Q) << 1;
          const uint32_t rows = BETA ? (uint32_t)(o_lane * (2 * c + 1)) : q >= RO ? 8u * (part & 1) : 0u;
          cb[q] = (e & 1023u) | ((e + (rows << 10)) & 0x3C00u);
        }
      }
      // Other codes: state s = sl + (uniform), hash or table base of the lane.
      const uint32_t sl = (uint32_t)(R * ul) + (BETA ? (uint32_t)o_lane << nb : (uint32_t)o_lane);
      const uint32_t tl =
          4u * V * ((uint32_t)ul * P.SU + (BETA ? (uint32_t)o_lane << nb : (uint32_t)o_lane * P.SC));

      int rho = (int)(((long long)KV * (t0 - 1) % nb + nb) % nb);
      for (int st = 0; st < n; ++st, ++k) {
        const int t = t0 + dt * st;
        // What the opposite sweep stored for the lane's outputs of this step (their
        // use is at the end of the first output, behind the tables' barrier).
        float po[MARG ? RO * ST : 1];
        if constexpr (MARG) {
          const float* src = slot + ((size_t)t * NB + ul) * (R * ST) + (size_t)o_lane * ST;
          if constexpr (PAIRS) {
            load_vec<H * ST>(src, po);
            load_vec<H * ST>(src + 8 * ST, po + H * ST);
          } else {
            load_vec<RO * ST>(src, po);
          }
        }
        float O = O0;
        if (st > 0) {
          O = block_max(wmax + ((k + 1) & 1) * kMaxWaves);
          if (MARG && wave == 0) step_out(t - dt, (k + 1) & 1);
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
        // Column-walk tables of the step: emissions E = -|d|^2 of LUT entries,
        // d = h ssk + nw (every wave has left the table this one replaces:
        // barrier at the end of each step).  Storing sweep: (E, E of 8 rows on),
        // forward in two tables by step parity, the next step's formed in this one;
        // GRAD (E, E', f, f'), f = sg . h.  Marginal sweep: (h, E, E').
        if constexpr (kCol) {
          auto emissions = [&](int tt, float& ep, float& em) {
            const float n0 = -wbuf[tt * V] * sk, n1 = -wbuf[tt * V + 1] * sk;
            const float d0 = fmaf(ce.x, ssk, n0), d1 = fmaf(ce.y, ssk, n1), d2 = fmaf(-ce.y, ssk, n1);
            const float e0 = fmaf(-d0, d0, 0.0f);
            ep = fmaf(-d1, d1, e0);
            em = fmaf(-d2, d2, e0);
          };
          auto build2 = [&](int tt) {
            float2* et = reinterpret_cast<float2*>(smem + 12288 * (tt & 1));
            if (tid < 512) {
              float ep, em;
              emissions(tt, ep, em);
              et[tid] = make_float2(ep, em);
              et[tid + 512] = make_float2(em, ep);
              et[tid + 1024] = make_float2(ep, em);
            }
          };
          if constexpr (!GRAD && !MARG) {
            if (st == 0) {
              build2(t);
              __syncthreads();
            }
            if (st + 1 < n) build2(t + dt);
          } else {
            if (tid < 512) {
              float4* et = reinterpret_cast<float4*>(smem);
              float ep, em;
              emissions(t, ep, em);
              if constexpr (MARG) {
                et[tid] = make_float4(ce.x, ce.y, ep, em);
                et[tid + 512] = make_float4(ce.x, -ce.y, em, ep);
                et[tid + 1024] = make_float4(ce.x, ce.y, ep, em);
              } else {
                const float f0 = sg[0] * ce.x, fp = fmaf(sg[V - 1], ce.y, f0), fm = fmaf(-sg[V - 1], ce.y, f0);
                et[tid] = make_float4(ep, em, fp, fm);
                et[tid + 512] = make_float4(em, ep, fm, fp);
                et[tid + 1024] = make_float4(ep, em, fp, fm);
              }
            }
            __syncthreads();
          }
        }
        const uint32_t tab = !GRAD && !MARG ? 12288u * (uint32_t)(t & 1) : 0u;

        // State elements: element k = 0..15 of the butterfly at state0 + (yu ^ koff(k)).
        const uint32_t yu = el_off((uint32_t)ul, rho);
        uint32_t K1 = el_off((uint32_t)NB, rho), K2 = el_off((uint32_t)NB << 1, rho),
                 K4 = el_off((uint32_t)NB << 2, rho), K8 = el_off((uint32_t)NB << 3, rho);
        auto koff = [&](int q) -> uint32_t {
          return ((q & 1) ? K1 : 0u) ^ ((q & 2) ? K2 : 0u) ^ ((q & 4) ? K4 : 0u) ^ ((q & 8) ? K8 : 0u);
        };
        const uint32_t yo = yu ^ el_off((uint32_t)(o_lane * NB), rho);  // of the lane's outputs
        float m[R], mu[GRAD ? R : 1];
#pragma unroll
        for (int q = 0; q < R; ++q) {
          if constexpr (GRAD) {
            const float2 v2 = *reinterpret_cast<const float2*>(smem + state0 + (yu ^ koff(q)));
            m[q] = v2.x;
            mu[q] = v2.y;
          } else {
            m[q] = *reinterpret_cast<const float*>(smem + state0 + (yu ^ koff(q)));
          }
        }
        // Codeword of output o(j), input i.  The lane's base and the strides are
        // opaque per step, so that the step's codewords (hashes, addresses) are not
        // all hoisted out of the step loop.
        const uint32_t base_s = kCol ? 0u : (uint32_t)opaque((int)(CODE == CODE_TABLE ? tl : CODE == CODE_HYB ? sl : CT::A * sl + CT::B));
        const uint32_t NT_s = kCol ? 0u : opaque_uniform((uint32_t)NT), SC_s = CODE == CODE_TABLE ? opaque_uniform(P.SC) : 1u;
        auto codeword_of = [&](int j, int i, float (&h)[V]) {
          const uint32_t p = (uint32_t)(BETA ? j : i), c = (uint32_t)(BETA ? i : j);
          if constexpr (CODE == CODE_TABLE) {
            const char* row = reinterpret_cast<const char*>(P.table + V * (p * NT_s + c * SC_s));
            const float* src = reinterpret_cast<const float*>(row + base_s);
            if constexpr (V == 2) {
              const float2 v = *reinterpret_cast<const float2*>(src);
              h[0] = v.x;
              h[1] = v.y;
            } else {
              h[0] = *src;
            }
          } else if constexpr (CODE == CODE_HYB) {
            code_hyb(base_s + p * NT_s + c, lut, P.Q, h[0], h[V - 1]);
          } else if constexpr (!kCol) {
            h[0] = raw_from_hash<CODE>(base_s + p * ANT + CT::A * c);
          }
        };
        float tmax = -INFINITY, acc[NS];
#pragma unroll
        for (int v = 0; v < NS; ++v) acc[v] = 0.0f;
        if (live) {
          if constexpr (!MARG) {  // the lane's share of the raw inputs: those of its output positions
            float own[RO * ST];
#pragma unroll
            for (int j = 0; j < RO; ++j) {
              if constexpr (GRAD) {
                const float2 v2 = *reinterpret_cast<const float2*>(smem + state0 + (yo ^ koff(o_uni(j))));
                own[2 * j] = v2.x;
                own[2 * j + 1] = v2.y;
              } else {
                own[j] = *reinterpret_cast<const float*>(smem + state0 + (yo ^ koff(o_uni(j))));
              }
            }
            float* dst = slot + ((size_t)t * NB + ul) * (R * ST) + (size_t)o_lane * ST;
            if constexpr (PAIRS) {
              store_vec<H * ST>(dst, own);
              store_vec<H * ST>(dst + 8 * ST, own + H * ST);
            } else {
              store_vec<RO * ST>(dst, own);
            }
          }
          const float M = max_of_inputs(m);
#pragma unroll
          for (int q = 0; q < R; ++q) m[q] -= M;
          const float oout = O - M;  // subtracted from an output's log sum
          const float kts = Kt + M;

          // Sums of one output: s = sum e; GRAD w = sum e z (z = f + mu_i);
          // marginal sweep: x[v] = sum e h_v, GRAD sum e (z + D) h_v; ENT y.
          struct Sums {
            float s, w, x[V], y;
          };
          // Adds a cell: e = 2^(y - shift), exponent y, path value z, codeword h.
          auto add = [&](Sums& a, bool first, float e, float y, float z, const float (&h)[V],
                         float Dp) __attribute__((always_inline)) {
            a.s = first ? e : a.s + e;
            if constexpr (GRAD) {
              const float ez = e * z;
              a.w = first ? ez : a.w + ez;
              if constexpr (MARG) {
                const float wgt = fmaf(e, Dp, ez);  // e (z + D)
#pragma unroll
                for (int v = 0; v < V; ++v) a.x[v] = first ? wgt * h[v] : fmaf(wgt, h[v], a.x[v]);
              }
            } else if constexpr (MARG) {
#pragma unroll
              for (int v = 0; v < V; ++v) a.x[v] = first ? e * h[v] : fmaf(e, h[v], a.x[v]);
              if constexpr (ENT) a.y = first ? e * y : fmaf(e, y, a.y);
            }
          };
          // Output o(j) from its sums: the new state element and, in the marginal
          // sweep, its terms of the step's sums with pms = (stored m~) + Kt + M.
          auto finish = [&](const Sums& a, float Mo, float pms, float Dp, float (&g)[NS], float& no, float& nuo) __attribute__((always_inline)) {
            no = flog2(a.s) + (Mo - oout);
            if constexpr (GRAD) nuo = a.w * frcp(a.s);
            if constexpr (MARG) {
              const float G = fexp2(pms + Mo);
              // GRAD: sum_s dll_t(s) is g_Z in exact arithmetic, but its computed
              // value cancels the common-mode rounding of (phi + psi - E[F]) in
              // the gradient, which grows with N: it is accumulated, not assumed.
              if constexpr (GRAD) g[0] = fmaf(G, fmaf(Dp, a.s, a.w), g[0]);
#pragma unroll
              for (int v = 0; v < V; ++v) g[v + (GRAD ? 1 : 0)] = fmaf(G, a.x[v], g[v + (GRAD ? 1 : 0)]);
              // log2 P of a cell is y + pms
              if constexpr (ENT) g[V] = fmaf(G, fmaf(pms, a.s, a.y), g[V]);
            }
          };
          auto put = [&](int j, float no, float nuo) __attribute__((always_inline)) {
            if constexpr (GRAD) {
              *reinterpret_cast<float2*>(smem + state0 + (yo ^ koff(o_uni(j)))) = make_float2(no, nuo);
            } else {
              *reinterpret_cast<float*>(smem + state0 + (yo ^ koff(o_uni(j)))) = no;
            }
            tmax = vmax_raw(tmax, no);
          };

          // Cell (j, i) of the column walk from its table entry: the entry at
          // hyb_pair_step(p, c) is p's, or with hyb_pair_far that of p + 8.
          struct Cell {
            float E, f, hx, hy;
          };
          auto col_cells = [&](int p, int c, uint32_t base, uint32_t twist, Cell& lo, Cell& hi) {  // of p mod 8, and 8 on
            const int p8 = p & 7;
            const bool far = hyb_pair_far(p8, c);
            if constexpr (MARG) {
              const float4 q = *reinterpret_cast<const float4*>(smem + ((base + hyb_pair_step(p8, c)) ^ twist));
              lo = {far ? q.w : q.z, 0.0f, q.x, far ? -q.y : q.y};
              hi = {far ? q.z : q.w, 0.0f, q.x, far ? q.y : -q.y};
            } else if constexpr (GRAD) {
              const float4 q = *reinterpret_cast<const float4*>(smem + ((base + hyb_pair_step(p8, c)) ^ twist));
              lo = {far ? q.y : q.x, far ? q.w : q.z, 0.0f, 0.0f};
              hi = {far ? q.x : q.y, far ? q.z : q.w, 0.0f, 0.0f};
            } else {
              const float2 q = *reinterpret_cast<const float2*>(
                  smem + (((base >> 1) + tab + (hyb_pair_step(p8, c) >> 1)) ^ twist));
              lo = {far ? q.y : q.x, 0.0f, 0.0f, 0.0f};
              hi = {far ? q.x : q.y, 0.0f, 0.0f, 0.0f};
            }
          };
          // GRAD: z of input i.  f = sg . h is formed first, as the storing sweep's table
          // has it, and rounded once onto mu, which is the larger: two roundings at mu's
          // size add 1.7 % to the gradient's error, the second operation 1.3 % to the time.
          auto path_value = [&](int i, const Cell& c) -> float {
            if constexpr (!GRAD) return 0.0f;
            else if constexpr (MARG && kCol) return mu[i] + fmaf(sg[V - 1], c.hy, sg[0] * c.hx);
            else return mu[i] + c.f;
          };
          // Output o(j)'s bases for even and odd inputs (alpha).
          auto col_bases = [&](int j, uint32_t& b0, uint32_t& b1) {
            b0 = hyb_col_base((uint32_t)(R * opaque(ul) + j + o_lane), P.Q) << 1;
            b1 = LPB == 4 ? (b0 & 1023u) | ((b0 + (8192u * (uint32_t)(part & 1))) & 0x3C00u) : b0;
          };
          auto col_cell = [&](int j, int i, uint32_t b0, uint32_t b1, uint32_t twist) -> Cell {  // dynamic j allowed
            const int p = BETA ? o_uni(j) : i, c = BETA ? i : j;
            Cell lo, hi;
            col_cells(p, c, BETA ? cb[i % NCB] : (i & 1) ? b1 : b0, twist, lo, hi);
            return (p & 8) ? hi : lo;
          };
          auto hv = [&](const Cell& c, float (&h)[V]) {
            h[0] = c.hx;
            if constexpr (V == 2) h[V - 1] = c.hy;
          };
          // Exponent and path value of a cell of a non-column code, accumulated onto
          // the inputs (one rounding per term, as in the other kernels).
          auto cell_yz = [&](int j, int i, float& y, float& z, float (&h)[V]) {
            codeword_of(j, i, h);
            y = m[i];
            if constexpr (GRAD) z = mu[i];
#pragma unroll
            for (int v = 0; v < V; ++v) {
              const float d = fmaf(h[v], ssk, nw[v]);
              y = fmaf(-d, d, y);
              if constexpr (GRAD) z = fmaf(sg[v], h[v], z);
            }
          };
          const float EF0 = MARG && GRAD ? EFg : 0.0f;

          // Output o(j) alone against its group maximum (the recompute of underflowed
          // groups, and low temperature on the other codes).  The column walk reads its entries
          // again after the maximum (twist hides that they are the same) rather than
          // keep 16 of them live.
          auto out_shifted = [&](int j, float pms, float Dp, float (&g)[NS]) __attribute__((always_inline)) {
            float y[R], Mo = 0.0f, h[V], z = 0.0f;
            uint32_t b0 = 0u, b1 = 0u;
            if constexpr (kCol) {
              if constexpr (!BETA) col_bases(j, b0, b1);
#pragma unroll
              for (int i = 0; i < R; ++i) {
                if (i % GRP == 0) __builtin_amdgcn_sched_barrier(0);
                y[i] = m[i] + col_cell(j, i, b0, b1, 0u).E;
              }
            } else {
#pragma unroll
              for (int i = 0; i < R; ++i) cell_yz(j, i, y[i], z, h);
            }
            Mo = max_of_inputs(y);
            Sums a;
            const uint32_t twist = kCol ? (uint32_t)opaque(0) : 0u;
#pragma unroll
            for (int i = 0; i < R; ++i) {
              if (kCol && i % GRP == 0) __builtin_amdgcn_sched_barrier(0);
              if constexpr (kCol) {
                Cell c = {0.0f, 0.0f, 0.0f, 0.0f};
                if constexpr (GRAD || MARG) c = col_cell(j, i, b0, b1, twist);
                hv(c, h);
                add(a, i == 0, fexp2(y[i] - Mo), y[i], path_value(i, c), h, Dp);
              } else {
                float yy;
                cell_yz(j, i, yy, z, h);
                add(a, i == 0, fexp2(y[i] - Mo), y[i], z, h, Dp);
              }
            }
            float no, nuo = 0.0f;
            finish(a, Mo, pms, Dp, g, no, nuo);
            put(j, no, nuo);
          };

          if constexpr (EXACT && !kCol) {
#pragma unroll
            for (int j = 0; j < RO; ++j) {
              __builtin_amdgcn_sched_barrier(0);
              out_shifted(j, MARG ? po[(MARG ? ST : 0) * j] + kts : 0.0f,
                          MARG && GRAD ? po[MARG && GRAD ? 2 * j + 1 : 0] - EF0 : 0.0f, acc);
            }
          } else {
            float smin = INFINITY, ga[NS];
#pragma unroll
            for (int v = 0; v < NS; ++v) ga[v] = 0.0f;
            auto pms_of = [&](int j) -> float { return MARG ? po[MARG ? ST * j : 0] + kts : 0.0f; };
            auto dp_of = [&](int j) -> float { return MARG && GRAD ? po[MARG && GRAD ? 2 * j + 1 : 0] - EF0 : 0.0f; };
            if constexpr (PAIRS) {
#pragma unroll
              for (int j = 0; j < H; ++j) {  // outputs o(j) and o(j) + 8
                __builtin_amdgcn_sched_barrier(0);
                Sums a0, a1;
                const float D0 = dp_of(j), D1 = dp_of(j + H);
                float M0 = 0.0f, M1 = 0.0f, x0[EXACT && KEEP ? R : 1], x1[EXACT && KEEP ? R : 1];
                const uint32_t twist = EXACT ? (uint32_t)opaque(0) : 0u;
                if constexpr (EXACT) {
#pragma unroll
                  for (int i = 0; i < R; ++i) {
                    if (i % GRP == 0) __builtin_amdgcn_sched_barrier(0);
                    Cell c0, c1;
                    col_cells(j, i, cb[i % NCB], 0u, c0, c1);
                    const float y0 = m[i] + c0.E, y1 = m[i] + c1.E;
                    if constexpr (KEEP) {
                      x0[i] = y0;
                      x1[i] = y1;
                    }
                    M0 = i ? vmax_raw(M0, y0) : y0;
                    M1 = i ? vmax_raw(M1, y1) : y1;
                  }
                }
#pragma unroll
                for (int i0 = 0; i0 < R; i0 += GRP) {
                  Cell c0[GRP], c1[GRP];
                  float y0[GRP], y1[GRP], e0[GRP], e1[GRP];
                  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                  for (int q = 0; q < GRP; ++q) {
                    const int i = i0 + q;
                    constexpr bool kept = EXACT && KEEP;
                    if constexpr (!kept || MARG) col_cells(j, i, cb[i % NCB], twist, c0[q], c1[q]);
                    y0[q] = kept ? x0[kept ? i : 0] : m[i] + c0[q].E;
                    y1[q] = kept ? x1[kept ? i : 0] : m[i] + c1[q].E;
                    e0[q] = fexp2(EXACT ? y0[q] - M0 : y0[q]);
                    e1[q] = fexp2(EXACT ? y1[q] - M1 : y1[q]);
                  }
                  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                  for (int q = 0; q < GRP; ++q) {
                    const int i = i0 + q;
                    float h0[V], h1[V], z0 = 0.0f, z1 = 0.0f;
                    hv(c0[q], h0);
                    hv(c1[q], h1);
                    if constexpr (GRAD && MARG) {
                      const float fx = sg[0] * c0[q].hx;
                      z0 = mu[i] + fmaf(sg[V - 1], c0[q].hy, fx);
                      z1 = mu[i] + fmaf(sg[V - 1], c1[q].hy, fx);
                    } else if constexpr (GRAD) {
                      z0 = mu[i] + c0[q].f;
                      z1 = mu[i] + c1[q].f;
                    }
                    add(a0, i == 0, e0[q], y0[q], z0, h0, D0);
                    add(a1, i == 0, e1[q], y1[q], z1, h1, D1);
                  }
                }
                smin = fminf(smin, fminf(a0.s, a1.s));
                float no, nuo = 0.0f;
                finish(a0, M0, pms_of(j), D0, ga, no, nuo);
                put(j, no, nuo);
                finish(a1, M1, pms_of(j + H), D1, ga, no, nuo);
                put(j + H, no, nuo);
              }
            } else {
#pragma unroll
              for (int j = 0; j < RO; ++j) {
                __builtin_amdgcn_sched_barrier(0);
                Sums a;
                const float D = dp_of(j);
                float Mo = 0.0f;
                if constexpr (kCol) {  // inputs p and p + 8 from one entry
                  const uint32_t twist = EXACT ? (uint32_t)opaque(0) : 0u;
                  float x[EXACT && KEEP ? R : 1];
                  if constexpr (EXACT) {
#pragma unroll
                    for (int i = 0; i < R / 2; ++i) {
                      if (i % GRP == 0) __builtin_amdgcn_sched_barrier(0);
                      Cell c0, c1;
                      col_cells(i, j, cb[(LPB == 4 && (i & 1) ? j + RO : j) % NCB], 0u, c0, c1);
                      const float y0 = m[i] + c0.E, y1 = m[i + R / 2] + c1.E;
                      Mo = i ? vmax3_raw(Mo, y0, y1) : vmax_raw(y0, y1);
                      if constexpr (KEEP) {
                        x[i] = y0;
                        x[i + R / 2] = y1;
                      }
                    }
                  }
#pragma unroll
                  for (int i0 = 0; i0 < R / 2; i0 += GRP) {
                    Cell c0[GRP], c1[GRP];
                    float y0[GRP], y1[GRP], e0[GRP], e1[GRP];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int q = 0; q < GRP; ++q) {
                      const int i = i0 + q;
                      constexpr bool kept = EXACT && KEEP;
                      if constexpr (!kept || MARG)
                        col_cells(i, j, cb[(LPB == 4 && (i & 1) ? j + RO : j) % NCB], twist, c0[q], c1[q]);
                      y0[q] = kept ? x[kept ? i : 0] : m[i] + c0[q].E;
                      y1[q] = kept ? x[kept ? i + 8 : 0] : m[i + 8] + c1[q].E;
                      e0[q] = fexp2(EXACT ? y0[q] - Mo : y0[q]);
                      e1[q] = fexp2(EXACT ? y1[q] - Mo : y1[q]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int q = 0; q < GRP; ++q) {
                      const int i = i0 + q;
                      float h0[V], h1[V];
                      hv(c0[q], h0);
                      hv(c1[q], h1);
                      add(a, i == 0, e0[q], y0[q], path_value(i, c0[q]), h0, D);
                      add(a, false, e1[q], y1[q], path_value(i + 8, c1[q]), h1, D);
                    }
                  }
                } else {
#pragma unroll
                  for (int i0 = 0; i0 < R; i0 += 8) {
                    float y[8], e[8], z[8], h[8][V];
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int q = 0; q < 8; ++q) {
                      z[q] = 0.0f;
                      cell_yz(j, i0 + q, y[q], z[q], h[q]);
                      e[q] = fexp2(y[q]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int q = 0; q < 8; ++q) add(a, i0 + q == 0, e[q], y[q], z[q], h[q], D);
                  }
                }
                smin = fminf(smin, a.s);
                float no, nuo = 0.0f;
                finish(a, Mo, pms_of(j), D, ga, no, nuo);
                put(j, no, nuo);
              }
            }
            if (!EXACT && smin < kUnderflow) {  // a group underflowed: redo the lane's outputs
              const float* src = slot + ((size_t)t * NB + ul) * (R * ST) + (size_t)o_lane * ST;
#pragma unroll
              for (int v = 0; v < NS; ++v) ga[v] = 0.0f;
#pragma unroll 1
              for (int j = 0; j < RO; ++j) {
                const int q = o_uni(j);
                out_shifted(j, MARG ? src[ST * q] + kts : 0.0f, MARG && GRAD ? src[ST * q + 1] - EF0 : 0.0f, ga);
              }
            }
#pragma unroll
            for (int v = 0; v < NS; ++v) acc[v] += ga[v];
          }
        }
        if constexpr (MARG) {
#pragma unroll
          for (int v = 0; v < NS; ++v) {
            const bool plain = GRAD ? v == 0 : v == V;  // sum dll, entropy: not scaled by kSigma
            const float s = wave_sum(acc[v]);
            if (lane == 0) apart[((k & 1) * nwaves + wave) * NS + v] = plain ? s : s * CT::kSigma;
          }
        }
        tmax = wave_max(tmax);
        if (lane == 0) wmax[(k & 1) * kMaxWaves + wave] = tmax;
        rho += dt * KV;
        rho = rho >= nb ? rho - nb : rho < 0 ? rho + nb : rho;
        __syncthreads();
      }
      if (MARG && wave == 0) step_out(t0 + dt * (n - 1), (k + 1) & 1);
      return off;
    };

    auto meet = [&](const float* own, const float* other, double CD) __attribute__((always_inline)) {
      const SoftMeet z = soft_meet<GRAD>(own, other, NT, CD, gZ, wsum);
      logZ2 = z.logZ2;
      EFg = z.EFg;
    };
    auto fill_state = [&](float value) __attribute__((always_inline)) {
      for (int j = tid; j < NT; j += nthr) {
        stv[ST * j] = value;
        if constexpr (GRAD) stv[2 * j + 1] = 0.0f;
      }
    };

    // Waves that do not exist never write their wmax entries.
    for (int i = tid; i < 2 * kMaxWaves; i += nthr) wmax[i] = -INFINITY;
    auto run = [&](auto exact) __attribute__((always_inline)) {
      using F = std::false_type;
      using Y = std::true_type;
      if (P.mode == SOFT_WHOLE) {
        fill_state((float)KV);  // m~_{-1} = log2(R)
        __syncthreads();
        const double C = sweep(F{}, F{}, exact, 0, N, 0.0, (float)KV);
        meet(stv, nullptr, C);
        fill_state(0.0f);
        __syncthreads();
        sweep(Y{}, Y{}, exact, N - 1, N, 0.0, 0.0f);
        return;
      }
      const int h = N / 2;
      float* mid = P.mid + (size_t)b * 2 * ST * NT;
      double* moff = P.moff + (size_t)b * (N + 2);
      if (P.mode == SOFT_FIRST) {
        fill_state(role ? 0.0f : (float)KV);
        __syncthreads();
        double off;
        if (role == 0) off = sweep(F{}, F{}, exact, 0, h, 0.0, (float)KV);
        else off = sweep(Y{}, F{}, exact, N - 1, N - h, 0.0, 0.0f);
        for (int j = tid; j < ST * NT; j += nthr) mid[(size_t)role * ST * NT + j] = stv[j];
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
      meet(stv, mid + (size_t)(1 - role) * ST * NT, moff[N] + moff[N + 1]);
      if (role == 0) sweep(F{}, Y{}, exact, h, N - h, moff[N], 0.0f);
      else sweep(Y{}, Y{}, exact, h - 1, h, moff[N + 1], 0.0f);
    };
    if (Tb < kExactBelowT) {
      run(std::true_type{});
    } else {
      run(std::false_type{});
    }
    if (!GRAD && P.mode != SOFT_FIRST && role == 0 && tid == 0 && P.logZ) P.logZ[b] = (float)(logZ2 * kLn2);
    __syncthreads();
  }
}

// The instances of one code, V and lanes per butterfly, by kind (bcjr_kernels.h).
#define BCJR_SOFT16_KINDS(CODE_, V_, LPB_)                                                                    \
  if (kind == 0) return reinterpret_cast<const void*>(&bcjr_soft16_kernel<false, CODE_, V_, LPB_, false>);    \
  if (kind == 1) return reinterpret_cast<const void*>(&bcjr_soft16_kernel<true, CODE_, V_, LPB_, false>);     \
  return reinterpret_cast<const void*>(&bcjr_soft16_kernel<false, CODE_, V_, LPB_, true>);

}  // namespace bcjr
