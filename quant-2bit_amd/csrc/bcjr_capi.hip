// C ABI of the engine (include/bcjr_hip.h): validation, launch geometry,
// workspace sizing and launches on the caller's stream.  No allocation, no host
// synchronisation, no exceptions across the boundary.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <functional>
#include <mutex>
#include <string>

#include "../../include/bcjr_hip.h"
#include "bcjr_device.h"
#include "bcjr_kernels.h"

namespace {

thread_local std::string g_last_error;

int fail(int status, const char* fmt, ...) __attribute__((format(printf, 2, 3)));
int fail(int status, const char* fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof(buf), fmt, ap);
  va_end(ap);
  g_last_error = buf;
  return status;
}

int hip_fail(hipError_t e, const char* what) {
  return fail(BCJR_EHIP, "%s: %s", what, hipGetErrorString(e));
}

struct DeviceInfo {
  bool valid = false;
  int num_cu = 0;
  size_t max_lds = 0;
};

std::mutex g_dev_mu;
DeviceInfo g_dev[64];

int device_info(DeviceInfo* out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  if (dev < 0 || dev >= 64) return fail(BCJR_EHIP, "device ordinal %d out of range", dev);
  std::lock_guard<std::mutex> lk(g_dev_mu);
  if (!g_dev[dev].valid) {
    int cu = 0, lds = 0;
    e = hipDeviceGetAttribute(&cu, hipDeviceAttributeMultiprocessorCount, dev);
    if (e != hipSuccess) return hip_fail(e, "hipDeviceGetAttribute(MultiprocessorCount)");
    e = hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, dev);
    if (e != hipSuccess) return hip_fail(e, "hipDeviceGetAttribute(MaxSharedMemoryPerBlock)");
    g_dev[dev].num_cu = cu;
    g_dev[dev].max_lds = (size_t)lds;
    g_dev[dev].valid = true;
  }
  *out = g_dev[dev];
  return BCJR_OK;
}

// Launch geometry of one operation for one problem.
struct Plan {
  int KV = 0, R = 0, NSUB = 0;
  int NT = 0, NB = 0, NU = 0;
  int nthr = 0, upt = 0;
  bool cache = false;
  bool fits = true;  // two-halves plans: there is a kernel and the LDS holds its state
  const void* fn = nullptr;
  size_t lds = 0;
  size_t slot_bytes = 0;
  int num_cu = 0;
  int max_blocks = 0;  // resident blocks on the device
  bcjr::Swizzle swz = {{31, 31, 31, 31}, {0, 0, 0, 0}};
};

int validate(const bcjr_problem* p) {
  if (!p) return fail(BCJR_EINVAL, "problem is NULL");
  if (p->V != 1 && p->V != 2) return fail(BCJR_EINVAL, "V=%d must be 1 or 2", p->V);
  if (p->k < 1) return fail(BCJR_EINVAL, "k=%d must be >= 1", p->k);
  const int KV = p->k * p->V;
  if (KV != 1 && KV != 2 && KV != 4)
    return fail(BCJR_EUNSUPPORTED, "k*V=%d: only 1, 2 or 4 bits per step are built", KV);
  if (p->L < 2 * KV || p->L > 16)
    return fail(BCJR_EUNSUPPORTED, "L=%d outside [%d, 16] for k*V=%d", p->L, 2 * KV, KV);
  if (KV == 1 && p->L > 11) return fail(BCJR_EUNSUPPORTED, "k*V=1 supports L <= 11 (got %d)", p->L);
  if (KV == 1 && p->code != BCJR_CODE_TABLE)
    return fail(BCJR_EUNSUPPORTED, "k*V=1 is built for the table code only (got code %d)", p->code);
  if (p->B < 0) return fail(BCJR_EINVAL, "B=%lld must be >= 0", (long long)p->B);
  if (p->N < 1 || p->N > 4096) return fail(BCJR_EINVAL, "N=%lld outside [1, 4096]", (long long)p->N);
  switch (p->code) {
    case BCJR_CODE_TABLE: break;
    case BCJR_CODE_1MAD:
    case BCJR_CODE_3INST:
      if (p->V != 1) return fail(BCJR_EINVAL, "1MAD/3INST codes are scalar (V=1), got V=%d", p->V);
      break;
    case BCJR_CODE_HYB:
      if (p->V != 2) return fail(BCJR_EINVAL, "HYB code is 2-D (V=2), got V=%d", p->V);
      if (p->Q < 1 || p->Q > 12) return fail(BCJR_EINVAL, "HYB Q=%d outside [1, 12]", p->Q);
      break;
    default: return fail(BCJR_EINVAL, "unknown code %d", p->code);
  }
  return BCJR_OK;
}

enum {
  OP_FWD = BCJR_OP_FORWARD,
  OP_BWD = BCJR_OP_BACKWARD,
  OP_VIT = BCJR_OP_VITERBI,
  OP_FWD_INTERNALS = 3,
  OP_FWD_ENTROPY = 4
};

// Bytes of one sequence slot of an operation's workspace (a validated problem):
// forward N * 2^(L-kV) floats (the raw alpha inputs of every step), backward
// twice that ((m~, mu) pairs), Viterbi one byte of backpointers per reduced
// state and step.  It depends on the problem only, so an undersized workspace
// is reported before any device query.
size_t slot_bytes_of(const bcjr_problem* p, int op) {
  const size_t NT = (size_t)1 << (p->L - p->k * p->V);
  size_t b = op == OP_BWD ? (size_t)p->N * 2 * NT * sizeof(float)
           : op == OP_VIT ? (size_t)p->N * NT
                          : (size_t)p->N * NT * sizeof(float);
  return (b + 255) & ~(size_t)255;
}

// Early argument checks shared by the launching entry points: the problem, then
// a workspace that holds at least one slot (BCJR_EWORKSPACE).
int check_ws(const bcjr_problem* p, int op, const void* ws, size_t ws_bytes) {
  int rc = validate(p);
  if (rc) return rc;
  if (p->B == 0) return BCJR_OK;
  if (!ws) return fail(BCJR_EINVAL, "ws must be non-NULL");
  const size_t slot = slot_bytes_of(p, op);
  if (ws_bytes < slot)
    return fail(BCJR_EWORKSPACE, "workspace of %zu bytes is smaller than one sequence slot (%zu bytes)",
                ws_bytes, slot);
  return BCJR_OK;
}

// Plans depend on (device, op, L, k, V, N, code, Q) only; they are cached so that
// steady-state calls (and calls made while a stream is being captured into a
// graph) do no attribute or occupancy queries.
struct PlanKey {
  int dev, op, L, k, V, code, Q, wide;
  long long N;
  bool operator==(const PlanKey& o) const {
    return dev == o.dev && op == o.op && L == o.L && k == o.k && V == o.V && code == o.code &&
           Q == o.Q && wide == o.wide && N == o.N;
  }
};
constexpr int kPlanCache = 128;  // a problem has up to two plans per operation
std::mutex g_plan_mu;
PlanKey g_plan_keys[kPlanCache];
Plan g_plans[kPlanCache];
int g_plan_count = 0, g_plan_next = 0;

int make_plan_uncached(const bcjr_problem* p, int op, bool wide, const DeviceInfo& di, Plan* pl);

// wide: the launch shape of a batch too small to fill the chip, where the
// operation has one of its own (make_soft16_plan), else the same plan.
int make_plan(const bcjr_problem* p, int op, Plan* pl, bool wide = false) {
  int rc = validate(p);
  if (rc) return rc;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  const PlanKey key = {dev, op, p->L, p->k, p->V, p->code, p->code == BCJR_CODE_HYB ? p->Q : 0, wide ? 1 : 0,
                       (long long)p->N};
  {
    std::lock_guard<std::mutex> lk(g_plan_mu);
    for (int i = 0; i < g_plan_count; ++i)
      if (g_plan_keys[i] == key) {
        *pl = g_plans[i];
        return BCJR_OK;
      }
  }
  DeviceInfo di;
  rc = device_info(&di);
  if (rc) return rc;
  rc = make_plan_uncached(p, op, wide, di, pl);
  if (rc) return rc;
  std::lock_guard<std::mutex> lk(g_plan_mu);
  const int slot = g_plan_count < kPlanCache ? g_plan_count++ : (g_plan_next++ % kPlanCache);
  g_plan_keys[slot] = key;
  g_plans[slot] = *pl;
  return BCJR_OK;
}

// LDS bank conflicts of an in-place layout: element S(rotr(k*NB + u, rho)) holds
// slot k of butterfly u.  Priced for 8-byte (m~, mu) pairs read and written by one
// lane per butterfly, the backward of kV <= 2.  Measured on gfx950: a 64-bit LDS read
// serves each 32-lane half of a wave from 32 eight-byte banks (conflict-free
// when the half's elements differ mod 32); a 64-bit write serves 16 lanes at a
// time from 32 four-byte banks (conflict-free when each quarter's elements
// differ mod 16).  One wave of butterflies (u = 0..63) suffices: higher bits of
// u XOR the same constant into every element of the wave.  The kV = 4 kernels take
// the same layouts: their lanes that share a butterfly read the same words, so a wave
// touches 4 or 16 butterflies of those 64; the forward's floats are not priced.
// Returns the extra passes summed over the rotations a sweep reaches (multiples of
// gcd(kV, nb)) and the slots.
int swizzle_cost(int L, int KV, const bcjr::Swizzle& s) {
  const int nb = L - KV, NB = 1 << (nb - KV), R = 1 << KV;
  const int lanes = std::min(NB, 64);
  const uint32_t mask = (1u << nb) - 1u;
  int g = KV, h = nb;
  while (h) {
    const int r = g % h;
    g = h;
    h = r;
  }
  int cost = 0;
  uint32_t el[64];
  for (int rho = 0; rho < nb; rho += g)
    for (int k = 0; k < R; ++k) {
      for (int l = 0; l < lanes; ++l) {
        const uint32_t j = (uint32_t)(k * NB + l);
        const uint32_t x = ((j | (j << nb)) >> rho) & mask;
        uint32_t e = x;
        for (int f = 0; f < 4; ++f) e ^= (x >> s.a[f]) & s.m[f];
        el[l] = e;
      }
      for (int group = 16; group <= 32; group *= 2)  // writes: 16 mod 16; reads: 32 mod 32
        for (int l0 = 0; l0 < lanes; l0 += group) {
          int cnt[32] = {0}, worst = 0;
          for (int l = l0; l < std::min(lanes, l0 + group); ++l) worst = std::max(worst, ++cnt[el[l] % group]);
          cost += worst - 1;
        }
    }
  return cost;
}

// Cheapest swizzle: up to four fields of 4 or 5 bits at shifts >= their width,
// taken in order of increasing count and kept only when strictly better; the
// search stops at the first conflict-free layout.
bcjr::Swizzle pick_swizzle(int L, int KV) {
  const int nb = L - KV;
  bcjr::Swizzle best = {{31, 31, 31, 31}, {0, 0, 0, 0}};
  int best_cost = swizzle_cost(L, KV, best);
  for (int nf = 1; nf <= 4 && best_cost > 0; ++nf) {
    int sh[4];
    // shifts sh[0] < ... < sh[nf-1] in [4, nb), widths from the bits of wbits
    std::function<void(int, int)> rec = [&](int f, int lo) {
      if (best_cost == 0) return;
      if (f == nf) {
        for (int wbits = 0; wbits < (1 << nf) && best_cost > 0; ++wbits) {
          bcjr::Swizzle s = {{31, 31, 31, 31}, {0, 0, 0, 0}};
          bool ok = true;
          for (int i = 0; i < nf; ++i) {
            const int w = 4 + ((wbits >> i) & 1);
            if (sh[i] < w) ok = false;
            s.a[i] = sh[i];
            s.m[i] = (1u << w) - 1u;
          }
          if (!ok) continue;
          const int cost = swizzle_cost(L, KV, s);
          if (cost < best_cost) {
            best_cost = cost;
            best = s;
          }
        }
        return;
      }
      for (int a = lo; a < nb; ++a) {
        sh[f] = a;
        rec(f + 1, a + 1);
      }
    };
    rec(0, 4);
  }
  return best;
}

// The search takes up to 55 ms (L = 15): once per (L, kV).
bcjr::Swizzle swizzle_of(int L, int KV) {
  static std::mutex mu;
  static bool have[17][5];
  static bcjr::Swizzle memo[17][5];
  std::lock_guard<std::mutex> lk(mu);
  if (!have[L][KV]) {
    memo[L][KV] = pick_swizzle(L, KV);
    have[L][KV] = true;
  }
  return memo[L][KV];
}

// State layout of the column walk's (m~, mu) pairs (L = 16, kV = 4), whose lane
// slot q holds butterfly col_walk_unit(q) rather than q: with this swizzle the 64-bit
// reads of 32 consecutive slots and the 64-bit writes of 16 of S(rotr(k*NB + u, rho))
// fall in distinct banks for all 256 slots, the 16 elements and the rotations 0, 4, 8
// (the search above assumes u = q).  The column walk's forward lays its floats out
// by col_walk_state_el.
constexpr bcjr::Swizzle kColWalkSwizzle = {{4, 6, 8, 31}, {3u, 31u, 15u, 0u}};

// Opts the plan's kernel in to its LDS and finds how many blocks the device holds.
int finish_plan(const bcjr_problem* p, const DeviceInfo& di, Plan* pl) {
  if (pl->lds > di.max_lds)
    return fail(BCJR_EUNSUPPORTED, "needs %zu bytes of LDS per workgroup (device limit %zu); reduce N=%lld",
                pl->lds, di.max_lds, (long long)p->N);
  hipError_t e = hipFuncSetAttribute(pl->fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)pl->lds);
  if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(MaxDynamicSharedMemorySize)");
  int per_cu = 0;
  e = hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, pl->fn, pl->nthr, pl->lds);
  if (e != hipSuccess) return hip_fail(e, "hipOccupancyMaxActiveBlocksPerMultiprocessor");
  if (per_cu < 1)
    return fail(BCJR_EUNSUPPORTED, "kernel cannot be resident (%d threads, %zu B LDS)", pl->nthr, pl->lds);
  pl->num_cu = di.num_cu;
  pl->max_blocks = per_cu * di.num_cu;
  return BCJR_OK;
}

// The soft kernels of 4-bit steps (bcjr_soft16.h).  Lanes per butterfly: the
// column walk 2 (512 threads, two workgroups per CU), or 4 (1,024 threads) where
// the workgroup has its CU to itself anyway (wide); other codes 4, and 16 for the
// NB <= 32 butterflies of L <= 13, which 4 would leave on one or two waves.
int make_soft16_plan(const bcjr_problem* p, int op, bool wide, const DeviceInfo& di, Plan* pl) {
  const int code = bcjr::soft_kernel_code(p->code, p->L, 4, p->Q);
  const int kind = op == OP_BWD ? 1 : op == OP_FWD_ENTROPY ? 2 : 0;
  const int lpb = code == bcjr::CODE_HYB_COL ? (wide ? 4 : 2) : p->L <= 13 ? 16 : 4;
  pl->KV = 4;
  pl->R = 16;
  pl->NSUB = 1;
  pl->NT = 1 << (p->L - 4);
  pl->NB = pl->NT >> 4;
  pl->NU = pl->NB;
  pl->upt = 1;
  const int per_wave = 64 / lpb;  // butterflies of a wave
  pl->nthr = (pl->NB + per_wave - 1) / per_wave * 64;
  pl->fn = bcjr::soft16_kernel_ptr(kind, p->V, code, lpb);
  pl->lds = bcjr::soft16_lds_bytes(p->L, p->V, (int)p->N, pl->nthr / 64, code, p->Q, kind);
  pl->swz = code == bcjr::CODE_HYB_COL ? kColWalkSwizzle : swizzle_of(p->L, 4);
  pl->slot_bytes = slot_bytes_of(p, op == OP_BWD ? OP_BWD : OP_FWD);
  return finish_plan(p, di, pl);
}

// The two-halves soft kernels of kV <= 2 (bcjr_halves.h), up to 1,024 threads:
// kV = 2 whole butterflies from L = 12 on, else a lane per output (N = 256, forward
// and backward, whole butterflies against a lane per output: L = 13, 128 sequences
// 0.28 against 0.37 and 0.41 against 0.49 ms; L = 12 0.24 against 0.27 and 0.32
// against 0.32 ms; L = 10, 64 sequences 0.21 against 0.18 and 0.26 against 0.21 ms).
struct HalvesShape {
  int lpb, upt, nthr;
};

HalvesShape halves_shape(const bcjr_problem* p) {
  const int KV = p->k * p->V, NB = 1 << (p->L - 2 * KV), lpb = KV == 2 && p->L >= 12 ? 1 : 1 << KV;
  const int upt = std::max(1, NB * lpb / 1024);
  return {lpb, upt, std::max(64, NB * lpb / upt)};
}

int make_halves_plan(const bcjr_problem* p, int op, const DeviceInfo& di, Plan* pl) {
  const int KV = p->k * p->V, kind = op == OP_BWD ? 1 : op == OP_FWD_ENTROPY ? 2 : 0;
  const HalvesShape sh = halves_shape(p);
  const bool in_place = bcjr::halves_in_place(op == OP_BWD, sh.upt, sh.lpb);
  pl->KV = KV;
  pl->R = 1 << KV;
  pl->NSUB = 1;
  pl->NT = 1 << (p->L - KV);
  pl->NB = pl->NT >> KV;
  pl->NU = pl->NB;
  pl->upt = sh.upt;
  pl->nthr = sh.nthr;
  pl->fn = bcjr::halves_kernel_ptr(kind, KV, p->V, p->code, sh.upt, sh.lpb);
  pl->lds = bcjr::halves_lds_bytes(p->L, KV, p->V, (int)p->N, pl->nthr / 64, p->code, p->Q, kind, in_place);
  pl->fits = pl->fn && pl->lds <= di.max_lds;  // long N (or large Q): a plan like any other, kept as "no"
  if (!pl->fits) return BCJR_OK;
  if (in_place) pl->swz = swizzle_of(p->L, KV);
  pl->slot_bytes = slot_bytes_of(p, op == OP_BWD ? OP_BWD : OP_FWD);
  return finish_plan(p, di, pl);
}

int make_plan_uncached(const bcjr_problem* p, int op, bool wide, const DeviceInfo& di, Plan* pl) {
  const int KV = p->k * p->V, R = 1 << KV, RO = R < 4 ? R : 4;
  if (KV == 4 && (op == OP_FWD || op == OP_BWD || op == OP_FWD_ENTROPY)) return make_soft16_plan(p, op, wide, di, pl);
  if (wide && op != OP_VIT) return make_halves_plan(p, op, di, pl);
  if (op == OP_FWD_ENTROPY) op = OP_FWD_INTERNALS;
  pl->KV = KV;
  pl->R = R;
  pl->NSUB = R / RO;
  pl->NT = 1 << (p->L - KV);
  pl->NB = pl->NT >> KV;
  if (op != OP_VIT) pl->NSUB = 1;  // the soft kernels take whole butterflies per unit
  pl->NU = pl->NB * pl->NSUB;
  const int max_thr = 512;
  int nthr = ((pl->NU + 63) / 64) * 64;
  nthr = std::min(nthr, max_thr);
  const int upt = (pl->NU + nthr - 1) / nthr;
  if (upt != 1 && upt != 2 && upt != 4 && upt != 8)
    return fail(BCJR_EUNSUPPORTED, "no launch shape for L=%d k*V=%d (units/thread %d)", p->L, KV, upt);
  pl->nthr = nthr;
  pl->upt = upt;
  const int nwaves = nthr / 64;
  const int N = (int)p->N;
  const int kcode = bcjr::soft_kernel_code(p->code, p->L, KV, p->Q);
  if (op == OP_FWD || op == OP_FWD_INTERNALS || op == OP_VIT) {
    const bool fwd = (op != OP_VIT);
    // The Viterbi kernel caches all of a thread's codewords in VGPRs up to 128
    // of them; the soft forward's cache is fixed per instance
    // (fwd_cached_units).
    pl->cache = !fwd && (pl->NSUB == 1) && (upt * R * R * p->V <= 128);
    int vcode = p->code;  // the Viterbi instance's code
    pl->fn = fwd ? bcjr::fwd_kernel_ptr(KV, p->V, kcode, upt, op == OP_FWD_INTERNALS)
                 : bcjr::vit_kernel_ptr(KV, p->V, p->code, upt, pl->cache, false);
    if (!fwd && pl->NU >= 1024) {
      // 1024 threads (four waves per SIMD instead of two) when an instance
      // exists: codewords cached within 64 VGPRs, or none cached (kV = 4).
      const int upt_w = pl->NU / 1024;
      const bool cache_w = (pl->NSUB == 1) && (upt_w * R * R * p->V <= 64);
      const int wcode = cache_w ? p->code : kcode;
      const void* fn_w = bcjr::vit_kernel_ptr(KV, p->V, wcode, upt_w, cache_w, true);
      // ... and its LDS fits (the HYB LUT copies of the uncached instances do
      // not beside a 2^14-state cost vector: k = 1, V = 2 at L = 16).
      if (fn_w && bcjr::vit_lds_bytes(p->L, KV, p->V, N, 16, wcode, p->Q, !cache_w) > di.max_lds) fn_w = nullptr;
      if (fn_w) {
        vcode = wcode;
        pl->fn = fn_w;
        pl->cache = cache_w;
        pl->nthr = nthr = 1024;
        pl->upt = upt_w;
      }
    }
    pl->lds = fwd ? bcjr::fwd_lds_bytes(p->L, KV, p->V, N, nwaves, kcode, p->Q)
                  : bcjr::vit_lds_bytes(p->L, KV, p->V, N, nwaves, vcode, p->Q,
                                        !pl->cache && pl->nthr == 1024);
    if (op == OP_FWD && KV == 2 && p->V == 1 && p->L >= 14 && p->code <= BCJR_CODE_3INST) {
      // Four waves per SIMD: 1024 threads, every codeword in VGPRs (bcjr_fwd4.hip).
      // Kept only where its larger LDS (N doubles and floats beside the state)
      // still fits; otherwise the 512-thread plan stands (at L = 16 it holds
      // N = 2704, the 1024-thread kernel N = 2702).
      const int upt4 = 1 << (p->L - 14);
      const void* fn4 = bcjr::fwd4_kernel_ptr(p->code, upt4);
      if (fn4 && bcjr::fwd4_lds_bytes(p->L, N) <= di.max_lds) {
        pl->fn = fn4;
        pl->nthr = nthr = 1024;
        pl->upt = upt4;
        pl->lds = bcjr::fwd4_lds_bytes(p->L, N);
      }
    }
    pl->slot_bytes = slot_bytes_of(p, fwd ? OP_FWD : OP_VIT);
  } else {
    pl->cache = false;
    pl->swz = swizzle_of(p->L, KV);
    pl->fn = bcjr::bwd_kernel_ptr(KV, p->V, kcode, upt);
    pl->lds = bcjr::bwd_lds_bytes(p->L, KV, p->V, N, nwaves, kcode, p->Q);
    pl->slot_bytes = slot_bytes_of(p, OP_BWD);
  }
  if (!pl->fn)
    return fail(BCJR_EUNSUPPORTED, "no kernel built for L=%d k=%d V=%d code=%d (units/thread %d)",
                p->L, p->k, p->V, p->code, upt);
  return finish_plan(p, di, pl);
}

int launch(const Plan& pl, long long B, size_t ws_bytes, void* params, hipStream_t stream) {
  if (B == 0) return BCJR_OK;
  long long slots = (long long)(ws_bytes / pl.slot_bytes);
  if (slots < 1)
    return fail(BCJR_EWORKSPACE, "workspace of %zu bytes is smaller than one sequence slot (%zu bytes)",
                ws_bytes, pl.slot_bytes);
  const long long grid = std::min<long long>(std::min<long long>(B, pl.max_blocks), slots);
  void* args[] = {params};
  hipError_t e = hipLaunchKernel(pl.fn, dim3((unsigned)grid), dim3((unsigned)pl.nthr), args, pl.lds, stream);
  if (e != hipSuccess) return hip_fail(e, "hipLaunchKernel");
  e = hipGetLastError();
  if (e != hipSuccess) return hip_fail(e, "kernel launch");
  return BCJR_OK;
}

size_t round256(size_t b) { return (b + 255) & ~(size_t)255; }

// Bytes the two-halves launches keep per sequence: its slot, the two state
// vectors where the sweeps meet, and the offsets of every step.
size_t halves_bytes(const bcjr_problem* p, int op) {
  const size_t NT = (size_t)1 << (p->L - p->k * p->V), st = op == OP_BWD ? 2 : 1;
  return slot_bytes_of(p, op == OP_BWD ? OP_BWD : OP_FWD) + round256(2 * st * NT * sizeof(float)) +
         round256(((size_t)p->N + 2) * sizeof(double));
}

// Fewest steps that take two halves: below, the second launch costs more than the
// steps it saves (one call among others, one launch -> two halves: 8 steps at L <= 12
// 15-17 -> 18-20 us, their k V = 2 backward 21-24 -> 18-25; 16 steps 19-38 -> 18-39;
// L = 14 and 16, 128 sequences, 4 steps 21-80 -> 25-85, 8 steps 33-135 -> 31-122; kV =
// 4, L = 8, 4 steps 15-16 -> 18-19, 8 steps 21-25 -> 19-20; L >= 12, 2 steps 15-79 ->
// 18-100, 4 steps 20-132 -> 19-127; L = 16, k = 1, V = 2, 4 steps 78-118 -> 53-89).
long long halves_min_steps(const bcjr_problem* p, int op) {
  const int KV = p->k * p->V;
  if (KV == 4) return p->L >= 12 ? 4 : 8;
  if (p->L == 16 && (p->V == 2 || op == OP_FWD_ENTROPY)) return 4;
  return p->L >= 14 || (KV == 2 && op == OP_BWD) ? 8 : 16;
}

// Largest load of the kV <= 2 halves, in quarters of a workgroup per CU.  A lane per
// output forms a butterfly's inputs once per output, so where one launch fills whole
// waves (kV = 1 from L = 8, kV = 2 at L = 10) or a table of two components is read
// that often, the halves lose their lead at 32 waves per CU (forward, N = 96, one
// launch -> two halves: kV = 1, L = 11, 128 sequences 1.46 times as fast, 192 0.80;
// L = 10, 768 sequences 1.18, 1,024 0.82; L = 9, whose waves one launch half fills,
// 2,048 1.05).  Whole butterflies of two components, whose codewords no register
// holds: up to 12 waves per CU, or the one workgroup of L >= 13 (HYB, L = 12, 384
// sequences 1.16, 512 0.96; L = 13, 128 1.41, 192 0.93; a table at L = 13 1.11 and
// 0.75), and a table's plain forward a little less (T = 0.06: L = 14, 96 sequences
// 0.99, 128 0.91; L = 12, 128 1.16, 192 0.97; L = 16, 128 1.49).
int halves_quarters_per_cu(const bcjr_problem* p, int op, const HalvesShape& sh) {
  const int waves = sh.nthr / 64;
  const bool table2 = p->V == 2 && p->code == BCJR_CODE_TABLE;
  if (sh.lpb > 1) {
    const bool early = p->k * p->V == 1 || p->L == 10 || (table2 && op != OP_BWD);
    return 4 * ((waves > 1 && early ? 24 : 32) / waves);
  }
  if (p->V == 1) return 4 * (32 / waves);
  if (table2 && op == OP_FWD) return p->L == 12 || p->L == 16 ? 4 : 3;
  return 4 * std::max(1, 12 / waves);
}

// Whether a soft call runs its sequences in two halves each (bcjr_soft16.h,
// bcjr_halves.h), and on which plan: when twice as many workgroups still all fit
// at once, so that the steps in sequence are halved and no sequence waits for
// another, and the two limits above say that it pays.  A sequence's last bits
// therefore depend on the batch it is in: the two forms sum in other orders.  Every
// workspace of the queried size, and every shorter one that takes several rounds,
// gives the same bits; one too short for that (launch_halves) runs in one launch,
// with the bits of a large batch.  kV = 4: the plan of one launch, or, column walk,
// one workgroup of twice the threads per CU where that is all there is.
// Measured, forward and backward, one launch -> two halves, N = 128: column walk
// 8 sequences 1.17 -> 0.62 and 1.83 -> 0.85 ms (narrow workgroup 0.70 and 1.01),
// 128 sequences 1.27 -> 0.70 and 1.95 -> 0.98 ms (0.79 and 1.11), 256 sequences on
// the narrow one 1.28 -> 1.07 and 1.97 -> 1.61 ms; a table, 128 sequences 2.44 ->
// 1.15 and 2.51 -> 1.43 ms; L = 12, 256 sequences 0.38 -> 0.26 and 0.42 -> 0.29 ms.
// kV = 4 gains up to all that is resident (L = 8, 10, 12, 14: 2,048, 1,536, 512, 512
// sequences 1.12, 1.39, 1.19, 1.17 times as fast).
int halves_plan(const bcjr_problem* p, int op, const Plan& pl, Plan* out, bool* halves) {
  *halves = false;
  if (p->N < halves_min_steps(p, op)) return BCJR_OK;
  if (pl.KV == 4) {
    *halves = 2 * p->B <= pl.max_blocks;
    *out = pl;
    if (*halves && bcjr::soft_kernel_code(p->code, p->L, 4, p->Q) == bcjr::CODE_HYB_COL && 2 * p->B <= pl.num_cu)
      return make_plan(p, op, out, true);
    return BCJR_OK;
  }
  // (no plan is made for a batch beyond the limit; of pl only the CU count counts)
  if (8 * p->B > (long long)pl.num_cu * halves_quarters_per_cu(p, op, halves_shape(p))) return BCJR_OK;
  const int rc = make_plan(p, op, out, true);
  if (rc || !out->fits) return rc;  // the LDS does not hold this N (or Q): one launch
  *halves = 2 * p->B <= out->max_blocks;
  return BCJR_OK;
}

// Bytes of the transposed codebook copy of the kV = 4 table kernels (0: none).
size_t table16_bytes(const bcjr_problem* p) {
  return p->k * p->V == 4 && p->code == BCJR_CODE_TABLE ? round256(((size_t)p->V << p->L) * sizeof(float)) : 0;
}

// A Viterbi launch; kV = 4 tables first get their transposed copy, as above.
int launch_viterbi(const bcjr_problem* p, bcjr::VitParams P, void* ws, size_t ws_bytes, hipStream_t stream) {
  Plan pl;
  const int rc = make_plan(p, OP_VIT, &pl);
  if (rc) return rc;
  char* w = static_cast<char*>(ws);
  const size_t tb = table16_bytes(p);
  P.tab16 = P.table;
  P.SC = 1;
  P.SU = 16;
  if (tb && ws_bytes >= tb + pl.slot_bytes) {
    hipError_t e = bcjr::launch_transpose16(P.table, reinterpret_cast<float*>(w), p->L, p->V, stream);
    if (e != hipSuccess) return hip_fail(e, "codebook transpose launch");
    P.tab16 = reinterpret_cast<const float*>(w);
    P.SC = (uint32_t)pl.NB;
    P.SU = 1;
    w += tb;
    ws_bytes -= tb;
  }
  P.ws = reinterpret_cast<uint8_t*>(w);
  return launch(pl, p->B, ws_bytes, &P, stream);
}

// The two launches of a batch in two halves; a workspace that does not hold all of
// it takes equal rounds.  *done = false where one launch (plan `one`) is the better
// use of a short workspace: N steps in series a round against 2 N for as many
// sequences as it has slots for, or no room for one sequence's halves.
int launch_halves(const bcjr_problem* p, int op, const Plan& one, const Plan& pl, bcjr::Soft16Params P, char* ws,
                  size_t ws_bytes, hipStream_t stream, bool* done) {
  const long long fit = (long long)(ws_bytes / halves_bytes(p, op));
  *done = false;
  if (fit < 1) return BCJR_OK;
  const long long flight = std::min<long long>(one.max_blocks, (long long)(ws_bytes / one.slot_bytes));
  const long long rounds = (p->B + fit - 1) / fit;
  if (rounds >= 2 * ((p->B + flight - 1) / flight)) return BCJR_OK;
  const long long round = (p->B + rounds - 1) / rounds;
  *done = true;
  const size_t st = op == OP_BWD ? 2 : 1, row = (size_t)p->N * p->V;
  char* mid = ws + (size_t)round * pl.slot_bytes;
  P.ws = reinterpret_cast<float*>(ws);
  P.mid = reinterpret_cast<float*>(mid);
  P.moff = reinterpret_cast<double*>(mid + (size_t)round * round256(2 * st * pl.NT * sizeof(float)));
  P.swz = pl.swz;
  for (long long b0 = 0; b0 < p->B; b0 += round) {
    bcjr::Soft16Params H = P;
    H.B = std::min<long long>(round, p->B - b0);
    H.seq += b0 * row;
    H.out += b0 * row;
    if (P.t_per_seq) H.T += b0;
    if (H.logZ) H.logZ += b0;
    if (H.H_out) H.H_out += b0 * p->N;
    if (H.g_soft) H.g_soft += b0 * row;
    if (H.g_logZ) H.g_logZ += b0;
    for (int mode : {(int)bcjr::SOFT_FIRST, (int)bcjr::SOFT_SECOND}) {
      H.mode = mode;
      void* args[] = {&H};
      hipError_t e = hipLaunchKernel(pl.fn, dim3((unsigned)(2 * H.B)), dim3((unsigned)pl.nthr), args, pl.lds, stream);
      if (e != hipSuccess) return hip_fail(e, "hipLaunchKernel");
      e = hipGetLastError();
      if (e != hipSuccess) return hip_fail(e, "kernel launch");
    }
  }
  return BCJR_OK;
}

// One soft call on the kV = 4 kernels, or in two halves: the table's transposed
// copy (kV = 4, when the workspace has room for it beside one slot; else the
// kernels read the table as it is), then the batch in two halves or in one launch.
// *done = false: the call is one for the whole-sequence kernels of kV <= 2.
int launch_soft(const bcjr_problem* p, int op, bcjr::Soft16Params P, void* ws, size_t ws_bytes, hipStream_t stream,
                bool* done) {
  Plan pl, hp;
  *done = false;
  int rc = make_plan(p, op, &pl);
  if (rc) return rc;
  bool halves = false;
  rc = halves_plan(p, op, pl, &hp, &halves);
  if (rc) return rc;
  if (pl.KV != 4 && !halves) return BCJR_OK;
  char* w = static_cast<char*>(ws);
  size_t left = ws_bytes;
  P.SC = 1;
  P.SU = 16;
  const size_t tb = table16_bytes(p);
  if (tb && left >= tb + pl.slot_bytes) {
    hipError_t e = bcjr::launch_transpose16(P.table, reinterpret_cast<float*>(w), p->L, p->V, stream);
    if (e != hipSuccess) return hip_fail(e, "codebook transpose launch");
    P.table = reinterpret_cast<const float*>(w);
    P.SC = (uint32_t)pl.NB;
    P.SU = 1;
    w += tb;
    left -= tb;
  }
  P.N = (int)p->N;
  P.L = p->L;
  P.Q = p->Q;
  P.t_per_seq = p->t_per_seq ? 1 : 0;
  P.slot_floats = pl.slot_bytes / sizeof(float);
  if (halves) {
    rc = launch_halves(p, op, pl, hp, P, w, left, stream, done);
    if (rc || *done) return rc;
  }
  if (pl.KV != 4) return BCJR_OK;
  *done = true;
  P.swz = pl.swz;
  P.ws = reinterpret_cast<float*>(w);
  P.mode = bcjr::SOFT_WHOLE;
  P.B = p->B;
  return launch(pl, p->B, left, &P, stream);
}

}  // namespace

// Sequence slots of bcjr_forward_noalloc: a static device array, one copy per
// GPU.  Host code never names it after set-up: its host-side symbol is only a
// stand-in, so the device address comes from hipGetSymbolAddress, once per
// device with that device current, and is kept per device.
// The slots are followed by room for what a batch in two halves keeps beside them
// (halves_bytes): 128 KiB and 8 (N + 2) bytes a sequence at L = 16, kV = 2, so a
// batch whose slots fit runs as bcjr_forward runs it (from 2^(L-kV) = 32 on: the
// offsets of a smaller trellis are as large as its slots).
constexpr size_t kNoallocBytes = BCJR_NOALLOC_SCRATCH_BYTES + ((size_t)17 << 20);
static __device__ __align__(256) unsigned char scratch[kNoallocBytes];

namespace {

std::mutex g_scratch_mu;
void* g_scratch_ptr[64];

int scratch_ptr(void** out) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return hip_fail(e, "hipGetDevice");
  if (dev < 0 || dev >= 64) return fail(BCJR_EHIP, "device ordinal %d out of range", dev);
  std::lock_guard<std::mutex> lk(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return hip_fail(e, "hipGetSymbolAddress(scratch)");
    if (!p) return fail(BCJR_EHIP, "hipGetSymbolAddress(scratch) returned NULL");
    g_scratch_ptr[dev] = p;
  }
  *out = g_scratch_ptr[dev];
  return BCJR_OK;
}

bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

int rht_impl(const float* W, float* out, int64_t batch, int64_t m, int64_t n, const float* sign_l,
             const float* sign_r, int inverse, hipStream_t stream) {
  if (batch < 0 || batch > INT32_MAX) return fail(BCJR_EINVAL, "batch=%lld outside [0, 2^31)", (long long)batch);
  if (m < 1 || m > 16384 || (m & (m - 1)))
    return fail(BCJR_EINVAL, "m=%lld must be a power of two in [1, 16384]", (long long)m);
  if (n < 1 || n > 16384 || (n & (n - 1)))
    return fail(BCJR_EINVAL, "n=%lld must be a power of two in [1, 16384]", (long long)n);
  if (batch == 0) return BCJR_OK;
  if (!W || !out || !sign_l || !sign_r) return fail(BCJR_EINVAL, "W, out, sign_l and sign_r must be non-NULL");
  const size_t bytes = (size_t)batch * m * n * sizeof(float);
  const char *w0 = reinterpret_cast<const char*>(W), *o0 = reinterpret_cast<const char*>(out);
  if (w0 < o0 + bytes && o0 < w0 + bytes) return fail(BCJR_EINVAL, "out must not alias W");
  DeviceInfo di;
  int rc = device_info(&di);
  if (rc) return rc;
  const float s = (float)(1.0 / sqrt((double)m * (double)n));
  const int blocks = di.num_cu * 8;
  const long long rows = batch * m;
  // forward: rows of W diag(sr) H_n, then row signs, then H_m and the scale;
  // inverse: rows of W H_n then diag(sr), then H_m, row signs and the scale.
  if (n >= 64 && aligned16(W) && aligned16(sign_r)) {  // tiled kernels: 2 passes over HBM for most shapes
    hipError_t e = inverse
        ? bcjr::launch_fwht_tiled(W, out, (int)batch, (int)m, (int)n, true, nullptr, nullptr, sign_r, sign_l, s,
                                  stream)
        : bcjr::launch_fwht_tiled(W, out, (int)batch, (int)m, (int)n, true, sign_r, sign_l, nullptr, nullptr, s,
                                  stream);
    return e == hipSuccess ? BCJR_OK : hip_fail(e, "bcjr_rht tiled passes");
  }
  hipError_t e =
      inverse ? bcjr::launch_fwht_rows(W, out, rows, (int)n, nullptr, sign_r, m, nullptr, 1.0f, blocks, stream)
              : bcjr::launch_fwht_rows(W, out, rows, (int)n, sign_r, nullptr, m, sign_l, 1.0f, blocks, stream);
  if (e != hipSuccess) return hip_fail(e, "bcjr_rht row pass");
  e = bcjr::launch_fwht_cols(out, (int)batch, (int)m, (int)n, inverse ? sign_l : nullptr, s, blocks, stream);
  return e == hipSuccess ? BCJR_OK : hip_fail(e, "bcjr_rht column pass");
}

}  // namespace

extern "C" {

int bcjr_workspace_bytes(const bcjr_problem* prob, int op, size_t* bytes) {
  if (!bytes) return fail(BCJR_EINVAL, "bytes is NULL");
  if (op != OP_FWD && op != OP_BWD && op != OP_VIT) return fail(BCJR_EINVAL, "unknown op %d", op);
  Plan pl;
  int rc = make_plan(prob, op, &pl);
  if (rc) return rc;
  const long long slots = std::max<long long>(1, std::min<long long>(prob->B, pl.max_blocks));
  *bytes = (size_t)slots * pl.slot_bytes;
  if (op != OP_VIT) {
    Plan hp;
    bool halves = false;
    rc = halves_plan(prob, op, pl, &hp, &halves);
    if (rc) return rc;
    // The forward's workspace is the entropy's too, which takes larger batches in two
    // halves at kV <= 2.
    if (op == OP_FWD && !halves && pl.KV <= 2) {
      rc = halves_plan(prob, OP_FWD_ENTROPY, pl, &hp, &halves);
      if (rc) return rc;
    }
    if (halves) *bytes = std::max(*bytes, (size_t)prob->B * halves_bytes(prob, op));
  }
  *bytes += table16_bytes(prob);
  return BCJR_OK;
}

int bcjr_forward(const bcjr_problem* prob, const float* seq, const float* T, const float* codebook_or_lut,
                 float* soft, float* logZ, void* ws, size_t ws_bytes, hipStream_t stream) {
  int rc0 = check_ws(prob, OP_FWD, ws, ws_bytes);
  if (rc0 || prob->B == 0) return rc0;
  if (!seq || !T || !soft || !ws) return fail(BCJR_EINVAL, "seq, T, soft and ws must be non-NULL");
  if (prob->code != BCJR_CODE_1MAD && prob->code != BCJR_CODE_3INST && !codebook_or_lut)
    return fail(BCJR_EINVAL, "code %d needs a codebook/LUT pointer", prob->code);
  bcjr::Soft16Params S = {};
  S.seq = seq;
  S.T = T;
  S.table = codebook_or_lut;
  S.out = soft;
  S.logZ = logZ;
  bool done = false;
  int rc = launch_soft(prob, OP_FWD, S, ws, ws_bytes, stream, &done);
  if (rc || done) return rc;
  Plan pl;
  rc = make_plan(prob, OP_FWD, &pl);
  if (rc) return rc;
  bcjr::FwdParams P = {};
  P.seq = seq;
  P.T = T;
  P.table = codebook_or_lut;
  P.soft = soft;
  P.logZ = logZ;
  P.ws = static_cast<float*>(ws);
  P.B = prob->B;
  P.N = (int)prob->N;
  P.L = prob->L;
  P.Q = prob->Q;
  P.t_per_seq = prob->t_per_seq ? 1 : 0;
  return launch(pl, prob->B, ws_bytes, &P, stream);
}

int bcjr_forward_noalloc(const bcjr_problem* prob, const float* seq, const float* T, const float* codebook_or_lut,
                         float* soft, float* logZ, hipStream_t stream) {
  int rc = validate(prob);
  if (rc || prob->B == 0) return rc;
  const size_t slot = slot_bytes_of(prob, OP_FWD);
  if (slot > BCJR_NOALLOC_SCRATCH_BYTES)
    return fail(BCJR_EWORKSPACE,
                "one sequence slot needs %zu bytes (N=%lld, L=%d, k*V=%d); the static scratch holds %zu",
                slot, (long long)prob->N, prob->L, prob->k * prob->V, (size_t)BCJR_NOALLOC_SCRATCH_BYTES);
  void* ws = nullptr;
  rc = scratch_ptr(&ws);
  if (rc) return rc;
  return bcjr_forward(prob, seq, T, codebook_or_lut, soft, logZ, ws, kNoallocBytes, stream);
}

int bcjr_forward_internals(const bcjr_problem* prob, const float* seq, const float* T,
                           const float* codebook_or_lut, float* soft, float* logZ, float* marginals,
                           float* log_alpha, float* log_beta, void* ws, size_t ws_bytes, hipStream_t stream) {
  int rc0 = check_ws(prob, OP_FWD, ws, ws_bytes);
  if (rc0 || prob->B == 0) return rc0;
  if (!seq || !T || !soft || !ws || !marginals || !log_alpha || !log_beta)
    return fail(BCJR_EINVAL, "seq, T, soft, ws, marginals, log_alpha and log_beta must be non-NULL");
  if (prob->code != BCJR_CODE_1MAD && prob->code != BCJR_CODE_3INST && !codebook_or_lut)
    return fail(BCJR_EINVAL, "code %d needs a codebook/LUT pointer", prob->code);
  Plan pl;
  int rc = make_plan(prob, OP_FWD_INTERNALS, &pl);
  if (rc) return rc;
  bcjr::FwdParams P = {};
  P.seq = seq;
  P.T = T;
  P.table = codebook_or_lut;
  P.soft = soft;
  P.logZ = logZ;
  P.ws = static_cast<float*>(ws);
  P.P_out = marginals;
  P.la_out = log_alpha;
  P.lb_out = log_beta;
  P.B = prob->B;
  P.N = (int)prob->N;
  P.L = prob->L;
  P.Q = prob->Q;
  P.t_per_seq = prob->t_per_seq ? 1 : 0;
  rc = launch(pl, prob->B, ws_bytes, &P, stream);
  if (rc) return rc;
  // kV = 4 and batches in two halves: soft and log Z as bcjr_forward gives them, bit
  // for bit, over the diagnostics kernel's own, which sums in another order (a forward
  // more, 2-9 % of the call at L = 16, 20-40 % on the smallest lattices).  Larger
  // kV <= 2 batches keep its own: the bits of bcjr_forward below L = 14 only.
  bcjr::Soft16Params S = {};
  S.seq = seq;
  S.T = T;
  S.table = codebook_or_lut;
  S.out = soft;
  S.logZ = logZ;
  bool done = false;
  return launch_soft(prob, OP_FWD, S, ws, ws_bytes, stream, &done);
}

int bcjr_forward_entropy(const bcjr_problem* prob, const float* seq, const float* T,
                         const float* codebook_or_lut, float* soft, float* logZ, float* entropy, void* ws,
                         size_t ws_bytes, hipStream_t stream) {
  int rc0 = check_ws(prob, OP_FWD, ws, ws_bytes);
  if (rc0 || prob->B == 0) return rc0;
  if (!seq || !T || !soft || !ws || !entropy)
    return fail(BCJR_EINVAL, "seq, T, soft, ws and entropy must be non-NULL");
  if (prob->code != BCJR_CODE_1MAD && prob->code != BCJR_CODE_3INST && !codebook_or_lut)
    return fail(BCJR_EINVAL, "code %d needs a codebook/LUT pointer", prob->code);
  bcjr::Soft16Params S = {};
  S.seq = seq;
  S.T = T;
  S.table = codebook_or_lut;
  S.out = soft;
  S.logZ = logZ;
  S.H_out = entropy;
  bool done = false;
  int rc = launch_soft(prob, OP_FWD_ENTROPY, S, ws, ws_bytes, stream, &done);
  if (rc || done) return rc;
  Plan pl;
  rc = make_plan(prob, OP_FWD_ENTROPY, &pl);
  if (rc) return rc;
  bcjr::FwdParams P = {};
  P.seq = seq;
  P.T = T;
  P.table = codebook_or_lut;
  P.soft = soft;
  P.logZ = logZ;
  P.ws = static_cast<float*>(ws);
  P.H_out = entropy;
  P.B = prob->B;
  P.N = (int)prob->N;
  P.L = prob->L;
  P.Q = prob->Q;
  P.t_per_seq = prob->t_per_seq ? 1 : 0;
  return launch(pl, prob->B, ws_bytes, &P, stream);
}

int bcjr_backward(const bcjr_problem* prob, const float* seq, const float* T, const float* codebook_or_lut,
                  const float* logZ, const float* g_soft, const float* g_logZ, float* g_seq, void* ws,
                  size_t ws_bytes, hipStream_t stream) {
  (void)logZ;
  int rc0 = check_ws(prob, OP_BWD, ws, ws_bytes);
  if (rc0 || prob->B == 0) return rc0;
  if (!seq || !T || !g_soft || !g_seq || !ws)
    return fail(BCJR_EINVAL, "seq, T, g_soft, g_seq and ws must be non-NULL");
  if (prob->code != BCJR_CODE_1MAD && prob->code != BCJR_CODE_3INST && !codebook_or_lut)
    return fail(BCJR_EINVAL, "code %d needs a codebook/LUT pointer", prob->code);
  bcjr::Soft16Params S = {};
  S.seq = seq;
  S.T = T;
  S.table = codebook_or_lut;
  S.out = g_seq;
  S.g_soft = g_soft;
  S.g_logZ = g_logZ;
  bool done = false;
  int rc = launch_soft(prob, OP_BWD, S, ws, ws_bytes, stream, &done);
  if (rc || done) return rc;
  Plan pl;
  rc = make_plan(prob, OP_BWD, &pl);
  if (rc) return rc;
  bcjr::BwdParams P = {};
  P.seq = seq;
  P.T = T;
  P.table = codebook_or_lut;
  P.g_soft = g_soft;
  P.g_logZ = g_logZ;
  P.g_seq = g_seq;
  P.ws = static_cast<float*>(ws);
  P.B = prob->B;
  P.N = (int)prob->N;
  P.L = prob->L;
  P.Q = prob->Q;
  P.t_per_seq = prob->t_per_seq ? 1 : 0;
  P.swz = pl.swz;
  return launch(pl, prob->B, ws_bytes, &P, stream);
}

int bcjr_viterbi(const bcjr_problem* prob, const float* seq, const float* codebook_or_lut, int32_t* walk,
                 int32_t* bitstream, int32_t* start_state, float* recon, float* mse, uint8_t* packed, void* ws,
                 size_t ws_bytes, hipStream_t stream) {
  int rc0 = check_ws(prob, OP_VIT, ws, ws_bytes);
  if (rc0 || prob->B == 0) return rc0;
  if (!seq || !ws) return fail(BCJR_EINVAL, "seq and ws must be non-NULL");
  if (prob->code != BCJR_CODE_1MAD && prob->code != BCJR_CODE_3INST && !codebook_or_lut)
    return fail(BCJR_EINVAL, "code %d needs a codebook/LUT pointer", prob->code);
  if (packed && 8 % (prob->k * prob->V) != 0) return fail(BCJR_EINVAL, "packing needs k*V to divide 8");
  bcjr::VitParams P = {};
  P.seq = seq;
  P.table = codebook_or_lut;
  P.walk = walk;
  P.bits = bitstream;
  P.start = start_state;
  P.recon = recon;
  P.mse = mse;
  P.packed = packed;
  P.B = prob->B;
  P.N = (int)prob->N;
  P.L = prob->L;
  P.Q = prob->Q;
  return launch_viterbi(prob, P, ws, ws_bytes, stream);
}

int bcjr_viterbi_constrained(const bcjr_problem* prob, const float* seq, const float* codebook_or_lut,
                             int overlap_bits, const int32_t* overlap, int32_t* walk, int32_t* bitstream,
                             int32_t* start_state, float* recon, float* mse, uint8_t* packed, void* ws,
                             size_t ws_bytes, hipStream_t stream) {
  int rc0 = check_ws(prob, OP_VIT, ws, ws_bytes);
  if (rc0 || prob->B == 0) return rc0;
  if (overlap_bits < 0 || overlap_bits > prob->L - prob->k * prob->V)
    return fail(BCJR_EINVAL, "overlap_bits=%d must lie in [0, L - k*V] = [0, %d]", overlap_bits,
                prob->L - prob->k * prob->V);
  if (!seq || !ws || !overlap) return fail(BCJR_EINVAL, "seq, overlap and ws must be non-NULL");
  if (prob->code != BCJR_CODE_1MAD && prob->code != BCJR_CODE_3INST && !codebook_or_lut)
    return fail(BCJR_EINVAL, "code %d needs a codebook/LUT pointer", prob->code);
  if (packed && 8 % (prob->k * prob->V) != 0) return fail(BCJR_EINVAL, "packing needs k*V to divide 8");
  bcjr::VitParams P = {};
  P.seq = seq;
  P.table = codebook_or_lut;
  P.walk = walk;
  P.bits = bitstream;
  P.start = start_state;
  P.recon = recon;
  P.mse = mse;
  P.packed = packed;
  P.overlap = overlap;
  P.overlap_bits = overlap_bits;
  P.B = prob->B;
  P.N = (int)prob->N;
  P.L = prob->L;
  P.Q = prob->Q;
  return launch_viterbi(prob, P, ws, ws_bytes, stream);
}

int bcjr_decode(const bcjr_problem* prob, const int32_t* bitstream, const uint8_t* packed,
                const int32_t* start_state, const float* codebook_or_lut, int32_t* walk, float* recon,
                hipStream_t stream) {
  int rc = validate(prob);
  if (rc) return rc;
  if (prob->B == 0) return BCJR_OK;
  if ((!bitstream && !packed) || !start_state)
    return fail(BCJR_EINVAL, "need start_state and one of bitstream / packed");
  if (recon && prob->code != BCJR_CODE_1MAD && prob->code != BCJR_CODE_3INST && !codebook_or_lut)
    return fail(BCJR_EINVAL, "code %d needs a codebook/LUT pointer", prob->code);
  const int KV = prob->k * prob->V;
  const void* fn = bcjr::decode_kernel_ptr(KV, prob->V, prob->code);
  if (!fn) return fail(BCJR_EUNSUPPORTED, "no decode kernel for k*V=%d V=%d code=%d", KV, prob->V, prob->code);
  bcjr::DecParams P = {bitstream, packed, start_state, codebook_or_lut, walk, recon,
                       prob->B, (int)prob->N, prob->L, prob->Q};
  void* args[] = {&P};
  const unsigned grid = (unsigned)((prob->B + 255) / 256);
  hipError_t e = hipLaunchKernel(fn, dim3(grid), dim3(256), args, 0, stream);
  if (e != hipSuccess) return hip_fail(e, "hipLaunchKernel(decode)");
  return BCJR_OK;
}

int bcjr_viterbi_trace(const bcjr_problem* prob, const float* seq, const float* codebook_or_lut, float* trace,
                       int32_t* backptr, hipStream_t stream) {
  int rc = validate(prob);
  if (rc) return rc;
  if (prob->B == 0) return BCJR_OK;
  if (!seq || !trace || !backptr) return fail(BCJR_EINVAL, "seq, trace and backptr must be non-NULL");
  if (prob->code != BCJR_CODE_1MAD && prob->code != BCJR_CODE_3INST && !codebook_or_lut)
    return fail(BCJR_EINVAL, "code %d needs a codebook/LUT pointer", prob->code);
  const int KV = prob->k * prob->V;
  const void* fn = bcjr::trace_kernel_ptr(KV, prob->V, prob->code);
  if (!fn) return fail(BCJR_EUNSUPPORTED, "no trace kernel for k*V=%d V=%d code=%d", KV, prob->V, prob->code);
  DeviceInfo di;
  rc = device_info(&di);
  if (rc) return rc;
  // The reduced vector and its argmin: NT floats + NT bytes (NT <= 2^14 for a
  // validated problem, so at most 16 reduced indices per thread of 1024).
  const int NT = 1 << (prob->L - KV);
  const int nthr = NT < 64 ? 64 : (NT > 1024 ? 1024 : NT);
  const size_t lds = (size_t)NT * (sizeof(float) + 1);
  if (lds > di.max_lds)
    return fail(BCJR_EUNSUPPORTED, "viterbi trace needs %zu bytes of LDS per workgroup (device limit %zu)", lds,
                di.max_lds);
  hipError_t e = hipFuncSetAttribute(fn, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
  if (e != hipSuccess) return hip_fail(e, "hipFuncSetAttribute(MaxDynamicSharedMemorySize)");
  const long long cap = (long long)di.num_cu * 2;
  const unsigned grid = (unsigned)(prob->B < cap ? prob->B : cap);
  bcjr::TraceParams P = {seq, codebook_or_lut, trace, backptr, prob->B, (int)prob->N, prob->L, prob->Q};
  void* args[] = {&P};
  e = hipLaunchKernel(fn, dim3(grid), dim3(nthr), args, lds, stream);
  if (e != hipSuccess) return hip_fail(e, "hipLaunchKernel(viterbi_trace)");
  return BCJR_OK;
}

static_assert(bcjr::BITS_FMT_U8 == BCJR_BITS_U8 && bcjr::BITS_FMT_I32 == BCJR_BITS_I32 &&
                  bcjr::BITS_FMT_PACKED == BCJR_BITS_PACKED,
              "bitstream layout ids");

int bcjr_dequant(const bcjr_problem* prob, const void* bitstream, int bits_format,
                 const int32_t* start_state, const float* codebook_or_lut, int64_t m, int64_t n, int Tx,
                 int Ty, double scale, float* out, hipStream_t stream) {
  int rc = validate(prob);
  if (rc) return rc;
  if (Tx < 1 || Ty < 1) return fail(BCJR_EINVAL, "tile %dx%d must be positive", Tx, Ty);
  if (m < 0 || n < 0 || m % Tx || n % Ty)
    return fail(BCJR_EINVAL, "matrix %lldx%lld is not a whole number of %dx%d tiles", (long long)m,
                (long long)n, Tx, Ty);
  if ((long long)Tx * Ty != prob->N * prob->V)
    return fail(BCJR_EINVAL, "tile %dx%d holds %lld weights, sequences N*V=%lld", Tx, Ty,
                (long long)Tx * Ty, (long long)(prob->N * prob->V));
  if (prob->B != (m / Tx) * (n / Ty))
    return fail(BCJR_EINVAL, "B=%lld but the matrix has %lld tiles", (long long)prob->B,
                (long long)((m / Tx) * (n / Ty)));
  if (bits_format != BCJR_BITS_U8 && bits_format != BCJR_BITS_I32 && bits_format != BCJR_BITS_PACKED)
    return fail(BCJR_EINVAL, "unknown bitstream format %d", bits_format);
  if (prob->B == 0) return BCJR_OK;
  if (!bitstream || !start_state || !out) return fail(BCJR_EINVAL, "bitstream, start_state and out are required");
  if (prob->code != BCJR_CODE_1MAD && prob->code != BCJR_CODE_3INST && !codebook_or_lut)
    return fail(BCJR_EINVAL, "code %d needs a codebook/LUT pointer", prob->code);
  const int KV = prob->k * prob->V;
  const bool out16 = (reinterpret_cast<uintptr_t>(out) & 15) == 0;
  // 16x16 tiles at k = 2: one thread per tile row, aligned vector loads of its bits.
  const size_t bits_align = bits_format == BCJR_BITS_PACKED ? 4 : 16;
  const bool t16 = Tx == 16 && Ty == 16 && prob->k == 2 && (m * n) / 4 < (1ll << 31) && out16 &&
                   (reinterpret_cast<uintptr_t>(bitstream) % bits_align) == 0;
  // Vector path: 4 columns of one tile row per thread, 16-byte stores, 32-bit indices.
  const bool vec4 = !t16 && Ty % 4 == 0 && (m * n) / 4 < (1ll << 31) && out16;
  const void* fn = t16 ? bcjr::dequant_t16_kernel_ptr(KV, prob->V, prob->code, bits_format)
                       : bcjr::dequant_kernel_ptr(KV, prob->V, prob->code, vec4);
  if (!fn) return fail(BCJR_EUNSUPPORTED, "no dequant kernel for k*V=%d V=%d code=%d", KV, prob->V, prob->code);
  auto log2_or_neg = [](int x) { return (x < 1 || (x & (x - 1))) ? -1 : __builtin_ctz((unsigned)x); };
  bcjr::DqParams P = {bits_format == BCJR_BITS_I32 ? static_cast<const int32_t*>(bitstream) : nullptr,
                      bits_format == BCJR_BITS_U8 ? static_cast<const uint8_t*>(bitstream) : nullptr,
                      bits_format == BCJR_BITS_PACKED ? static_cast<const uint8_t*>(bitstream) : nullptr,
                      start_state, codebook_or_lut, out, m, n, (int)prob->N, prob->L, prob->Q, Tx, Ty,
                      log2_or_neg(Tx), log2_or_neg(Ty), (double)(float)scale == scale ? 1 : 0, scale};
  void* args[] = {&P};
  // t16: one workgroup per 16-row x 64-column unit; others: one thread per 4 or 1 elements
  const long long blocks = t16 ? (m / 16) * ((n / 4 + 15) / 16) : (vec4 ? m * n / 4 + 255 : m * n + 255) / 256;
  long long cap = 16384;
  size_t lds = 0;
  if (t16 && prob->code == BCJR_CODE_HYB) {  // LUT staged in LDS: persistent grid
    DeviceInfo di;
    int rc2 = device_info(&di);
    if (rc2) return rc2;
    cap = (long long)di.num_cu * 8;
    lds = (size_t)(2 << prob->Q) * sizeof(float);
  }
  const unsigned grid = (unsigned)(blocks < cap ? blocks : cap);
  hipError_t e = hipLaunchKernel(fn, dim3(grid), dim3(256), args, lds, stream);
  if (e != hipSuccess) return hip_fail(e, "hipLaunchKernel(dequant)");
  return BCJR_OK;
}

int bcjr_codebook(const bcjr_problem* prob, const float* lut, float* codebook_out, hipStream_t stream) {
  if (!prob) return fail(BCJR_EINVAL, "problem is NULL");
  if (prob->L < 1 || prob->L > 24) return fail(BCJR_EINVAL, "L=%d outside [1, 24]", prob->L);
  if (!codebook_out) return fail(BCJR_EINVAL, "codebook_out is NULL");
  const void* fn = bcjr::codebook_kernel_ptr(prob->code);
  if (!fn) return fail(BCJR_EINVAL, "code %d has no generator", prob->code);
  if (prob->code == BCJR_CODE_HYB && (!lut || prob->Q < 1 || prob->Q > 12))
    return fail(BCJR_EINVAL, "HYB needs a LUT and Q in [1, 12]");
  bcjr::CbParams P = {lut, codebook_out, 1ll << prob->L, prob->Q};
  void* args[] = {&P};
  const unsigned grid = (unsigned)((P.S + 255) / 256);
  hipError_t e = hipLaunchKernel(fn, dim3(grid), dim3(256), args, 0, stream);
  if (e != hipSuccess) return hip_fail(e, "hipLaunchKernel(codebook)");
  return BCJR_OK;
}

int bcjr_hadamard(const float* x, float* out, int64_t rows, int64_t n, float scale, hipStream_t stream) {
  if (rows < 0) return fail(BCJR_EINVAL, "rows=%lld must be >= 0", (long long)rows);
  if (n < 1 || n > 16384 || (n & (n - 1)))
    return fail(BCJR_EINVAL, "n=%lld must be a power of two in [1, 16384]", (long long)n);
  if (rows == 0) return BCJR_OK;
  if (!x || !out) return fail(BCJR_EINVAL, "x and out must be non-NULL");
  DeviceInfo di;
  int rc = device_info(&di);
  if (rc) return rc;
  hipError_t e;
  if (n >= 64 && rows <= INT32_MAX && aligned16(x))
    e = bcjr::launch_fwht_tiled(x, out, 1, (int)rows, (int)n, false, nullptr, nullptr, nullptr, nullptr, scale,
                                stream);
  else
    e = bcjr::launch_fwht_rows(x, out, rows, (int)n, nullptr, nullptr, rows, nullptr, scale, di.num_cu * 8, stream);
  return e == hipSuccess ? BCJR_OK : hip_fail(e, "bcjr_hadamard launch");
}


int bcjr_rht(const float* W, float* out, int64_t m, int64_t n, const float* sign_l, const float* sign_r,
             int inverse, hipStream_t stream) {
  return rht_impl(W, out, 1, m, n, sign_l, sign_r, inverse, stream);
}

int bcjr_rht_batched(const float* W, float* out, int64_t batch, int64_t m, int64_t n, const float* sign_l,
                     const float* sign_r, int inverse, hipStream_t stream) {
  return rht_impl(W, out, batch, m, n, sign_l, sign_r, inverse, stream);
}

const char* bcjr_strerror(int status) {
  switch (status) {
    case BCJR_OK: return "ok";
    case BCJR_EINVAL: return "invalid argument";
    case BCJR_EUNSUPPORTED: return "unsupported configuration";
    case BCJR_EWORKSPACE: return "workspace too small";
    case BCJR_EHIP: return "HIP runtime error";
    default: return "unknown status";
  }
}

const char* bcjr_last_error(void) { return g_last_error.c_str(); }

const char* bcjr_version(void) { return "bcjr_hip 0.1.0 (gfx950)"; }

}  // extern "C"
