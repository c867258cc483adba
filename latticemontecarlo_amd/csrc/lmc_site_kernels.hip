// gfx950 kernels of the swap / site energy change (EnergyChangePredictorPairSite), the
// CanonicalMc driver and the full-lattice cluster-expansion energy (EnergyPredictor).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <mutex>
#include <type_traits>

#include "lmc_dev_common.h"
#include "lmc_device.h"
#include "lmc_rng.h"

namespace lmc {
namespace {
// ---------------------------------------------------------------------------------------------
// Swap / site energy change (EnergyChangePredictorPairSite.cpp:69-192).
struct SiteLds {
  uint32_t cl[kMaxSiteClusters];
  int32_t off[kSiteSlots];
  double w[kMaxW];
  uint8_t env[2][48];           // environments of the swap's sites
  int slot[2];                  // partner slots (q around p, p around q)
  double part[kThreads / 64];   // per-wave partial sums
  double term[kThreads];        // a swap's terms by cluster
};

__device__ void LoadSiteTables(const KTables &t, SiteLds &L) {
  for (int i = threadIdx.x; i < t.n_site; i += blockDim.x) L.cl[i] = t.site_cl[i];
  for (int i = threadIdx.x; i < kSiteSlots; i += blockDim.x) L.off[i] = t.site_off[i];
  for (int i = threadIdx.x; i < t.nw; i += blockDim.x) L.w[i] = t.w[i];
}

__device__ __forceinline__ double SiteWeight(const KTables &t, const SiteLds &L, const uint8_t *e,
                                             uint32_t d, int centre) {
  const int S = t.S, label = d & 7, o1 = (d >> 4) & 63, o2 = (d >> 10) & 63;
  if (label == 0) return L.w[centre];
  if (label < 4) return L.w[S + (label - 1) * S * S + centre * S + e[o1]];
  return L.w[S + 3 * S * S + (label - 4) * S * S * S + (centre * S + e[o1]) * S + e[o2]];
}

// Sum over clusters containing site x of w(x -> en) - w(x -> eo), skipping clusters that
// contain env slot `skip` (the partner of a coupled swap): this thread's share.
__device__ double SitePartial(const KTables &t, const SiteLds &L, int which, int eo, int en,
                              int skip) {
  const uint8_t *e = L.env[which];
  double acc = 0.0;
  for (int c = threadIdx.x; c < t.n_site; c += blockDim.x) {
    const uint32_t d = L.cl[c];
    const int o1 = (d >> 4) & 63, o2 = (d >> 10) & 63;
    if (skip >= 0 && (o1 == skip || o2 == skip)) continue;
    acc += SiteWeight(t, L, e, d, en) - SiteWeight(t, L, e, d, eo);
  }
  return acc;
}

// Fixed-order block sum, valid in thread 0: DPP sums within each wave, then the wave sums in
// wave order. One barrier; L.part is rewritten only after the caller's next barrier.
__device__ double BlockSum(SiteLds &L, double v) {
  v = WaveSum(v);
  if ((threadIdx.x & 63) == 0) L.part[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < kThreads / 64; ++w) r += L.part[w];
  return r;
}

// Species in the 43-site environment of x (slot i read by lane i of the calling wave).
__device__ void GatherSite(const SiteLds &L, uint8_t *dst, const uint8_t *occ, int n,
                           const XYZ &c, int S, int lane) {
  if (lane < kSiteSlots) {
    int dx, dy, dz;
    Unpack(L.off[lane], dx, dy, dz);
    const uint8_t v = occ[SiteAt(c, n, dx, dy, dz)];
    dst[lane] = v < S ? v : 0;  // codes are validated by the callers; keep LDS indices in range
  }
}

// Periodic minimum image of a coordinate difference on the 2n axis, in [-n, n).
__device__ __forceinline__ int MinImage(int v, int n) {  // |v| < 2n
  const int m = 2 * n;
  v += v < 0 ? m : 0;
  return v >= n ? v - m : v;
}

// Slot of b in the environment of a: the first slot whose offset is the minimum-image
// difference b - a, or -1 beyond the third shell. Lane i of the calling wave tests slot i.
__device__ int PartnerSlot(const SiteLds &L, int n, const XYZ &a, const XYZ &b, int lane) {
  const int dx = MinImage(b.X - a.X, n), dy = MinImage(b.Y - a.Y, n), dz = MinImage(b.Z - a.Z, n);
  bool hit = false;
  if (lane >= 1 && lane < kSiteSlots) {
    int x, y, z;
    Unpack(L.off[lane], x, y, z);
    hit = x == dx && y == dy && z == dz;
  }
  const uint64_t m = __ballot(hit);
  return m ? __builtin_ctzll(m) : -1;
}

// Environments and partner slots of a swap p <-> q: wave 0 gathers around p, wave 1 around q.
// Results in L.env and L.slot after the caller's barrier.
__device__ void GatherPair(SiteLds &L, const uint8_t *occ, int n, int64_t p, int64_t q, int S) {
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  if (wave > 1) return;
  const XYZ a = ToXYZ(wave ? q : p, n), b = ToXYZ(wave ? p : q, n);
  GatherSite(L, L.env[wave], occ, n, a, S, lane);
  const int s = PartnerSlot(L, n, a, b, lane);
  if (lane == 0) L.slot[wave] = s;
}

// dE of swapping species ep at p and eq at q, from the environments of GatherPair. Far pairs:
// dE(p) + dE(q) on the unswapped config (...WithoutCoupling :136-146). Near pairs: clusters
// containing both keep their multiset and are skipped (...WithCoupling :96-134). All threads
// call; the result is valid in thread 0. Added in the serial trials' order (a lane's clusters lane,
// lane + 64, ..., then the wave sum): the two give the same bits.
__device__ double SwapDe(const KTables &t, SiteLds &L, int ep, int eq) {
  static_assert(kThreads >= kMaxSiteClusters, "one cluster per thread");
  L.term[threadIdx.x] = SitePartial(t, L, 0, ep, eq, L.slot[0]) + SitePartial(t, L, 1, eq, ep, L.slot[1]);
  __syncthreads();
  double v = 0.0;
  if (threadIdx.x < 64) {
    for (int i = threadIdx.x; i < kThreads; i += 64) v += L.term[i];
    v = WaveSum(v);
  }
  return v;
}

__global__ __launch_bounds__(kThreads) void SwapDeKernel(KTables t, const uint8_t *occ,
                                                         const int64_t *off, const int32_t *ncell,
                                                         const int64_t *pairs, double *de) {
  __shared__ SiteLds L;
  const int r = blockIdx.x;
  const int64_t p = pairs[2 * r], q = pairs[2 * r + 1];
  const uint8_t *o = occ + off[r];
  if (!ValidSite(ncell[r], p) || !ValidSite(ncell[r], q) || o[p] >= t.S || o[q] >= t.S) {
    if (threadIdx.x == 0) de[r] = __builtin_nan("");
    return;
  }
  const int ep = o[p], eq = o[q];
  if (ep == eq) {
    if (threadIdx.x == 0) de[r] = 0.0;
    return;
  }
  LoadSiteTables(t, L);
  __syncthreads();
  GatherPair(L, o, ncell[r], p, q, t.S);
  __syncthreads();
  const double v = SwapDe(t, L, ep, eq);
  if (threadIdx.x == 0) de[r] = v;
}

// GetDeFromLatticeIdSite (EnergyChangePredictorPairSite.cpp:154-192): site sites[r] changes from
// species from[r] (null: the species it holds) to codes[r], the rest of the occupancy as is.
__global__ __launch_bounds__(kThreads) void SiteDeKernel(KTables t, const uint8_t *occ,
                                                         const int64_t *off, const int32_t *ncell,
                                                         const int64_t *sites, const uint8_t *from,
                                                         const uint8_t *codes, double *de) {
  __shared__ SiteLds L;
  const int r = blockIdx.x;
  const uint8_t *o = occ + off[r];
  if (!ValidSite(ncell[r], sites[r]) || o[sites[r]] >= t.S || codes[r] >= t.S ||
      (from && from[r] >= t.S)) {
    if (threadIdx.x == 0) de[r] = __builtin_nan("");
    return;
  }
  LoadSiteTables(t, L);
  __syncthreads();
  const int eo = from ? from[r] : o[sites[r]], en = codes[r];
  if (eo == en) {
    if (threadIdx.x == 0) de[r] = 0.0;
    return;
  }
  if (threadIdx.x < 64)
    GatherSite(L, L.env[0], o, ncell[r], ToXYZ(sites[r], ncell[r]), t.S, threadIdx.x);
  __syncthreads();
  const double v = BlockSum(L, SitePartial(t, L, 0, eo, en, -1));
  if (threadIdx.x == 0) de[r] = v;
}

// SimulatedAnnealing::UpdateTemperature (SimulatedAnnealing.cpp:99-133) with maximum_steps N:
// the window, trigger and cooldown lengths and the per-step decay factor exp(-3/N).
struct AnnealSchedule {
  uint64_t window, trigger, cooldown;
  double decay;
};
__device__ AnnealSchedule MakeAnnealSchedule(uint64_t N) {
  AnnealSchedule s;
  s.window = max(1ull, static_cast<unsigned long long>(N * 0.001));
  s.trigger = max(1ull, static_cast<unsigned long long>(N * 0.05));
  s.cooldown = max(1ull, static_cast<unsigned long long>(N * 0.10));
  s.decay = exp(-3.0 / static_cast<double>(max(1ull, static_cast<unsigned long long>(N))));
  return s;
}

// The temperature update after the trial of step `steps` with the energy after the trial.
__device__ void AnnealUpdate(CmcAnneal &A, const AnnealSchedule &s, bool accepted,
                             uint64_t steps, double energy) {
  ++A.window_trials;
  if (accepted) {
    ++A.window_accepts;
    if (energy < A.recent_best - 1e-4) {
      A.recent_best = energy;
      A.last_improvement = steps;
    }
  }
  if (A.window_trials >= s.window) {
    const double acc = static_cast<double>(A.window_accepts) / static_cast<double>(A.window_trials);
    if (acc > 0.50) A.T *= 0.99;
    A.window_trials = 0;
    A.window_accepts = 0;
  }
  // the acceptance estimate last: the division only runs when the other conditions hold
  if (A.reheats < 5 && steps - A.last_improvement >= s.trigger &&
      steps - A.last_reheat >= s.cooldown &&
      (A.window_trials > 0u ? static_cast<double>(A.window_accepts) /
                                  static_cast<double>(A.window_trials)
                            : 1.0) < 0.05) {
    A.T *= 1.10;
    A.last_improvement = steps;
    A.last_reheat = steps;
    A.recent_best = energy;
    ++A.reheats;
  }
  A.T *= s.decay;
}

constexpr uint32_t kMaxPairAttempts = 1u << 20;

// A pair draw attempt is Philox counter 2 attempt + 1 of the trial's (the round's) first step;
// CanonicalMcAbstract.cpp:43-101 redraws until the species differ, so the lowest attempt with different
// species is the sequential answer.

// Site coordinates X, Y < 2^11 and Z / 2 < 2^10 in one word (every box has n <= 1000).
__device__ __forceinline__ uint32_t PackSiteXYZ(uint32_t site, uint32_t n) {
  const uint32_t plane = 2u * n * n, X = site / plane, rest = site - X * plane, Y = rest / n;
  return X | Y << 11 | (rest - Y * n) << 22;
}
__device__ __forceinline__ XYZ UnpackSiteXYZ(uint32_t v) {
  const int X = v & 2047, Y = (v >> 11) & 2047;
  return {X, Y, static_cast<int>(v >> 22) * 2 + ((X + Y) & 1)};
}

// Site at offset (dx, dy, dz), |d| <= n, of c: SiteAt in 32 bits without compares (24-bit factors).
__device__ __forceinline__ uint32_t SiteNear(const XYZ &c, uint32_t n, int dx, int dy, int dz) {
  const uint32_t m = 2 * n;
  auto wrap = [&](int v) {
    const uint32_t u = static_cast<uint32_t>(v);
    return min(min(u, u + m), u - m);
  };
  const uint32_t X = wrap(c.X + dx), Y = wrap(c.Y + dy), Z = wrap(c.Z + dz);
  return __umul24(X, 2 * __umul24(n, n)) + (__umul24(Y, n) + (Z >> 1));
}

// Metropolis uniform of step `steps`.
__device__ __forceinline__ double TrialUniform(const CmcDev &c, int r, uint64_t steps) {
  const U4 u = Philox4x32_10(c.seed[r], steps, c.rid[r], 0xFFFFFFFEu);
  return UnitOpenRight(Join64(u.x, u.y));
}

// Cluster i of the site table, decoded once: the weight index of centre species x with the
// other sites' species e1, e2 is base + x kx + e1 k1 + e2 k2 (SiteWeight's three cases).
struct SiteCluster {
  int base, kx, k1, k2;
  int o1, o2;      // environment slots read (0 where unused)
  int r1, r2;      // raw slots (63 = none), for the partner test
  bool live;
};
__device__ SiteCluster DecodeSiteCluster(const KTables &t, const uint32_t *cl, int i) {
  SiteCluster q{};
  q.live = i < t.n_site;
  if (!q.live) return q;
  const uint32_t d = cl[i];
  const int S = t.S, label = d & 7;
  q.r1 = (d >> 4) & 63;
  q.r2 = (d >> 10) & 63;
  if (label == 0) {
    q.kx = 1;
  } else if (label < 4) {
    q.base = S + (label - 1) * S * S;
    q.kx = S;
    q.k1 = 1;
    q.o1 = q.r1;
  } else {
    q.base = S + 3 * S * S + (label - 4) * S * S * S;
    q.kx = S * S;
    q.k1 = S;
    q.k2 = 1;
    q.o1 = q.r1;
    q.o2 = q.r2;
  }
  return q;
}

// The dump cadence, evaluated for consecutive steps with one division per change of cadence.
// Canonical MC (CanonicalMcAbstract.cpp:69-81): steps % every == 0 with every =
// 10^(floor(log10(steps + 1)) - 1), at least 1 and at most L, while steps <= 10 L, and L past
// that. Annealing (`plain`, SimulatedAnnealing.cpp:90): steps % L == 0.
struct LogClock {
  uint64_t L = 0, every = 1, rem = 0, change = 0;  // change: the first step of another cadence
  bool plain = false;
  __device__ void Reset(uint64_t s) {
    every = L;
    change = ~0ull;
    if (!plain && s <= 10 * L) {
      uint64_t p = 1;
      for (uint64_t t = s + 1; t >= 100; t /= 10) p *= 10;
      every = p < L ? p : L;
      const uint64_t next = p <= (~0ull) / 100 ? 100 * p - 1 : ~0ull;  // s + 1 reaches 100 p
      change = next < 10 * L + 1 ? next : 10 * L + 1;
    }
    rem = s % every;
  }
  // Whether step s is due; s is the step Reset saw, then each following step once, in order.
  __device__ bool Due(uint64_t s) {
    if (s >= change) Reset(s);
    const bool due = rem == 0;
    if (++rem == every) rem = 0;
    return due;
  }
};

// CanonicalMcSerial (CanonicalMcSerial.cpp:40-51, CanonicalMcAbstract.cpp:43-101) with an
// optional linear temperature ramp t0 -> t1 over maximum_steps, or the adaptive annealing
// schedule. One workgroup per replica. kLdsOcc: the replica's occupancy (N bytes, N a multiple
// of 4) lives in dynamic LDS for the launch and is written back at its end.
//
// Bound by the latency of one trial's chain (draw, species, environments, weights, Metropolis), so
// kCmcWaves trials run side by side on the same occupancy and are taken in order up to the first that
// an accepted one before it would have changed: the trajectory is the sequential one. A round:
//   1. wave w finds the pair of step s + w among the 63 attempts that it drew ahead (lane 63 drew the
//      Metropolis uniform), gathers both environments, adds the change of the site clusters (four to a
//      lane) for both sites and tests the step;
//   2. an accepted trial has marked its two sites in the occupancy (top bit); the later waves look at
//      the sites that they read (attempts up to the winning one, environments) again, and the first
//      that read a site of an accepted trial before it ends the round;
//   3. the commit wave swaps, records, adds the energies in order, and sets the next round's betas,
//      while the other waves draw the attempts of the next round's steps.
// 64 replicas of 30^3 cells at 5 at.% solute, 2 000 trials: 2 760 -> 820 us (two trials to a round, each
// by a whole workgroup of four waves, before); 6^3 cells 2 940 -> 1 800, 1 at.% 3 990 -> 2 500, annealing
// 2 920 -> 1 170.
// In a small box accepted trials often end a round early: the next rounds then try fewer, and more again
// after one that was taken whole (8 waves instead of 15: 15 % slower at 30^3 cells, 28 % faster at
// 6^3). A wave that missed its pair in the first 63 attempts draws 127 ahead
// until one of the first eight wins.
// kLog: the log records and the averaging ring are compiled in (taken when c.log_every is set).
constexpr int kCmcWaves = 15;
constexpr int kCmcRing = 32;  // at least two rounds, a power of two
constexpr int kCmcThreads = (kCmcWaves + 1) * 64;
constexpr int kCmcFirst = 63;  // attempts of a trial's first draw; lane 63 draws its uniform
constexpr int kClustersPerLane = kMaxSiteClusters / 64;

struct CmcLds {
  double w[kMaxW];
  uint16_t env[kCmcWaves][64];  // species around p (low byte) and q of each trial
  double de[kCmcWaves];
  double beta[kCmcRing], T[kCmcRing];  // by step modulo kCmcRing; annealing: by wave
  uint32_t p[kCmcWaves], q[kCmcWaves];
  uint8_t ep[kCmcWaves], eq[kCmcWaves];
  uint8_t flag[kCmcWaves], conflict[kCmcWaves];
  int limit;  // annealing: trials of the next round whose temperatures are known
};
constexpr uint8_t kMark = 0x80;  // species codes are below it
enum : uint8_t { kTrialAccepted = 1, kTrialLost = 2 };  // lost: no pair within kMaxPairAttempts

template <bool kLdsOcc, bool kLog>
__global__ __launch_bounds__(kCmcThreads) void CmcKernel(KTables t, CmcDev c, uint64_t ntrials,
                                                         uint64_t trace_base) {
  __shared__ CmcLds L;
  extern __shared__ uint32_t occ_words[];
  const int r = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const bool commit = wave == kCmcWaves;
  for (int i = tid; i < t.nw; i += kCmcThreads) L.w[i] = t.w[i];
  const int n = c.ncell[r];
  const uint64_t N = 4ull * n * n * n;
  uint8_t *occ = c.occ + c.off[r];
  if constexpr (kLdsOcc) {
    const uint32_t *src = reinterpret_cast<const uint32_t *>(occ);
    for (uint64_t i = tid; i < N / 4; i += kCmcThreads) occ_words[i] = src[i];
    occ = reinterpret_cast<uint8_t *>(occ_words);
  }
  uint64_t steps = c.steps[r];
  const uint64_t maxs = c.max_steps[r], seed = c.seed[r];
  const uint32_t rid = c.rid[r];
  uint64_t acc = 0;
  double energy = 0, abse = 0;
  CmcAnneal A{};
  AnnealSchedule sched{};
  LogClock clk;
  uint64_t log_i = 0, ring_i = 0, ring_at = 0;  // records, energies added, ring slot
  if (commit) {
    acc = c.accepted[r];
    energy = c.energy[r];
    abse = c.abs_energy[r];
    if (c.anneal) {
      A = c.anneal[r];
      sched = MakeAnnealSchedule(maxs);
    }
    if constexpr (kLog) {
      clk.L = c.log_every;
      clk.plain = c.anneal != nullptr;
      clk.Reset(steps);
      log_i = c.log_n[r];
      if (lane == 0) c.log_lo[r] = log_i;
      if (c.avg_m) {
        ring_i = c.ring_n[r];
        ring_at = ring_i % c.ring_cap;
      }
    }
  }
  // the ramp's temperature of a step (CanonicalMcAbstract: beta = 1 / kB / T)
  auto ramp_T = [&](uint64_t step) {
    return c.t0[r] + (c.t1[r] - c.t0[r]) * (static_cast<double>(step) / static_cast<double>(maxs));
  };
  // Temperatures and betas of kCmcWaves steps from `step` on (commit wave). Annealing: the temperatures
  // are those of the decay alone, so the round ends with the trial that closes an acceptance window or
  // may reheat.
  auto set_betas = [&](uint64_t step) {
    double T;
    if (c.anneal) {
      T = A.T;
      for (int k = 1; k < kCmcWaves; ++k)
        if (lane >= k) T *= sched.decay;
      const uint64_t trials = A.window_trials + static_cast<uint64_t>(lane) + 1;  // once lane's trial is done
      const uint64_t at = step + static_cast<uint64_t>(lane);
      const bool reheat = A.reheats < 5 && at - A.last_improvement >= sched.trigger &&
                          at - A.last_reheat >= sched.cooldown &&
                          static_cast<double>(A.window_accepts) / static_cast<double>(trials) < 0.05;
      const uint64_t stop = __ballot(lane < kCmcWaves && (trials >= sched.window || reheat));
      if (lane == 0) L.limit = stop ? __builtin_ctzll(stop) + 1 : kCmcWaves;
    } else {
      T = ramp_T(step + static_cast<uint64_t>(lane));
    }
    if (lane < kCmcWaves) {
      const int at = c.anneal ? lane : static_cast<int>((step + lane) & (kCmcRing - 1));
      L.T[at] = T;
      L.beta[at] = 1.0 / kBoltzmann / (c.anneal ? fmax(T, 1e-12) : T);
    }
  };
  // a log record of the step about to be tried (commit wave)
  auto put_log = [&](uint64_t step, double T, double second) {
    if (log_i < c.log_cap && lane == 0) {
      CmcLogRecord &rec = c.log[static_cast<uint64_t>(r) * c.log_cap + log_i];
      rec.steps = step;
      rec.temperature = T;
      rec.energy = energy;
      rec.second = second;
      rec.abs_energy = abse;
      rec.count = ring_i;
    }
    ++log_i;  // counts past the capacity too, so the host can report the loss
  };
  // attempts (and the uniform, in lane 63 of the first draw) of a step, and their coordinates
  uint32_t a = 0, b = 0, xa = 0, xb = 0, a2 = 0, b2 = 0;
  bool dilute = false, second = false;  // second: a2, b2 hold the 64 attempts after the first 63
  double uni = 0.0;
  auto pack = [&](uint32_t site) { return PackSiteXYZ(site, n); };
  auto draw = [&](uint64_t step) {
    const U4 u = Philox4x32_10(seed, step, rid, lane == kCmcFirst ? 0xFFFFFFFEu : 2u * lane + 1u);
    second = dilute;
    if (second) {
      const U4 v = Philox4x32_10(seed, step, rid, 2u * (kCmcFirst + lane) + 1u);
      a2 = static_cast<uint32_t>(MulHi64(Join64(v.x, v.y), N));
      b2 = static_cast<uint32_t>(MulHi64(Join64(v.z, v.w), N));
    }
    a = static_cast<uint32_t>(MulHi64(Join64(u.x, u.y), N));
    b = static_cast<uint32_t>(MulHi64(Join64(u.z, u.w), N));
    xa = pack(a);
    xb = pack(b);
    uni = UnitOpenRight(Join64(u.x, u.y));
  };
  SiteCluster cl[kClustersPerLane];
  int ox = 0, oy = 0, oz = 0;  // the lane's environment offset
  if (commit) {
    set_betas(steps);
  } else {
    draw(steps + wave);
#pragma unroll
    for (int k = 0; k < kClustersPerLane; ++k) cl[k] = DecodeSiteCluster(t, t.site_cl, lane + 64 * k);
    if (lane < kSiteSlots) Unpack(t.site_off[lane], ox, oy, oz);
  }
  __syncthreads();
  uint64_t it = 0;
  bool lost = false;
  int active = kCmcWaves;  // trials of a round
  while (it < ntrials && steps <= maxs) {
    int limit = c.anneal ? L.limit : kCmcWaves;  // read before the commit wave sets the next one
    int win = -1;           // winning attempt of the first draw, -1: of a later one
    uint32_t sp = 0, sq = 0;  // the lane's sites of both environments
    uint64_t seen = 0;        // the lanes whose second attempts were looked at
    if (commit) {
      if (!c.anneal) set_betas(steps + kCmcWaves);  // the next round may start anywhere up to there
    } else if (wave < active) {
      // another wave of the round may have marked a site by now
      uint64_t m = __ballot(lane < kCmcFirst && ((occ[a] ^ occ[b]) & ~kMark) != 0);
      if (m) win = __builtin_ctzll(m);
      uint32_t base = kCmcFirst;
      dilute = !m || (dilute && win >= 8);
      uint32_t ta = a, tb = b, txa = xa, txb = xb;
      if (!m && second) {
        ta = a2;
        tb = b2;
        m = __ballot(((occ[ta] ^ occ[tb]) & ~kMark) != 0);
        base += 64;
        if (m) {
          txa = pack(ta);
          txb = pack(tb);
          seen = (m ^ (m - 1));
          win = kCmcFirst;  // all of the first
        }
      }
      for (; !m && base < kMaxPairAttempts; base += 128) {  // two draws side by side
        uint32_t more[2][2];
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          const U4 u = Philox4x32_10(seed, steps + wave, rid, 2u * (base + 64u * k + lane) + 1u);
          more[k][0] = static_cast<uint32_t>(MulHi64(Join64(u.x, u.y), N));
          more[k][1] = static_cast<uint32_t>(MulHi64(Join64(u.z, u.w), N));
        }
#pragma unroll
        for (int k = 0; k < 2; ++k) {
          if (m) continue;
          ta = more[k][0];
          tb = more[k][1];
          m = __ballot(base + 64u * k + lane < kMaxPairAttempts && ((occ[ta] ^ occ[tb]) & ~kMark) != 0);
        }
        txa = pack(ta);
        txb = pack(tb);
      }
      uint8_t flag = kTrialLost;
      if (m) {
        const int at = __builtin_ctzll(m);
        auto lane_of = [&](uint32_t v) {
          return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), at));
        };
        const uint32_t p = lane_of(ta), q = lane_of(tb);
        const XYZ xp = UnpackSiteXYZ(lane_of(txa)), xq = UnpackSiteXYZ(lane_of(txb));
        sp = SiteNear(xp, n, ox, oy, oz);
        sq = SiteNear(xq, n, ox, oy, oz);
        const int vp = occ[sp] & ~kMark, vq = occ[sq] & ~kMark;
        // lane 0 is the site itself; codes are validated at creation
        const int ep = __builtin_amdgcn_readlane(vp, 0), eq = __builtin_amdgcn_readlane(vq, 0);
        const int S = t.S;
        L.env[wave][lane] = static_cast<uint16_t>((vp < S ? vp : 0) | (vq < S ? vq : 0) << 8);
        // partner slots: the first offset equal to the minimum image
        int slot_p = 64, slot_q = 64;
        const int dx = MinImage(xq.X - xp.X, n), dy = MinImage(xq.Y - xp.Y, n), dz = MinImage(xq.Z - xp.Z, n);
        const int nx = MinImage(xp.X - xq.X, n), ny = MinImage(xp.Y - xq.Y, n), nz = MinImage(xp.Z - xq.Z, n);
        if (dx * dx + dy * dy + dz * dz <= 6) {
          const bool in = lane >= 1 && lane < kSiteSlots;
          const uint64_t mq = __ballot(in && ox == dx && oy == dy && oz == dz);
          const uint64_t mp = __ballot(in && ox == nx && oy == ny && oz == nz);
          if (mq) slot_p = __builtin_ctzll(mq);
          if (mp) slot_q = __builtin_ctzll(mp);
        }
        WaveFence();
        uint32_t e1[kClustersPerLane], e2[kClustersPerLane];
#pragma unroll
        for (int k = 0; k < kClustersPerLane; ++k) {
          e1[k] = L.env[wave][cl[k].o1];
          e2[k] = L.env[wave][cl[k].o2];
        }
        Stage();
        double w[kClustersPerLane][4];  // p's cluster after and before, q's
#pragma unroll
        for (int k = 0; k < kClustersPerLane; ++k) {
          const int rest_p = cl[k].base + (e1[k] & 255) * cl[k].k1 + (e2[k] & 255) * cl[k].k2;
          const int rest_q = cl[k].base + (e1[k] >> 8) * cl[k].k1 + (e2[k] >> 8) * cl[k].k2;
          const int at_p = ep * cl[k].kx, at_q = eq * cl[k].kx;
          w[k][0] = L.w[rest_p + at_q];
          w[k][1] = L.w[rest_p + at_p];
          w[k][2] = L.w[rest_q + at_p];
          w[k][3] = L.w[rest_q + at_q];
        }
        Stage();
        double de = 0.0;
        if (slot_p < 64 || slot_q < 64) {  // clusters with both sites keep their species
#pragma unroll
          for (int k = 0; k < kClustersPerLane; ++k) {
            if (cl[k].r1 == slot_p || cl[k].r2 == slot_p) w[k][0] = w[k][1] = 0.0;
            if (cl[k].r1 == slot_q || cl[k].r2 == slot_q) w[k][2] = w[k][3] = 0.0;
          }
        }
#pragma unroll
        for (int k = 0; k < kClustersPerLane; ++k)  // lanes past the last cluster add w - w
          de += (w[k][0] - w[k][1]) + (w[k][2] - w[k][3]);
        de = WaveSum(de);
        const double u = ReadLane(uni, kCmcFirst);
        const bool accept = de < 0 || u < exp(-de * L.beta[c.anneal ? wave : (steps + wave) & (kCmcRing - 1)]);
        flag = accept ? kTrialAccepted : 0;
        if (lane == 0) {
          L.de[wave] = de;
          L.p[wave] = p;
          L.q[wave] = q;
          L.ep[wave] = static_cast<uint8_t>(ep);
          L.eq[wave] = static_cast<uint8_t>(eq);
          if (accept) {
            occ[p] = static_cast<uint8_t>(ep) | kMark;
            occ[q] = static_cast<uint8_t>(eq) | kMark;
          }
        }
      }
      if (lane == 0) L.flag[wave] = flag;
    }
    __syncthreads();
    const int slot = lane < kCmcWaves ? lane : 0;
    const uint8_t flag = L.flag[slot];
    const uint32_t tp = L.p[slot], tq = L.q[slot];
    const bool swap = lane < active && (flag & kTrialAccepted);
    const uint64_t accepted = __ballot(swap);
    const uint64_t lost_at = __ballot(lane < active && (flag & kTrialLost));
    if (lost_at & 1) {  // every thread sees the same flags
      lost = true;
      if (commit && swap) {
        occ[tp] = L.ep[slot];
        occ[tq] = L.eq[slot];
      }
      break;
    }
    limit = min(limit, active);
    if (ntrials - it < static_cast<uint64_t>(limit)) limit = static_cast<int>(ntrials - it);
    if (maxs - steps < static_cast<uint64_t>(limit)) limit = static_cast<int>(maxs - steps) + 1;
    if (lost_at) limit = min(limit, __builtin_ctzll(lost_at));  // tried again as a round's first
    int adv = limit;
    if (accepted & ((1ull << (limit - 1)) - 1)) {  // one before the last: what did the later trials read?
      if (!commit && wave < limit) {
        const uint64_t before = accepted & ((1ull << wave) - 1);
        const uint32_t p = L.p[wave], q = L.q[wave];
        const bool drew = lane <= win, in = lane < kSiteSlots;
        const bool drew2 = (seen >> lane) & 1;
        constexpr int kReads = 6;
        const uint32_t read[kReads] = {drew ? a : p, drew ? b : p, drew2 ? a2 : p, drew2 ? b2 : p, in ? sp : p, in ? sq : p};
        uint8_t v[kReads];
#pragma unroll
        for (int k = 0; k < kReads; ++k) v[k] = occ[read[k]];
        // its own two sites against theirs, its other sites through the marks
        bool hit = lane < wave && swap && (tp == p || tp == q || tq == p || tq == q);
        bool marked = false;
#pragma unroll
        for (int k = 0; k < kReads; ++k) marked |= (v[k] & kMark) != 0 && read[k] != p && read[k] != q;
        if (win < 0 && before) hit = true;
        if (__ballot(marked)) {  // by one of the trials before it?
          for (uint64_t e = before; e; e &= e - 1) {
            const int i = __builtin_ctzll(e);
            const uint32_t pi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(tp), i));
            const uint32_t qi = static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(tq), i));
#pragma unroll
            for (int k = 0; k < kReads; ++k) hit |= read[k] == pi || read[k] == qi;
          }
        }
        const uint64_t mh = __ballot(hit);
        if (lane == 0) L.conflict[wave] = mh ? 1 : 0;
      }
      __syncthreads();
      const uint64_t stop = __ballot(lane < limit && L.conflict[slot]);
      if (stop) adv = __builtin_ctzll(stop);
    }
    active = min(adv == limit ? active + 2 : max(max(adv + 3, active - 2), 4), kCmcWaves);
    if (commit) {
      const double tde = L.de[slot];
      const bool mine = lane < adv && swap;
      if (swap && !mine) {  // not taken this round: the marks go
        occ[tp] = L.ep[slot];
        occ[tq] = L.eq[slot];
      }
      // a taken trial may share a site with one that was not taken (that is what ended the round): its
      // species are written after
      WaveFence();
      if (lane < adv) {
        const uint64_t index = trace_base + it + static_cast<uint64_t>(lane);
        if (index < c.trace_cap) {
          const uint64_t o = static_cast<uint64_t>(r) * c.trace_cap + index;
          c.tr_p[o] = tp;
          c.tr_q[o] = tq;
          c.tr_de[o] = tde;
          c.tr_acc[o] = mine ? 1 : 0;
        }
      }
      if (mine) {  // the accepted trials' sites are disjoint
        if (c.atom) {
          const int64_t o = c.off[r];
          const XYZ xp = ToXYZ32(tp, n), xq = ToXYZ32(tq, n);
          AtomJump(c.atom + o, c.shift + 3 * o, tp, tq, ImageChange(xq.X - xp.X, n),
                   ImageChange(xq.Y - xp.Y, n), ImageChange(xq.Z - xp.Z, n));
        }
        occ[tp] = L.eq[slot];
        occ[tq] = L.ep[slot];
      }
      // energies, records and the schedule in trial order
      const int at0 = static_cast<int>(steps & (kCmcRing - 1));
      if (kLog || c.anneal) {
        for (int j = 0; j < adv; ++j) {
          const uint64_t step = steps + static_cast<uint64_t>(j);
          const bool on = (accepted >> j) & 1;
          if constexpr (kLog) {
            if (c.avg_m) {  // ThermodynamicAveraging::AddEnergy before Dump (CanonicalMcSerial.cpp:45)
              if (lane == 0) c.ring[static_cast<uint64_t>(r) * c.ring_cap + ring_at] = energy;
              if (++ring_at == c.ring_cap) ring_at = 0;
              ++ring_i;
            }
          }
          if (c.anneal) {
            const bool lower = energy < A.lowest - 1e-4;  // Dump (SimulatedAnnealing.cpp:80-97)
            if (lower) A.lowest = energy;
            if constexpr (kLog) {
              if (lower) put_log(step, A.T, A.lowest);
              if (clk.Due(step)) put_log(step, A.T, A.lowest);
            }
          } else if constexpr (kLog) {
            if (clk.Due(step)) put_log(step, L.T[(at0 + j) & (kCmcRing - 1)], 0.0);
          }
          if (on) {
            const double de = ReadLane(tde, j);
            energy += de;
            abse += de;
            ++acc;
          }
          if (c.anneal) AnnealUpdate(A, sched, on, step, energy);
        }
      } else {
        const double taken = mine ? tde : 0.0;
#pragma unroll
        for (int j = 0; j < kCmcWaves; ++j) {
          const double de = ReadLane(taken, j);
          energy += de;
          abse += de;
        }
        acc += __builtin_popcountll(__ballot(mine));
      }
      if (c.anneal) set_betas(steps + static_cast<uint64_t>(adv));
    } else if (wave < active) {
      draw(steps + static_cast<uint64_t>(adv + wave));
    }
    steps += static_cast<uint64_t>(adv);
    it += static_cast<uint64_t>(adv);
    __syncthreads();
  }
  if constexpr (kLdsOcc) {
    __syncthreads();
    uint32_t *dst = reinterpret_cast<uint32_t *>(c.occ + c.off[r]);
    for (uint64_t i = tid; i < N / 4; i += kCmcThreads) dst[i] = occ_words[i];
  }
  if (commit && lane == 0) {
    if (lost) atomicOr(c.error, 2);
    c.steps[r] = steps;
    c.accepted[r] = acc;
    c.energy[r] = energy;
    c.abs_energy[r] = abse;
    if (c.anneal) c.anneal[r] = A;
    if constexpr (kLog) {
      c.log_n[r] = log_i;
      if (c.avg_m) c.ring_n[r] = ring_i;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// CanonicalMcOmp (lmc/mc/src/CanonicalMcOmp.cpp:40-92): rounds of up to K swap trials. A round
// draws its pairs through one attempt stream (attempt a of the round starting at step s0 is
// Philox counter (s0, replica, 2a + 1), redrawn while the species agree); each event takes the
// first pair with neither site within 3NN of (or on) an earlier event's sites, and the 50th
// draw of an event ends the round. All dE are taken on the round's starting occupancy (the
// exclusion keeps them exact), the Metropolis tests of a round are independent of each other
// (uniform of step s: counter (s, replica, 0xFFFFFFFE)), and the accepted swaps touch disjoint
// sites. A new round starts only while steps <= maximum_steps; a started round runs to its end,
// across launches if need be (the round is kept in c.omp_*).
//
// One 1024-thread workgroup per replica (the canonical workloads have few replicas, so a CU
// each; 16 waves hide the phases' latencies). Per round:
//   draw   : passes of 1024 attempts, one per thread, species checked in parallel; the first valid
//            attempts of a pass (24 more than events are wanted: a few meet another one) ranked by
//            ballots; their pairs, spread evenly over the threads, tested for conflicts; then wave 0
//            takes them in order by ballots (the reference's do/while with its draw count), while wave 1
//            draws the round's Metropolis uniforms;
//   dE     : a wave gathers an environment at a time and notes which sites are not of the replica's
//            most frequent species; eight threads to an environment add those sites' terms and their
//            pairs' (see OmpTables);
//   trials : event lanes test their Metropolis steps in parallel, and the accepted swaps are applied; the
//            energies are added in trial order (and the log records taken) beside the next draw walk.
// Bound by the latency of these phases. 64 replicas of 30^3 cells, 5 at.% solute, 20 000 trials in
// rounds of 64: 15.5 -> 6.6 ms (all site clusters of both sites for every event, conflicts by rows and one
// lane walking the draws and the energies, before); 6^3 cells, 2 000 trials: 12.1 -> 6.5 ms. Two attempts
// to a thread: 0.88 -> 0.72 ms at 1 at.%, 2 000 trials.
constexpr int kOmpThreads = 1024;
constexpr int kOmpMaxK = 64;
constexpr int kOmpPass = kOmpThreads;          // attempts per draw pass
constexpr int kOmpMaxValid = 128;              // valid attempts resolved per pass
constexpr int kOmpSpare = 24;
constexpr int kOmpShare = kOmpThreads / (2 * kOmpMaxK);  // threads per environment
static_assert(kOmpShare == 8 && kOmpMaxK + kOmpSpare <= kOmpMaxValid, "");

struct OmpDraw {  // one draw pass: its valid attempts in attempt order
  uint32_t va[kOmpMaxValid], vb[kOmpMaxValid], xa[kOmpMaxValid], xb[kOmpMaxValid];
  uint32_t conf[kOmpMaxValid][kOmpMaxValid / 32];  // bit j: conflicts with valid attempt j
  uint32_t excl[kOmpMaxValid];                     // meets an earlier pass's event
  int vidx[kOmpMaxValid];
};

// The cluster sum of a centre species x over an environment, over the sites that are not of the
// reference species r only: E(x) = base(x) + sum f1[shell][x][c] + sum over their pairs of
// f2[label][x][c][c'], with g[label][x][c] = w3(x, c, r) - w3(x, r, r),
//   f2 = (w3(x, c, c') - w3(x, c, r)) - g(x, c'), f1 = w2(x, c) - w2(x, r) + sum of g over the sites that
// form a triplet with it. Exact for every composition; the bases of a swap's two sites cancel.
struct OmpTables {
  double f[kMaxW];  // as w: f1 at S, f2 at S + 3 S S
  double g[kMaxW / 4];
  uint64_t with[kSiteSlots];               // the slots that form a triplet with a slot and the centre
  uint8_t label[kSiteSlots][kSiteSlots];   // its label 1..4, 0 for none
  uint8_t shell[kSiteSlots];               // 0..2
};

struct OmpLds {
  OmpTables t;
  int32_t off[kSiteSlots];
  uint8_t env[2 * kOmpMaxK][48];
  uint64_t other[2 * kOmpMaxK];  // slots not of the reference species
  int slot[2 * kOmpMaxK];
  uint32_t ch[2 * kOmpMaxK];  // sites of the round's events so far
  uint32_t p[kOmpMaxK], q[kOmpMaxK], xp[kOmpMaxK], xq[kOmpMaxK];
  uint8_t ep[kOmpMaxK], eq[kOmpMaxK];
  double de[kOmpMaxK], uni[kOmpMaxK], beta[kOmpMaxK];
  int8_t acc[kOmpMaxK];
  OmpDraw d;
  int wave_valid[kOmpThreads / 64];
  int8_t slot_lut[125];  // env slot of offset (dx, dy, dz) in [-2, 2]^3, -1 beyond the 3rd shell
  // round control
  int len, pos, nch, ct, finished, error;
  uint32_t att0;
};

// Tables of reference species ref (all threads; a barrier follows).
__device__ void LoadOmpTables(const KTables &t, OmpLds &O, int ref) {
  const int tid = threadIdx.x, S = t.S, SS = S * S, w3 = S + 3 * SS;
  OmpTables &T = O.t;
  for (int i = tid; i < kSiteSlots * kSiteSlots; i += kOmpThreads) T.label[i / kSiteSlots][i % kSiteSlots] = 0;
  if (tid < kSiteSlots) {
    T.with[tid] = 0;
    T.shell[tid] = 0;
    O.off[tid] = t.site_off[tid];
  }
  if (tid < 125) O.slot_lut[tid] = -1;
  if (tid < kOmpMaxValid) {
    O.d.excl[tid] = 0;
    for (int w = 0; w < kOmpMaxValid / 32; ++w) O.d.conf[tid][w] = 0;
  }
  for (int i = tid; i < 4 * SS; i += kOmpThreads) {
    const int at = w3 + (i / SS) * SS * S + (i % SS) * S + ref, x = i / S % S;
    T.g[i] = t.w[at] - t.w[w3 + (i / SS) * SS * S + (x * S + ref) * S + ref];
  }
  __syncthreads();
  for (int i = tid; i < t.n_site; i += kOmpThreads) {
    const uint32_t d = t.site_cl[i];
    const int label = d & 7, a = (d >> 4) & 63, b = (d >> 10) & 63;
    if (label >= 4) {
      T.label[a][b] = T.label[b][a] = static_cast<uint8_t>(label - 3);
      atomicOr(reinterpret_cast<unsigned long long *>(&T.with[a]), 1ull << b);
      atomicOr(reinterpret_cast<unsigned long long *>(&T.with[b]), 1ull << a);
    } else if (label) {
      T.shell[a] = static_cast<uint8_t>(label - 1);
    }
  }
  for (int i = tid; i < 4 * SS * S; i += kOmpThreads) {
    const int l = i / (SS * S), x = i / SS % S, c = i / S % S, e = i % S;
    const double *w = t.w + w3 + l * SS * S;
    T.f[w3 + i] = c == ref || e == ref ? 0.0
                                       : (w[(x * S + c) * S + e] - w[(x * S + c) * S + ref]) -
                                             T.g[l * SS + x * S + e];
  }
  if (tid >= 1 && tid < kSiteSlots) {
    int x, y, z;
    Unpack(O.off[tid], x, y, z);
    O.slot_lut[(x + 2) * 25 + (y + 2) * 5 + (z + 2)] = static_cast<int8_t>(tid);
  }
  __syncthreads();
  for (int i = tid; i < 3 * SS; i += kOmpThreads) {
    const int sh = i / SS;
    int at = 1;  // a slot of that shell; all of them have the same triplets
    while (T.shell[at] != sh) ++at;
    double v = t.w[S + i] - t.w[S + sh * SS + (i / S % S) * S + ref];
    for (int b = 1; b < kSiteSlots; ++b)
      if (T.label[at][b]) v += T.g[(T.label[at][b] - 1) * SS + i % SS];
    T.f[S + i] = v;
  }
  __syncthreads();
}

// Whether site b lies on site a or in its 1st-3rd neighbour shells (squared minimum-image
// distance at most 6 in (a/2)^2; FCC distances are even).
__device__ __forceinline__ bool Near(const XYZ &a, const XYZ &b, int n) {
  const int m = 2 * n;
  const int dx = abs(b.X - a.X), dy = abs(b.Y - a.Y), dz = abs(b.Z - a.Z);
  const int x = min(dx, m - dx), y = min(dy, m - dy), z = min(dz, m - dz);
  return x * x + y * y + z * z <= 6;
}

// Metropolis uniforms and ramp betas of the round's events, the first at step s0 (one wave).
__device__ __forceinline__ void OmpDrawTests(const CmcDev &c, OmpLds &O, int r, uint64_t s0, uint64_t maxs, int K) {
  const int e = threadIdx.x & 63;
  if (e >= K) return;
  const uint64_t step = s0 + static_cast<uint64_t>(e);
  O.uni[e] = TrialUniform(c, r, step);
  const double T = c.t0[r] + (c.t1[r] - c.t0[r]) * (static_cast<double>(step) / static_cast<double>(maxs));
  O.beta[e] = 1.0 / kBoltzmann / T;
}

// The round starting at step s0: pairs, environments, partner slots and dE into O (all threads). Wave 2
// calls add_sums, the sums of the trials before it, beside the draw walk.
template <typename Sums>
__device__ __forceinline__ void BuildOmpRound(const KTables &t, const CmcDev &c, OmpLds &O, int r, uint64_t s0, uint64_t maxs,
                              const uint8_t *occ, uint64_t N, int n, int K, int ref, int &per_thread,
                              const Sums &add_sums) {
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  OmpDraw &D = O.d;
  if (tid == 0) {
    O.len = 0;
    O.nch = 0;
    O.ct = 0;
    O.finished = 0;
    O.att0 = 0;
  }
  __syncthreads();
  bool first = true;
  while (!O.finished) {
    // thread t holds attempts t, or 2 t and 2 t + 1
    const int per = per_thread;
    uint32_t a[2], b[2];
    bool valid[2] = {false, false};
    uint64_t m[2] = {0, 0};
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (k >= per) continue;
      const U4 u4 = Philox4x32_10(c.seed[r], s0, c.rid[r],
                                  2u * (O.att0 + static_cast<uint32_t>(per * tid + k)) + 1u);
      a[k] = static_cast<uint32_t>(MulHi64(Join64(u4.x, u4.y), N));
      b[k] = static_cast<uint32_t>(MulHi64(Join64(u4.z, u4.w), N));
      valid[k] = occ[a[k]] != occ[b[k]];
      m[k] = __ballot(valid[k]);
    }
    if (lane == 0) O.wave_valid[wave] = __builtin_popcountll(m[0]) + __builtin_popcountll(m[1]);
    __syncthreads();
    // valid attempts of the waves before this one, and in all (a running sum over each row of 16 lanes)
    int run = O.wave_valid[lane & 15];
    run += __builtin_amdgcn_update_dpp(0, run, 0x111, 0xF, 0xF, true);
    run += __builtin_amdgcn_update_dpp(0, run, 0x112, 0xF, 0xF, true);
    run += __builtin_amdgcn_update_dpp(0, run, 0x114, 0xF, 0xF, true);
    run += __builtin_amdgcn_update_dpp(0, run, 0x118, 0xF, 0xF, true);
    const int total = __builtin_amdgcn_readlane(run, 15);
    const uint64_t lower = (1ull << lane) - 1;
    int u = (wave ? __builtin_amdgcn_readlane(run, wave - 1) : 0) + __builtin_popcountll(m[0] & lower) +
            __builtin_popcountll(m[1] & lower);
    const int len0 = O.len, nch0 = O.nch;
    const int cap = K - len0 + kOmpSpare;  // at most kOmpMaxValid
    const int nv = total < cap ? total : cap;
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      if (valid[k] && u < nv) {
        D.va[u] = a[k];
        D.vb[u] = b[k];
        D.xa[u] = PackSiteXYZ(a[k], n);
        D.xb[u] = PackSiteXYZ(b[k], n);
        D.vidx[u] = per * tid + k;
      }
      u += valid[k] ? 1 : 0;
    }
    __syncthreads();
    if (nv > 0) {
      const float inv = 1.0f / static_cast<float>(nv);
      auto meet = [&](const XYZ &s, int v) {
        return Near(s, UnpackSiteXYZ(D.xa[v]), n) || Near(s, UnpackSiteXYZ(D.xb[v]), n);
      };
      // every pair of attempts once: (v, v + d mod nv) for d up to half way round
      for (int i = tid; i < nv * (nv / 2); i += kOmpThreads) {
        const int d = static_cast<int>((i + 0.5f) * inv), v = i - d * nv;  // i < 2^13: exact
        const int w = v + d + 1 >= nv ? v + d + 1 - nv : v + d + 1;
        if (meet(UnpackSiteXYZ(D.xa[v]), w) || meet(UnpackSiteXYZ(D.xb[v]), w)) {
          const int lo = min(v, w);
          atomicOr(&D.conf[max(v, w)][lo >> 5], 1u << (lo & 31));
        }
      }
      for (int i = tid; i < nv * nch0; i += kOmpThreads) {  // against the events of earlier passes
        const int j = static_cast<int>((i + 0.5f) * inv), v = i - j * nv;  // i < 2^14: exact
        if (meet(UnpackSiteXYZ(O.ch[j]), v)) D.excl[v] = 1;
      }
    }
    __syncthreads();
    if (wave == 0) {
      // The reference's draw loop over the pass's valid attempts, in order: an attempt is taken
      // unless it meets an earlier pass's event or conflicts with an attempt taken before it.
      // Lane l decides attempts l and l + 64 as soon as every earlier attempt it conflicts with
      // is decided (ballots; the chains of conflicts are short), then the draw count and K cut
      // the taken set, and the taken attempts become the next events.
      const int v0 = lane, v1 = lane + 64;
      const uint64_t c0 = v0 < nv ? D.conf[v0][0] | (static_cast<uint64_t>(D.conf[v0][1]) << 32) : 0;
      const uint64_t c1lo = v1 < nv ? D.conf[v1][0] | (static_cast<uint64_t>(D.conf[v1][1]) << 32) : 0;
      const uint64_t c1hi = v1 < nv ? D.conf[v1][2] | (static_cast<uint64_t>(D.conf[v1][3]) << 32) : 0;
      bool d0 = v0 >= nv || D.excl[v0] != 0, d1 = v1 >= nv || D.excl[v1] != 0;
      bool a0 = false, a1 = false;
      uint64_t dlo = __ballot(d0), dhi = __ballot(d1), alo = 0, ahi = 0;
      while (~dlo | ~dhi) {
        if (!d0 && !(c0 & ~dlo)) {
          d0 = true;
          a0 = !(c0 & alo);
        }
        if (!d1 && !(c1lo & ~dlo) && !(c1hi & ~dhi)) {
          d1 = true;
          a1 = !(c1lo & alo) && !(c1hi & ahi);
        }
        dlo = __ballot(d0);
        dhi = __ballot(d1);
        alo = __ballot(a0);
        ahi = __ballot(a1);
      }
      // An event's draws: from the taken attempt before it (the first one's go on from the pass before).
      // The 50th draw of an event ends the round, and so does event K.
      const uint64_t below = (1ull << lane) - 1, b0 = alo & below, b1 = ahi & below;
      auto top = [](uint64_t v) { return 63 - __builtin_clzll(v); };
      const int ct = O.ct;
      const int n0 = b0 ? v0 - top(b0) : ct + v0 + 1;
      const int n1 = b1 ? lane - top(b1) : alo ? v1 - top(alo) : ct + v1 + 1;
      const uint64_t late0 = __ballot(a0 && n0 >= 50), late1 = __ballot(a1 && n1 >= 50);
      const int cut = late0 ? __builtin_ctzll(late0) : late1 ? 64 + __builtin_ctzll(late1) : kOmpMaxValid;
      const int e0 = len0 + __builtin_popcountll(b0);
      const int e1 = len0 + __builtin_popcountll(alo) + __builtin_popcountll(b1);
      const bool t0 = a0 && v0 < cut && e0 < K, t1 = a1 && v1 < cut && e1 < K;
      auto take = [&](int v, int e) {
        O.p[e] = D.va[v];
        O.q[e] = D.vb[v];
        O.xp[e] = O.ch[2 * e] = D.xa[v];
        O.xq[e] = O.ch[2 * e + 1] = D.xb[v];
      };
      if (t0) take(v0, e0);
      if (t1) take(v1, e1);
      const uint64_t tlo = __ballot(t0), thi = __ballot(t1);
      if (lane == 0) {
        const int len = len0 + __builtin_popcountll(tlo) + __builtin_popcountll(thi);
        const int last = thi ? 64 + top(thi) : tlo ? top(tlo) : -1;
        const int open = last < 0 ? ct + nv : nv - 1 - last;  // draws of the event to come
        bool fin = len == K || cut < kOmpMaxValid || open >= 50;
        O.ct = open;
        O.len = len;
        O.nch = 2 * len;
        // the next pass starts after the last attempt looked at
        O.att0 += total > cap ? static_cast<uint32_t>(D.vidx[nv - 1] + 1)
                                : static_cast<uint32_t>(kOmpPass * per);
        if (!fin && O.att0 >= kMaxPairAttempts) {
          O.error = 1;
          fin = true;
        }
        O.finished = fin ? 1 : 0;
      }
      for (int v = lane; v < kOmpMaxValid; v += 64) {  // for the next pass
        D.excl[v] = 0;
        for (int w = 0; w < kOmpMaxValid / 32; ++w) D.conf[v][w] = 0;
      }
    } else if (wave == 1 && first) {
      OmpDrawTests(c, O, r, s0, maxs, K);
    } else if (wave == 2 && first) {
      add_sums();
    }
    first = false;
    __syncthreads();
    // too few valid attempts in a round's first pass: two to a thread from the next pass on, until one to a
    // thread would do (in a small box it is the conflicts that cost passes, and more attempts would not help)
    if (len0 == 0) {
      const bool few = total < per * (K + 8);
      per_thread = few && (per == 2 || !O.finished) ? 2 : 1;
    }
  }
  const int len = O.len;
  {  // environments, a wave each
    int ox = 0, oy = 0, oz = 0;
    const bool in = lane < kSiteSlots;
    if (in) Unpack(O.off[lane], ox, oy, oz);
#pragma unroll 4
    for (int e2 = wave; e2 < 2 * len; e2 += kOmpThreads / 64) {
      const XYZ x = UnpackSiteXYZ(e2 & 1 ? O.xq[e2 >> 1] : O.xp[e2 >> 1]);
      const int v = in ? occ[SiteNear(x, n, ox, oy, oz)] : ref;
      const int code = v < t.S ? v : 0;  // codes are validated at creation
      const uint64_t m = __ballot(lane > 0 && code != ref && in);
      if (in) O.env[e2][lane] = static_cast<uint8_t>(code);
      if (lane == 0) {
        O.other[e2] = m;
        (e2 & 1 ? O.eq : O.ep)[e2 >> 1] = static_cast<uint8_t>(v);
      }
    }
    if (tid < 2 * len) {  // partner slots
      const XYZ xp = UnpackSiteXYZ(O.xp[tid >> 1]), xq = UnpackSiteXYZ(O.xq[tid >> 1]);
      const XYZ &p = (tid & 1) ? xq : xp, &q = (tid & 1) ? xp : xq;
      const int dx = MinImage(q.X - p.X, n), dy = MinImage(q.Y - p.Y, n), dz = MinImage(q.Z - p.Z, n);
      const bool near = dx >= -2 && dx <= 2 && dy >= -2 && dy <= 2 && dz >= -2 && dz <= 2;
      O.slot[tid] = near ? O.slot_lut[(dx + 2) * 25 + (dy + 2) * 5 + (dz + 2)] : -1;
    }
  }
  __syncthreads();
  {  // dE: thread g of an environment adds the terms of the sites in slots g, g + 8, ...
    const int e2 = tid / kOmpShare, g = tid % kOmpShare, S = t.S, SS = S * S;
    double v = 0.0;
    if (e2 < 2 * len) {
      const uint8_t *env = O.env[e2];
      const int eo = env[0], en = O.env[e2 ^ 1][0], skip = O.slot[e2];
      const OmpTables &T = O.t;
      uint64_t other = O.other[e2];
      if (skip >= 0) other &= ~(1ull << skip);  // clusters with both sites keep their species
      for (uint64_t i = other & (0x0101010101010101ull << g); i; i &= i - 1) {
        const int a = __builtin_ctzll(i), ca = env[a];
        const double *f1 = T.f + S + T.shell[a] * SS + ca;
        v += f1[en * S] - f1[eo * S];
        if (skip >= 0 && T.label[a][skip]) {
          const double *h = T.g + (T.label[a][skip] - 1) * SS + ca;
          v -= h[en * S] - h[eo * S];
        }
        const double *f2 = T.f + S + 3 * SS + ca * S;
        for (uint64_t j = other & T.with[a] & ((~0ull << a) << 1); j;) {  // four pairs' loads side by side
          int at[4];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            const int b = j ? __builtin_ctzll(j) : a;
            const int l = T.label[a][b], e = env[b];
            at[k] = j ? (l - 1) * SS * S + e : ref;  // past the last pair: a term of the reference, zero
            j &= j - 1;
          }
          double w[4][2];
#pragma unroll
          for (int k = 0; k < 4; ++k) {
            w[k][0] = f2[at[k] + en * SS];
            w[k][1] = f2[at[k] + eo * SS];
          }
#pragma unroll
          for (int k = 0; k < 4; ++k) v += w[k][0] - w[k][1];
        }
      }
    }
    v += RowShr<1>(v);
    v += RowShr<2>(v);
    v += RowShr<4>(v);  // lanes 7 and 15 of a row: the sums of its environments
    v += RowShr<8>(v);
    if ((lane & 15) == 15 && e2 < 2 * len) {
      const int e = e2 >> 1;
      const int64_t o = static_cast<int64_t>(r) * c.omp_k + e;
      O.de[e] = v;
      c.omp_p[o] = O.p[e];
      c.omp_q[o] = O.q[e];
      c.omp_de[o] = v;
    }
  }
  if (tid == 0) O.pos = 0;
  __syncthreads();
}

template <bool kLdsOcc, bool kLog>
__global__ __launch_bounds__(kOmpThreads) void CmcOmpKernel(KTables t, CmcDev c,
                                                            uint64_t ntrials,
                                                            uint64_t trace_base) {
  __shared__ OmpLds O;
  __shared__ uint64_t s_steps;
  extern __shared__ uint32_t occ_words[];
  const int r = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int n = c.ncell[r], ref = c.omp_ref[r];
  LoadOmpTables(t, O, ref);
  const uint64_t N = 4ull * n * n * n;
  const int K = c.omp_k;
  uint8_t *occ = c.occ + c.off[r];
  if constexpr (kLdsOcc) {
    const uint32_t *src = reinterpret_cast<const uint32_t *>(occ);
    for (uint64_t i = tid; i < N / 4; i += kOmpThreads) occ_words[i] = src[i];
    occ = reinterpret_cast<uint8_t *>(occ_words);
  }
  const uint64_t maxs = c.max_steps[r];
  uint64_t acc = 0, log_i = 0, ring_i = 0, ring_at = 0;
  double energy = 0, abse = 0;
  LogClock clk;
  const bool sums = (tid >> 6) == 2;  // the wave that keeps the sums (the records: its first lane)
  if (sums) {
    acc = c.accepted[r];
    energy = c.energy[r];
    abse = c.abs_energy[r];
  }
  if (tid == 0) {
    s_steps = c.steps[r];
    O.len = c.omp_len[r];
    O.pos = c.omp_pos[r];
    O.error = 0;
  }
  if (sums && lane == 0) {
    if constexpr (kLog) {
      clk.L = c.log_every;
      clk.Reset(c.steps[r]);
      log_i = c.log_n[r];
      c.log_lo[r] = log_i;
      if (c.avg_m) {
        ring_i = c.ring_n[r];
        ring_at = ring_i % c.ring_cap;
      }
    }
  }
  __syncthreads();
  // a round left by the previous launch: its pairs and dE, species and coordinates again (its
  // untried sites are untouched by the swaps tried so far)
  if (O.pos < O.len) {
    for (int e = tid; e < O.len; e += kOmpThreads) {
      const int64_t o = static_cast<int64_t>(r) * K + e;
      O.p[e] = static_cast<uint32_t>(c.omp_p[o]);
      O.q[e] = static_cast<uint32_t>(c.omp_q[o]);
      O.de[e] = c.omp_de[o];
      O.xp[e] = PackSiteXYZ(O.p[e], n);
      O.xq[e] = PackSiteXYZ(O.q[e], n);
      O.ep[e] = occ[O.p[e]];
      O.eq[e] = occ[O.q[e]];
    }
    if (tid < 64) OmpDrawTests(c, O, r, s_steps - static_cast<uint64_t>(O.pos), maxs, K);
    __syncthreads();
  }
  // Energies of the trials sum_pos .. sum_pos + sum_m - 1 of the round, tried from step sum_step on, in
  // trial order, with the averaging ring and log records (the wave of the sums).
  int sum_pos = 0, sum_m = 0;
  uint64_t sum_step = 0;
  auto add_sums = [&] {
    if constexpr (kLog) {
      if (lane == 0) {
#pragma unroll 4
        for (int e = sum_pos; e < sum_pos + sum_m; ++e) {
          const uint64_t step = sum_step + static_cast<uint64_t>(e - sum_pos);
          if (c.avg_m) {
            c.ring[static_cast<uint64_t>(r) * c.ring_cap + ring_at] = energy;
            if (++ring_at == c.ring_cap) ring_at = 0;
            ++ring_i;
          }
          if (clk.Due(step)) {
            if (log_i < c.log_cap) {
              CmcLogRecord &rec = c.log[static_cast<uint64_t>(r) * c.log_cap + log_i];
              rec.steps = step;
              rec.temperature =
                  c.t0[r] + (c.t1[r] - c.t0[r]) * (static_cast<double>(step) / static_cast<double>(maxs));
              rec.energy = energy;
              rec.second = 0.0;
              rec.abs_energy = abse;
              rec.count = ring_i;
            }
            ++log_i;
          }
          if (O.acc[e]) {
            energy += O.de[e];
            abse += O.de[e];
            ++acc;
          }
        }
      }
    } else {
      const bool on = lane >= sum_pos && lane < sum_pos + sum_m && O.acc[lane];
      const double taken = on ? O.de[lane] : 0.0;
      acc += __builtin_popcountll(__ballot(on));
#pragma unroll 16
      for (int e = 0; e < kOmpMaxK; ++e) {
        const double de = ReadLane(taken, e);
        energy += de;
        abse += de;
      }
    }
    sum_m = 0;
  };
  uint64_t it = 0;
  int per_thread = 1;
  while (it < ntrials) {
    // every thread reads the round state before BuildOmpRound's first lane rewrites it
    const bool need = O.pos == O.len;
    const bool stop = need && s_steps > maxs;
    __syncthreads();
    if (stop) break;
    if (need) {
      BuildOmpRound(t, c, O, r, s_steps, maxs, occ, N, n, K, ref, per_thread, add_sums);
      if (O.error) break;
    }
    const int pos = O.pos;
    const uint64_t left = ntrials - it;
    const int m = static_cast<uint64_t>(O.len - pos) < left ? O.len - pos : static_cast<int>(left);
    const uint64_t s0 = s_steps;
    // Metropolis tests of the round's next m events, in parallel
    for (int e = pos + tid; e < pos + m; e += kOmpThreads) {
      const double de = O.de[e];
      const bool a = de < 0 || O.uni[e] < exp(-de * O.beta[e]);
      O.acc[e] = a ? 1 : 0;
      const uint64_t ti = trace_base + it + static_cast<uint64_t>(e - pos);
      if (ti < c.trace_cap) {
        const uint64_t o = static_cast<uint64_t>(r) * c.trace_cap + ti;
        c.tr_p[o] = O.p[e];
        c.tr_q[o] = O.q[e];
        c.tr_de[o] = de;
        c.tr_acc[o] = a ? 1 : 0;
      }
    }
    __syncthreads();
    sum_pos = pos;
    sum_m = m;
    sum_step = s0;
    if (tid == 0) {
      s_steps = s0 + static_cast<uint64_t>(m);
      O.pos = pos + m;
    }
    // the accepted swaps (disjoint sites)
    const int e = tid - kOmpThreads / 2;  // off wave 0
    if (e >= pos && e < pos + m && O.acc[e]) {
      const uint32_t p = O.p[e], q = O.q[e];
      if (c.atom) {
        const int64_t o = c.off[r];
        const XYZ xp = UnpackSiteXYZ(O.xp[e]), xq = UnpackSiteXYZ(O.xq[e]);
        AtomJump(c.atom + o, c.shift + 3 * o, p, q, ImageChange(xq.X - xp.X, n),
                 ImageChange(xq.Y - xp.Y, n), ImageChange(xq.Z - xp.Z, n));
      }
      occ[p] = O.eq[e];
      occ[q] = O.ep[e];
    }
    it += static_cast<uint64_t>(m);
    __syncthreads();
  }
  if constexpr (kLdsOcc) {
    __syncthreads();
    uint32_t *dst = reinterpret_cast<uint32_t *>(c.occ + c.off[r]);
    for (uint64_t i = tid; i < N / 4; i += kOmpThreads) dst[i] = occ_words[i];
  }
  if (sums) add_sums();
  if (tid == 0) {
    if (O.error) atomicOr(c.error, 2);
    c.steps[r] = s_steps;
    c.omp_len[r] = O.len;
    c.omp_pos[r] = O.pos;
  }
  if (sums && lane == 0) {
    c.accepted[r] = acc;
    c.energy[r] = energy;
    c.abs_energy[r] = abse;
    if constexpr (kLog) {
      c.log_n[r] = log_i;
      if (c.avg_m) c.ring_n[r] = ring_i;
    }
  }
}

// The most frequent species of each replica (the lowest code of equal ones): the reference of its rounds.
// Swaps keep the composition, so every launch of a run has the same one.
__global__ __launch_bounds__(kOmpThreads) void CmcReferenceKernel(CmcDev c, int S, uint8_t *ref) {
  __shared__ unsigned long long count[kMaxSpecies];
  const int r = blockIdx.x, tid = threadIdx.x;
  if (tid < kMaxSpecies) count[tid] = 0;
  __syncthreads();
  const int n = c.ncell[r];
  const uint64_t N = 4ull * n * n * n;
  const uint8_t *occ = c.occ + c.off[r];
  for (uint64_t base = 0; base < N; base += kOmpThreads) {
    const uint64_t i = base + tid;
    const int v = i < N ? occ[i] : kMaxSpecies;
    for (int s = 0; s < S; ++s) {
      const uint64_t m = __ballot(v == s);
      if ((tid & 63) == 0 && m) atomicAdd(&count[s], static_cast<unsigned long long>(__builtin_popcountll(m)));
    }
  }
  __syncthreads();
  if (tid == 0) {
    int best = 0;
    for (int s = 1; s < S; ++s)
      if (count[s] > count[best]) best = s;
    ref[r] = static_cast<uint8_t>(best);
  }
}

// ThermodynamicAveraging::GetThermodynamicAverage (ThermodynamicAveraging.cpp:25-40) of the log
// records of the last launch: over the last min(avg_m, count) energies of the ring, the mean m
// and sum((e - m) exp(-(e - m) beta)) / sum(exp(-(e - m) beta)) + m, beta = 1 / kB / T of the
// record. Grid (R, G): workgroup (x, y) takes records lo + y, lo + y + G, ... of replica x.
__device__ __forceinline__ double BlockSum256(double v, double *red) {
  v = WaveSum(v);
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  const double s = red[0] + red[1] + red[2] + red[3];
  __syncthreads();
  return s;
}

__global__ __launch_bounds__(kThreads) void CmcAverageKernel(CmcDev c) {
  static_assert(kThreads == 256, "BlockSum256 reduces four waves");
  __shared__ double red[4];
  const int r = blockIdx.x;
  const uint64_t lo = c.log_lo[r];
  const uint64_t hi = c.log_n[r] < c.log_cap ? c.log_n[r] : c.log_cap;
  const double *ring = c.ring + static_cast<uint64_t>(r) * c.ring_cap;
  for (uint64_t i = lo + blockIdx.y; i < hi; i += gridDim.y) {
    CmcLogRecord &rec = c.log[static_cast<uint64_t>(r) * c.log_cap + i];
    const uint64_t cnt = rec.count;
    const uint64_t w = cnt < c.avg_m ? cnt : c.avg_m;  // >= 1: the record's own energy
    const uint64_t first = (cnt - w) % c.ring_cap;
    double sum = 0.0;
    for (uint64_t j = threadIdx.x; j < w; j += kThreads) {
      const uint64_t x = first + j;
      sum += ring[x < c.ring_cap ? x : x - c.ring_cap];
    }
    const double mean = BlockSum256(sum, red) / static_cast<double>(w);
    const double beta = 1.0 / kBoltzmann / rec.temperature;
    double num = 0.0, den = 0.0;
    for (uint64_t j = threadIdx.x; j < w; j += kThreads) {
      const uint64_t x = first + j;
      const double e = ring[x < c.ring_cap ? x : x - c.ring_cap] - mean;
      const double ex = exp(-e * beta);
      num += e * ex;
      den += ex;
    }
    num = BlockSum256(num, red);
    den = BlockSum256(den, red);
    if (threadIdx.x == 0) rec.second = num / den + mean;
  }
}

// ---------------------------------------------------------------------------------------------
// EnergyPredictor::GetEncode / GetEnergy (EnergyPredictor.cpp:40-96, :173-177): ordered cluster
// counts over the whole lattice, integer histogram per replica, then theta . (count / N).
__constant__ int8_t c_nn1[12][3] = {{1, 1, 0},  {1, -1, 0},  {-1, 1, 0}, {-1, -1, 0},
                                    {1, 0, 1},  {1, 0, -1},  {-1, 0, 1}, {-1, 0, -1},
                                    {0, 1, 1},  {0, 1, -1},  {0, -1, 1}, {0, -1, -1}};
__constant__ int8_t c_nn2[6][3] = {{2, 0, 0}, {-2, 0, 0}, {0, 2, 0}, {0, -2, 0}, {0, 0, 2}, {0, 0, -2}};
__constant__ int8_t c_nn3[24][3] = {
    {2, 1, 1},  {2, 1, -1},  {2, -1, 1},  {2, -1, -1},  {-2, 1, 1},  {-2, 1, -1},
    {-2, -1, 1}, {-2, -1, -1}, {1, 2, 1},  {1, 2, -1},   {-1, 2, 1},  {-1, 2, -1},
    {1, -2, 1},  {1, -2, -1},  {-1, -2, 1}, {-1, -2, -1}, {1, 1, 2},  {1, -1, 2},
    {-1, 1, 2},  {-1, -1, 2},  {1, 1, -2},  {1, -1, -2},  {-1, 1, -2}, {-1, -1, -2}};

__device__ __forceinline__ int Code(uint8_t v, int S) { return v < S ? v : 0; }

__device__ __forceinline__ int Shell(int x, int y, int z) {
  const int r2 = x * x + y * y + z * z;
  return r2 == 2 ? 1 : r2 == 4 ? 2 : r2 == 6 ? 3 : 0;
}

// Index of a pair (shell 1..3) or triplet (label 4..7) of species in a count row: its ECI, or past the
// ECIs for clusters with two or more vacancies, which have none.
__device__ __forceinline__ int PairIndex(const KTables &t, int shell, int a, int b) {
  if (a == t.x_code && b == t.x_code) return t.n_eci + shell - 1;
  return t.eci2[((shell - 1) * t.S + a) * t.S + b];
}
__device__ __forceinline__ int TripletIndex(const KTables &t, int label, int a, int b, int c) {
  const int x = (a == t.x_code) + (b == t.x_code) + (c == t.x_code);
  if (x >= 2) {  // the third species
    const int other = a != t.x_code ? a : b != t.x_code ? b : c;
    return t.n_eci + 3 + (label - 4) * t.S + other;
  }
  return t.eci3[(label - 4) * t.S * t.S * t.S + (a * t.S + b) * t.S + c];
}
// a count row: at most 561 ECIs (8 species), 3 pairs and 4 * 8 triplets without one
constexpr int kMaxCountRow = 640;

// The species that the counts leave out: the most frequent one of 64 sites spread over the box (any
// choice is exact). Called by a whole wave.
__device__ __forceinline__ int ReferenceSpecies(const uint8_t *o, uint64_t N, int S) {
  const int v = Code(o[(static_cast<uint64_t>(threadIdx.x & 63) * N) >> 6], S);
  int ref = 0, most = -1;
  for (int c = 0; c < S; ++c) {
    const int n = __builtin_popcountll(__ballot(v == c));
    if (n > most) {
      most = n;
      ref = c;
    }
  }
  return ref;
}

// The 21 neighbour offsets that follow the site in (x, y, z) order: each pair and each triplet of the box
// is seen once, from its first member. label[a][c]: the label of the triplet (site, a, c > a), 0 for none.
// The ordered enumeration meets a pair twice, a triplet of label 4 six times, of 5 and 6 twice (from
// either end of its two first-neighbour bonds), of 7 once.
constexpr int kHalf = 21;
struct NeighbourTables {
  int8_t off[kHalf][3], shell[kHalf];
  uint8_t label[kHalf][kHalf];
  uint32_t with[kHalf];  // the c with a label
};
__host__ __device__ constexpr int ShellOfOffset(int x, int y, int z) {
  const int r2 = x * x + y * y + z * z;
  return r2 == 2 ? 1 : r2 == 4 ? 2 : r2 == 6 ? 3 : 0;
}
constexpr NeighbourTables MakeNeighbourTables() {
  NeighbourTables n{};
  int at = 0;
  for (int x = 0; x <= 2; ++x)
    for (int y = -2; y <= 2; ++y)
      for (int z = -2; z <= 2; ++z)
        if (ShellOfOffset(x, y, z) && (x > 0 || y > 0 || (y == 0 && z > 0))) {
          n.off[at][0] = static_cast<int8_t>(x);
          n.off[at][1] = static_cast<int8_t>(y);
          n.off[at][2] = static_cast<int8_t>(z);
          n.shell[at++] = static_cast<int8_t>(ShellOfOffset(x, y, z));
        }
  for (int a = 0; a < kHalf; ++a)
    for (int c = a + 1; c < kHalf; ++c) {
      const int third = ShellOfOffset(n.off[c][0] - n.off[a][0], n.off[c][1] - n.off[a][1], n.off[c][2] - n.off[a][2]);
      int times[4] = {0, 0, 0, 0};
      ++times[n.shell[a]];
      ++times[n.shell[c]];
      ++times[third];
      const int label = times[0] ? 0 : times[1] == 3 ? 4 : times[1] == 2 ? (times[2] ? 5 : 6)
                        : times[1] == 1 && times[2] == 1 ? 7 : 0;
      n.label[a][c] = static_cast<uint8_t>(label);
      if (label) n.with[a] |= 1u << c;
    }
  return n;
}
__constant__ NeighbourTables c_nb = MakeNeighbourTables();

// Ordered cluster counts of the clusters without the reference species (EnergyPredictor.cpp:40-96);
// EncodeKernel derives the others. A workgroup lists the non-reference sites of 4 096 at a time, then a
// thread takes a listed site: the species of the neighbours that follow it (21 independent byte loads),
// then the pairs and triplets of non-reference ones through bit masks. The histogram has a copy per
// lane (as many as fit), a copy to a bank: atomics of a wave on one counter do not queue.
// Bound by the LDS atomics and the gathers of the listed sites. 64 boxes of 28^3-32^3 cells, the whole
// call: 4 720 -> 84 us at 5 at.% solute, 2 580 -> 480 us at 75 % (LDS atomics of all 187 ordered clusters
// of every site, on a few hot counters, before).
constexpr int kCountChunk = 4096, kHistWords = 8192;
__global__ __launch_bounds__(kThreads) void TotalCountsKernel(KTables t, const uint8_t *occ,
                                                              const int64_t *off,
                                                              const int32_t *ncell,
                                                              unsigned long long *counts, int row) {
  __shared__ unsigned int hist[kHistWords];
  __shared__ uint16_t list[kCountChunk];
  __shared__ uint16_t eci2[3 * kMaxSpecies * kMaxSpecies], eci3[4 * kMaxSpecies * kMaxSpecies * kMaxSpecies];
  __shared__ uint8_t label[kHalf][kHalf];
  __shared__ uint32_t with[kHalf];
  __shared__ int s_len;
  const int r = blockIdx.x, tid = threadIdx.x, lane = tid & 63;  // grid (R, slices of the box)
  const int n = ncell[r];
  const uint64_t N = 4ull * n * n * n;
  if (blockIdx.y * static_cast<uint64_t>(kCountChunk) >= N) return;
  const uint8_t *o = occ + off[r];
  const int S = t.S;
  const int copies = row <= kHistWords / 32 ? 32 : row <= kHistWords / 16 ? 16 : 8;  // row <= 640
  for (int i = tid; i < row * copies; i += kThreads) hist[i] = 0;
  for (int i = tid; i < 3 * S * S; i += kThreads)
    eci2[i] = static_cast<uint16_t>(PairIndex(t, i / (S * S) + 1, i / S % S, i % S) * copies);
  for (int i = tid; i < 4 * S * S * S; i += kThreads)
    eci3[i] = static_cast<uint16_t>(TripletIndex(t, i / (S * S * S) + 4, i / (S * S) % S, i / S % S, i % S) * copies);
  for (int i = tid; i < kHalf * kHalf; i += kThreads) label[i / kHalf][i % kHalf] = c_nb.label[i / kHalf][i % kHalf];
  if (tid < kHalf) with[tid] = c_nb.with[tid];
  unsigned int *mine = hist + (lane & (copies - 1));
  const int ref = ReferenceSpecies(o, N, S);
  const int64_t plane = 2ll * n * n;
  for (uint64_t base = blockIdx.y * static_cast<uint64_t>(kCountChunk); base < N;
       base += gridDim.y * static_cast<uint64_t>(kCountChunk)) {
    if (tid == 0) s_len = 0;
    __syncthreads();
    uint8_t v[kCountChunk / kThreads];
#pragma unroll
    for (int u = 0; u < kCountChunk / kThreads; ++u) {
      const uint64_t s = base + u * kThreads + tid;
      v[u] = o[s < N ? s : N - 1];
    }
#pragma unroll
    for (int u = 0; u < kCountChunk / kThreads; ++u) {
      const bool on = base + u * kThreads + tid < N && Code(v[u], S) != ref;
      const uint64_t m = __ballot(on);
      int at = 0;
      if (lane == 0 && m) at = atomicAdd(&s_len, __builtin_popcountll(m));
      at = __builtin_amdgcn_readfirstlane(at);
      if (on) list[at + __builtin_popcountll(m & ((1ull << lane) - 1))] = static_cast<uint16_t>(u * kThreads + tid);
    }
    __syncthreads();
    for (int i = tid; i < s_len; i += kThreads) {
      const uint64_t s = base + list[i];
      uint32_t X, Y, Zh;
      if (N <= 0xFFFFFFFFull) {  // 32-bit divisions but for boxes past 1 023 cells
        const uint32_t p = static_cast<uint32_t>(plane), u = static_cast<uint32_t>(s);
        X = u / p;
        Y = (u - X * p) / n;
        Zh = u - X * p - Y * n;
      } else {
        X = static_cast<uint32_t>(s / plane);
        const uint64_t rest = s - X * plane;
        Y = static_cast<uint32_t>(rest / n);
        Zh = static_cast<uint32_t>(rest - static_cast<uint64_t>(Y) * n);
      }
      const uint32_t m = 2 * n, Z = 2 * Zh + ((X + Y) & 1);
      int64_t xs[3];
      uint32_t ys[5], zs[5];  // within a plane
      auto wrap = [&](uint32_t w) { return min(min(w, w + m), w - m); };
#pragma unroll
      for (int d = 0; d < 5; ++d) {
        if (d < 3) xs[d] = wrap(X + d) * plane;
        ys[d] = wrap(Y + d - 2) * n;
        zs[d] = wrap(Z + d - 2) >> 1;
      }
      constexpr NeighbourTables nb = MakeNeighbourTables();
      uint8_t e[kHalf];
#pragma unroll
      for (int j = 0; j < kHalf; ++j) e[j] = o[xs[nb.off[j][0]] + (ys[nb.off[j][1] + 2] + zs[nb.off[j][2] + 2])];
      const int e1 = Code(o[s], S);
      uint32_t other = 0, code[3] = {0, 0, 0};  // the non-reference neighbours; species, 4 bits each
#pragma unroll
      for (int j = 0; j < kHalf; ++j) {
        const uint32_t c = Code(e[j], S);
        other |= static_cast<uint32_t>(c != static_cast<uint32_t>(ref)) << j;
        code[j >> 3] |= c << (4 * (j & 7));
      }
      constexpr uint32_t second = [] {  // bit masks of the shells
        uint32_t w = 0;
        for (int j = 0; j < kHalf; ++j) w |= static_cast<uint32_t>(nb.shell[j] == 2) << j;
        return w;
      }();
      constexpr uint32_t third = [] {
        uint32_t w = 0;
        for (int j = 0; j < kHalf; ++j) w |= static_cast<uint32_t>(nb.shell[j] == 3) << j;
        return w;
      }();
      auto species = [&](int j) {
        const uint32_t w = j < 8 ? code[0] : j < 16 ? code[1] : code[2];
        return static_cast<int>((w >> (4 * (j & 7))) & 15u);
      };
      atomicAdd(&mine[t.eci1[e1] * copies], 1u);
      for (uint32_t b = other; b; b &= b - 1) {
        const int a = __builtin_ctz(b), sh = ((second >> a) & 1) + 2 * ((third >> a) & 1), e2 = species(a);
        atomicAdd(&mine[eci2[(sh * S + e1) * S + e2]], 2u);
        for (uint32_t c = other & with[a]; c; c &= c - 1) {
          const int j = __builtin_ctz(c), l = label[a][j] - 4;
          atomicAdd(&mine[eci3[((l * S + e1) * S + e2) * S + species(j)]], l == 0 ? 6u : l == 3 ? 1u : 2u);
        }
      }
    }
    __syncthreads();
  }
  for (int i = tid; i < row; i += kThreads) {
    unsigned long long sum = 0;
    for (int k = 0; k < copies; ++k) sum += hist[i * copies + ((k + tid) & (copies - 1))];
    if (sum) atomicAdd(&counts[static_cast<int64_t>(r) * row + i], sum);
  }
}

// Membership of site s in the sorted list set[m].
__device__ __forceinline__ bool InSet(const int64_t *set, int m, int64_t s) {
  int lo = 0, hi = m;
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (set[mid] < s) lo = mid + 1;
    else hi = mid;
  }
  return lo < m && set[lo] == s;
}

// EnergyPredictor::GetEncodeOfCluster (EnergyPredictor.cpp:97-172): the ordered cluster counts
// of the sites in set[m] (sorted, unique) whose member sites all lie in the set, enumerated as in
// GetEncode: from every first site, its neighbours, and for 1NN neighbours the triplets closed
// through the second site's 1NN and 2NN shells.
__global__ __launch_bounds__(kThreads) void ClusterCountsKernel(KTables t, const uint8_t *occ, int n,
                                                                const int64_t *set, int m,
                                                                unsigned long long *counts) {
  __shared__ unsigned int hist[kMaxCountRow];
  for (int i = threadIdx.x; i < t.n_eci; i += blockDim.x) hist[i] = 0;
  __syncthreads();
  const int S = t.S;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x) {
    const int64_t s1 = set[i];
    const XYZ c = ToXYZ(s1, n);
    const int e1 = Code(occ[s1], S);
    atomicAdd(&hist[t.eci1[e1]], 1u);
    for (int a = 0; a < 12; ++a) {
      const int ax = c_nn1[a][0], ay = c_nn1[a][1], az = c_nn1[a][2];
      const int64_t s2 = SiteAt(c, n, ax, ay, az);
      if (!InSet(set, m, s2)) continue;
      const int e2 = Code(occ[s2], S);
      atomicAdd(&hist[t.eci2[(0 * S + e1) * S + e2]], 1u);
      for (int b = 0; b < 12; ++b) {
        const int x = ax + c_nn1[b][0], y = ay + c_nn1[b][1], z = az + c_nn1[b][2];
        const int sh = Shell(x, y, z);
        if (!sh) continue;
        const int64_t s3 = SiteAt(c, n, x, y, z);
        if (!InSet(set, m, s3)) continue;
        const int e3 = Code(occ[s3], S);
        atomicAdd(&hist[t.eci3[(sh - 1) * S * S * S + (e1 * S + e2) * S + e3]], 1u);
      }
      for (int b = 0; b < 6; ++b) {
        const int x = ax + c_nn2[b][0], y = ay + c_nn2[b][1], z = az + c_nn2[b][2];
        if (Shell(x, y, z) != 3) continue;
        const int64_t s3 = SiteAt(c, n, x, y, z);
        if (!InSet(set, m, s3)) continue;
        const int e3 = Code(occ[s3], S);
        atomicAdd(&hist[t.eci3[3 * S * S * S + (e1 * S + e2) * S + e3]], 1u);
      }
    }
    for (int a = 0; a < 6; ++a) {
      const int64_t s2 = SiteAt(c, n, c_nn2[a][0], c_nn2[a][1], c_nn2[a][2]);
      if (InSet(set, m, s2)) atomicAdd(&hist[t.eci2[(1 * S + e1) * S + Code(occ[s2], S)]], 1u);
    }
    for (int a = 0; a < 24; ++a) {
      const int64_t s2 = SiteAt(c, n, c_nn3[a][0], c_nn3[a][1], c_nn3[a][2]);
      if (InSet(set, m, s2)) atomicAdd(&hist[t.eci2[(2 * S + e1) * S + Code(occ[s2], S)]], 1u);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < t.n_eci; i += blockDim.x)
    if (hist[i]) atomicAdd(&counts[i], hist[i]);
}

// Number of x in the multiset {a, b} or {a, b, c}.
__device__ __forceinline__ int Times(int x, int a, int b) { return (x == a) + (x == b); }
__device__ __forceinline__ int Times(int x, int a, int b, int c) { return (x == a) + (x == b) + (x == c); }

// The counts with the reference species s from those without it (one wave, c the count row in LDS). Every
// site takes part in the same number of ordered clusters at every position, so with C{..} the ordered
// count of a multiset of species, N sites, z neighbours, and m triplets per site and position:
//   C{s} = N - sum C{a}
//   sum over all pairs of (number of a's) C = 2 z C{a}, which gives C{a, s}; C{s, s} from z N
//   sum over c of (number of c's in {a, b, c}) C{a, b, c} = sum over the position left out of k C{a, b} of
//   the shell between the other two, with k third sites per such pair; this gives C{a, b, s}
//   sum of (number of a's) C = 3 m C{a} gives C{a, s, s}; C{s, s, s} from m N.
__device__ void CompleteCounts(const KTables &t, unsigned long long *c, int s, unsigned long long N) {
  const int S = t.S, lane = threadIdx.x & 63;
  const int z[3] = {12, 6, 24}, m[4] = {48, 24, 48, 24};
  // third sites per pair of positions (1, 2), (2, 3), (1, 3) of a triplet, and the pair's shell
  const int k[4][3] = {{4, 4, 4}, {2, 2, 4}, {4, 4, 2}, {2, 4, 1}};
  const int shell[4][3] = {{1, 1, 1}, {1, 1, 2}, {1, 1, 3}, {1, 2, 3}};
  auto one = [&](int a) -> unsigned long long & { return c[t.eci1[a]]; };
  auto two = [&](int sh, int a, int b) -> unsigned long long & { return c[PairIndex(t, sh, a, b)]; };
  auto three = [&](int l, int a, int b, int d) -> unsigned long long & { return c[TripletIndex(t, 4 + l, a, b, d)]; };
  if (lane == 0) {
    unsigned long long rest = N;
    for (int a = 0; a < S; ++a)
      if (a != s) rest -= one(a);
    one(s) = rest;
  }
  __syncthreads();
  for (int i = lane; i < 3 * S; i += 64) {
    const int sh = i / S + 1, a = i % S;
    if (a == s) continue;
    unsigned long long rest = 2ull * z[sh - 1] * one(a);
    for (int b = 0; b < S; ++b)
      if (b != s) rest -= Times(a, a, b) * two(sh, a, b);
    two(sh, a, s) = rest;
  }
  __syncthreads();
  if (lane < 3) {
    unsigned long long rest = z[lane] * N;
    for (int a = 0; a < S; ++a)
      for (int b = a; b < S; ++b)
        if (!(a == s && b == s)) rest -= two(lane + 1, a, b);
    two(lane + 1, s, s) = rest;
  }
  __syncthreads();
  for (int i = lane; i < 4 * S * S; i += 64) {
    const int l = i / (S * S), a = i / S % S, b = i % S;
    if (a > b || a == s || b == s) continue;
    unsigned long long rest = 0;
    for (int p = 0; p < 3; ++p) rest += k[l][p] * two(shell[l][p], a, b);
    for (int d = 0; d < S; ++d)
      if (d != s) rest -= Times(d, a, b, d) * three(l, a, b, d);
    three(l, a, b, s) = rest;
  }
  __syncthreads();
  for (int i = lane; i < 4 * S; i += 64) {
    const int l = i / S, a = i % S;
    if (a == s) continue;
    unsigned long long rest = 3ull * m[l] * one(a);
    for (int b = 0; b < S; ++b)
      for (int d = b; d < S; ++d)
        if (!(b == s && d == s)) rest -= Times(a, a, b, d) * three(l, a, b, d);
    three(l, a, s, s) = rest;
  }
  __syncthreads();
  if (lane < 4) {
    unsigned long long rest = m[lane] * N;
    for (int a = 0; a < S; ++a)
      for (int b = a; b < S; ++b)
        for (int d = b; d < S; ++d)
          if (!(a == s && b == s && d == s)) rest -= three(lane, a, b, d);
    three(lane, s, s, s) = rest;
  }
  __syncthreads();
}

// The encode count / N_label of each replica (EnergyPredictor.cpp:89-95) and theta . encode; one wave per
// replica, counts in rows of `row`. occ: the counts lack the reference species (null: they are whole).
// Clusters with two vacancies have no ECI and count for the first one.
__global__ __launch_bounds__(64) void EncodeKernel(KTables t, const unsigned long long *counts, int row,
                                                   const uint8_t *occ, const int64_t *off,
                                                   const int32_t *ncell, double *encode, double *energy) {
  __shared__ unsigned long long c[kMaxCountRow];
  __shared__ double x[kMaxCountRow], w[kMaxCountRow];
  const int r = blockIdx.x, lane = threadIdx.x;
  for (int i = lane; i < row; i += 64) c[i] = counts[static_cast<int64_t>(r) * row + i];
  __syncthreads();
  if (occ) {
    const int n = ncell[r];
    const unsigned long long N = 4ull * n * n * n;
    if (n > 0) CompleteCounts(t, c, ReferenceSpecies(occ + off[r], N, t.S), N);
    if (lane == 0)
      for (int i = t.n_eci; i < row; ++i) c[0] += c[i];
    __syncthreads();
  }
  for (int i = lane; i < t.n_eci; i += 64) {
    x[i] = static_cast<double>(c[i]) / t.norm_tot[i];
    w[i] = t.theta[i];
    if (encode) encode[static_cast<int64_t>(r) * t.n_eci + i] = x[i];
  }
  __syncthreads();
  if (energy && lane == 0) {
    double e = 0.0;
    for (int i = 0; i < t.n_eci; ++i) e += w[i] * x[i];
    energy[r] = e;
  }
}

__global__ void ZeroKernel(unsigned long long *p, int64_t n) {
  const int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

}  // namespace

hipError_t LaunchSwapDe(const KTables &t, const uint8_t *occ, const int64_t *off,
                        const int32_t *ncell, const int64_t *pairs, int32_t R, double *de,
                        hipStream_t s) {
  if (R <= 0) return hipSuccess;
  hipLaunchKernelGGL(SwapDeKernel, dim3(R), dim3(kThreads), 0, s, t, occ, off, ncell, pairs, de);
  return hipGetLastError();
}

hipError_t LaunchSiteDe(const KTables &t, const uint8_t *occ, const int64_t *off,
                        const int32_t *ncell, const int64_t *sites, const uint8_t *from,
                        const uint8_t *codes, int32_t R, double *de, hipStream_t s) {
  if (R <= 0) return hipSuccess;
  hipLaunchKernelGGL(SiteDeKernel, dim3(R), dim3(kThreads), 0, s, t, occ, off, ncell, sites, from,
                     codes, de);
  return hipGetLastError();
}

// The occupancy goes to LDS when the largest replica fits beside the static LDS of the kernel.
hipError_t LaunchCmc(const KTables &t, const CmcDev &c, uint64_t trials, uint64_t trace_base,
                     hipStream_t s) {
  if (c.R <= 0 || trials == 0) return hipSuccess;
  // static LDS of the occupancy-in-LDS kernels, the same on every device of this build
  static std::mutex mu;
  static size_t stat = 0, stat_omp = 0;  // 0 until a query succeeds
  size_t st_serial, st_omp;
  {
    std::lock_guard<std::mutex> lock(mu);
    if (!stat) {
      hipFuncAttributes fa, fb, fc, fd;
      if (hipFuncGetAttributes(&fa, reinterpret_cast<const void *>(CmcKernel<true, false>)) !=
              hipSuccess ||
          hipFuncGetAttributes(&fb, reinterpret_cast<const void *>(CmcKernel<true, true>)) !=
              hipSuccess ||
          hipFuncGetAttributes(&fc, reinterpret_cast<const void *>(CmcOmpKernel<true, false>)) !=
              hipSuccess ||
          hipFuncGetAttributes(&fd, reinterpret_cast<const void *>(CmcOmpKernel<true, true>)) !=
              hipSuccess)
        return hipErrorInvalidDevice;
      stat_omp = std::max(fc.sharedSizeBytes, fd.sharedSizeBytes);
      stat = std::max(fa.sharedSizeBytes, fb.sharedSizeBytes);
    }
    st_serial = stat;
    st_omp = stat_omp;
  }
  const size_t lds_block = CurrentDeviceLimits().lds_block;
  const size_t dyn = static_cast<size_t>(c.max_sites);
  auto launch = [&](auto kernel_lds, auto kernel_hbm, size_t st, int threads) {
    if (c.lds_occupancy && dyn % 4 == 0 && st + dyn <= lds_block) {
      if (dyn > 65536 - st) {
        const hipError_t e = RaiseDynamicLds(reinterpret_cast<const void *>(kernel_lds), dyn);
        if (e != hipSuccess) return e;
      }
      hipLaunchKernelGGL(kernel_lds, dim3(c.R), dim3(threads), dyn, s, t, c, trials, trace_base);
    } else {
      hipLaunchKernelGGL(kernel_hbm, dim3(c.R), dim3(threads), 0, s, t, c, trials, trace_base);
    }
    return hipGetLastError();
  };
  if (c.omp_k > 0)
    return c.log_every
               ? launch(CmcOmpKernel<true, true>, CmcOmpKernel<false, true>, st_omp, kOmpThreads)
               : launch(CmcOmpKernel<true, false>, CmcOmpKernel<false, false>, st_omp, kOmpThreads);
  return c.log_every ? launch(CmcKernel<true, true>, CmcKernel<false, true>, st_serial, kCmcThreads)
                     : launch(CmcKernel<true, false>, CmcKernel<false, false>, st_serial, kCmcThreads);
}

hipError_t LaunchCmcReference(const KTables &t, const CmcDev &c, uint8_t *ref, hipStream_t s) {
  if (c.R <= 0) return hipSuccess;
  hipLaunchKernelGGL(CmcReferenceKernel, dim3(c.R), dim3(kOmpThreads), 0, s, c, t.S, ref);
  return hipGetLastError();
}

hipError_t LaunchCmcAverage(const CmcDev &c, hipStream_t s) {
  if (c.R <= 0 || !c.log_every || !c.avg_m) return hipSuccess;
  hipLaunchKernelGGL(CmcAverageKernel, dim3(c.R, 64), dim3(kThreads), 0, s, c);
  return hipGetLastError();
}

int TotalCountRow(const KTables &t) { return t.n_eci + 3 + 4 * t.S; }

hipError_t LaunchTotalEncode(const KTables &t, const uint8_t *occ, const int64_t *off,
                             const int32_t *ncell, int32_t R, unsigned long long *counts,
                             double *encode, double *energy, hipStream_t s) {
  if (R <= 0) return hipSuccess;
  const int row = TotalCountRow(t);
  if (row > kMaxCountRow) return hipErrorInvalidValue;
  const int64_t nc = static_cast<int64_t>(R) * row;
  hipLaunchKernelGGL(ZeroKernel, dim3((nc + 255) / 256), dim3(256), 0, s, counts, nc);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  // slices of a box: enough workgroups for the chip when there are few boxes
  const int slices = std::max(64, std::min(1024, 4096 / R));
  hipLaunchKernelGGL(TotalCountsKernel, dim3(R, slices), dim3(kThreads), 0, s, t, occ, off, ncell, counts, row);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(EncodeKernel, dim3(R), dim3(64), 0, s, t, counts, row, occ, off, ncell, encode, energy);
  return hipGetLastError();
}

hipError_t LaunchClusterEncode(const KTables &t, const uint8_t *occ, int32_t n, const int64_t *set,
                               int32_t m, unsigned long long *counts, double *encode,
                               double *energy, hipStream_t s) {
  hipLaunchKernelGGL(ZeroKernel, dim3((t.n_eci + 255) / 256), dim3(256), 0, s, counts,
                     static_cast<int64_t>(t.n_eci));
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const int blocks = std::max(1, std::min(64, (m + kThreads - 1) / kThreads));
  hipLaunchKernelGGL(ClusterCountsKernel, dim3(blocks), dim3(kThreads), 0, s, t, occ, n, set, m,
                     counts);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(EncodeKernel, dim3(1), dim3(64), 0, s, t, counts, t.n_eci, nullptr, nullptr, nullptr, encode,
                     energy);
  return hipGetLastError();
}

// The cluster-count scratch of lmc_total_energy_noalloc: one copy per device, held until the
// process ends. Host code never passes `scratch` itself (its host-side name is not a device
// address); it passes the address TotalEnergyScratch looked up on the current device.
constexpr size_t kScratchCounts = size_t{1} << 19;  // 64-bit counts of ECIs
// a count row holds up to as many entries again for clusters without an ECI
static __device__ __align__(256) unsigned long long scratch[2 * kScratchCounts];

constexpr int kMaxScratchDevices = 64;
std::mutex g_scratch_mu;
unsigned long long *g_scratch_ptr[kMaxScratchDevices] = {};

size_t TotalEnergyScratchCapacity() { return kScratchCounts; }

hipError_t TotalEnergyScratch(unsigned long long **ptr) {
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  if (dev < 0 || dev >= kMaxScratchDevices) return hipErrorInvalidDevice;
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (!g_scratch_ptr[dev]) {  // once per device, with that device current
    void *p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_ptr[dev] = static_cast<unsigned long long *>(p);
  }
  *ptr = g_scratch_ptr[dev];
  return hipSuccess;
}

}  // namespace lmc
