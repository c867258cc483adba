// gfx950 kernels of the vacancy-jump evaluation and of the residence-time steps
// (KineticMcFirst, KineticMcChain), on the quadratic form of lmc_pairs.h (lmc_pair_device.h).
//
// KMC step of one replica:
//   1. gather : species of the 134 sites around the vacancy; the loads are issued as soon as the
//               previous step has chosen its jump, ahead of its bookkeeping;
//   2. sums   : terms of the non-reference sites and of their near pairs, per event;
//   3. events : lane l finishes event l % 16 (neighbour ids ascending): Ea, dE and the rate
//               exp(-Ea beta) (JumpEvent.cpp:6-13);
//   4. select : cumulative rates by a scan within each row of 16 lanes against u2 times the total
//               (KineticMcFirstOmp.cpp:52-82, KineticMcAbstract.cpp:106-123), residence time
//               with u1, jump (KineticMcAbstract.cpp:140-182). Philox numbers are drawn 64 steps
//               at a time, one step per lane.
// One wave makes the whole step (its replica then needs no barrier), or it shares step 2 with three
// helper waves. Tables are copied to LDS once per launch; the value tables are read from global memory
// when they do not fit.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <map>
#include <mutex>
#include <type_traits>

#include "lmc_pair_device.h"
#include "lmc_replica.h"
#include "lmc_rng.h"

namespace lmc {
namespace {

// Waves per SIMD that the scheduler aims at. Left to itself it keeps registers for more waves than the
// LDS lets in and makes every list batch a chain of single loads (a wave has its SIMD almost alone).
#define LMC_WAVES(lo, hi) __attribute__((amdgpu_waves_per_eu(lo, hi)))

constexpr int kEvalWaves = 8;  // waves of an evaluation workgroup
// kMaxSparse where they share the dense sums. Back-to-back calls of 12 vacancies (E0, ternary / Quartic,
// quaternary) at 11, 16, 21, 27 and 32 such sites, us: sparse 6.1, 6.5, 6.9, 7.4 and 8.2 / 7.3, 8.0, 8.3, 9.2
// and 10.0, dense 7.0 / 8.8 at any content.
constexpr int kMaxShared = 20;
constexpr int kTeam = 4;       // waves of a replica in the team shape
constexpr int kChainTeam = kTeam + 1;  // of a team that makes chain steps, with the one that keeps the energies

// Dynamic LDS of a workgroup (byte offsets): value tables, replicas' and waves' working sets.
struct KmcLayout {
  PairLayout tab;
  int team, wave, extra, wd, bytes;  // wd: the state clusters' weights (teams)
};

__device__ __forceinline__ int WaveIndex() {
  return __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x) >> 6);
}

// The 12 jumps of each replica r (vacancy vac[r] in occupancy occ + off[r] of ncell[r]^3 cells), or
// with kScan of a vacancy placed at each site vac[r] of the single occupancy occ (scan_n^3 cells)
// whose site sub_site holds sub_code. One wave per replica or site; the workgroups stride over
// them, so that one copy of the tables serves many. kShare: a workgroup to each, whose waves share the sums
// where they are dense.
template <bool kQ, int kTab, bool kScan, bool kShare>
__global__ __launch_bounds__(64 * kEvalWaves) LMC_WAVES(1, 2) void EvalJumpsKernel(
    KTables t, KmcLayout lay, const uint8_t *occ, const int64_t *off, const int32_t *ncell,
    const int64_t *vac, int32_t R, int64_t *nb, double *ea, double *de, int32_t *err,
    uint8_t *env_out, double *ekra_out, int ref, int scan_n, int64_t sub_site, int sub_code) {
  __shared__ PairShared<kQ> G;
  extern __shared__ __align__(16) char dyn[];
  const int lane = LaneId(), wave = WaveIndex();
  const PairTab T =
      LoadPairTables<kQ, kTab>(t, G, dyn, lay.tab, ref, threadIdx.x, 64 * kEvalWaves);
  __syncthreads();
  TeamLds &S = reinterpret_cast<TeamLds *>(dyn + lay.team)[kShare ? 0 : wave];
  WaveLds &W = reinterpret_cast<WaveLds *>(dyn + lay.wave)[wave];
  int &listed = *reinterpret_cast<int *>(dyn + lay.extra);  // kShare: the first wave's K
  if (kShare && wave != 0) {
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(listed) > kMaxShared) (void)DenseTerms<kQ, kEvalWaves>(G, T, S, W, 0, wave);
    __syncthreads();
    return;
  }
  const LaneSites ls = LoadSites<!kScan>(t, 0);
  const ExpConst E = MakeExpConst();
  constexpr int kSites = kShare ? 1 : kEvalWaves;  // of a workgroup at a time
  for (int64_t r = static_cast<int64_t>(blockIdx.x) * kSites + wave; r < R;
       r += static_cast<int64_t>(gridDim.x) * kSites) {
    const int n = kScan ? scan_n : ncell[r];
    const int64_t site = vac[r];
    if (!ValidSite(n, site)) {
      if (lane == 0) atomicOr(err, 8);
      if (kShare) {
        if (lane == 0) listed = 0;
        __syncthreads();
        __syncthreads();
      }
      continue;
    }
    const uint8_t *o = kScan ? occ : occ + off[r];
    const XYZ c = n <= 1000 ? ToXYZ32(static_cast<uint32_t>(site), static_cast<uint32_t>(n)) : ToXYZ(site, n);
    Around<uint64_t> a;
    GatherAround(ls, o, n, c, a);
    if (kScan) Substitute(a, static_cast<uint64_t>(sub_site), sub_code);
    const int dir = EventDirection(G, c, n);
    const bool bad = CheckCodes(t, a, dir, err);
    const int M = Bpermute(dir, a.code[0]);
    const EventConst ec = LoadConst(t, G, M);
    const int K = ListSites<kQ, kShare ? kMaxShared : kMaxSparse>(t, G, T, S, ls, a);
    PairSums s{0.0, 0.0, 0.0};
    if (kShare) {
      if (lane == 0) listed = K;
      __syncthreads();
      if (K > kMaxShared) (void)DenseTerms<kQ, kEvalWaves>(G, T, S, W, dir, 0);
      else s = PairTerms<kQ, 1>(G, T, S, W, ls, K, MakeRow<kQ>(t, T, dir, M), 0);
      __syncthreads();
      for (int w = 0; K > kMaxShared && w < kEvalWaves; ++w) {
        const double(&x)[3] = (&W)[w].sum[dir];
        s.de += x[0];
        s.la += x[1];
        if (kQ) s.lb += x[2];
      }
    } else {
      s = PairTerms<kQ, 1>(G, T, S, W, ls, K, MakeRow<kQ>(t, T, dir, M), 0);
    }
    const EventValue e = FinishEvent<kQ>(E, ec, s, bad);
    const uint64_t id = Bpermute64(dir, a.id[0]);
    if (lane < 12) {
      if (EventError(e)) atomicOr(err, 1);
      const int64_t w = r * 12 + lane;
      nb[w] = static_cast<int64_t>(id);
      ea[w] = e.ea;
      de[w] = e.de;
      if (ekra_out) ekra_out[w] = e.ekra;
    }
    if (env_out) {  // environment rows of the events in rank order (60 slot codes, zero padded)
      WaveFence();
#pragma unroll
      for (int u = 0; u < 3; ++u)
        if (lane + 64 * u <= kPairSites) S.code[lane + 64 * u] = static_cast<uint16_t>(a.code[u]);
      WaveFence();
      for (int q = 0; q < 12; ++q) {
        const int d = ReadLaneInt(dir, q);
        env_out[(r * 12 + q) * 64 + lane] = lane < kEnvSlots ? static_cast<uint8_t>(S.code[t.site_of[d * kEnvSlots + lane]]) : 0;
      }
      WaveFence();
    }
  }
}

// Uniforms of the steps of one replica: lane l holds those of step base + l.
struct StepDraws {
  double u2, log_u1;
  uint64_t base;
  bool ok;
};
// u2 and log(u1) of step Q.steps; every 64 steps the wave draws the next 64.
__device__ __forceinline__ void DrawStep(StepDraws &d, const ReplicaLds &Q, double &u2, double &log_u1) {
  if (!d.ok || Q.steps - d.base >= 64) {  // uniform
    const U4 u = Philox4x32_10(Q.seed, Q.steps + LaneId(), Q.rid, 0u);
    d.u2 = UnitOpenRight(Join64(u.z, u.w));
    d.log_u1 = log(UnitOpenLeft(Join64(u.x, u.y)));
    d.base = Q.steps;
    d.ok = true;
  }
  const int i = __builtin_amdgcn_readfirstlane(static_cast<int>(Q.steps - d.base));
  u2 = ReadLane(d.u2, i);
  log_u1 = ReadLane(d.log_u1, i);
}

// UpdateTemperature (KineticMcAbstract.cpp:45-50) and the RateCorrector factor at that temperature
// (RateCorrector.hpp:17-24), formed again only when the temperature has changed.
struct StepClock {
  double corr, corr_T;
};
__device__ __forceinline__ void UpdateTemperature(const KmcDev &k, ReplicaLds &Q, StepClock &C) {
  if (k.n_tt > 0) {
    Q.T = ScheduleTemperature(k.tt_time, k.tt_temp, k.n_tt, Q.time);
    Q.beta = 1.0 / kBoltzmann / Q.T;
  }
  if ((Q.flags & 1) && Q.T != C.corr_T) {
    C.corr = Q.cv / (1.64 * exp(-(0.66 / kBoltzmann / Q.T - 0.7))) / (1 - 13 * Q.cs);
    C.corr_T = Q.T;
  }
}

// A chosen jump: target site and its coordinates, the move (a/2 units), migrating species, barrier,
// energy change.
struct Jump {
  uint32_t site;
  XYZ to, move;
  int mig;
  double ea, de;
};

// The jumps of the events as their lanes hold them, for one readlane each: x | y << 16, and
// z | packed move << 16 (two bits per component, plus one).
struct EventTargets {
  uint32_t site, xy, zm;
};
__device__ __forceinline__ EventTargets MakeTargets(const LaneSites &ls, const Around<uint32_t> &a, int dir) {
  return {static_cast<uint32_t>(Bpermute(dir, static_cast<int>(a.id[0]))),
          static_cast<uint32_t>(Bpermute(dir, static_cast<int>(a.near.x | (a.near.y << 16)))),
          static_cast<uint32_t>(Bpermute(dir, static_cast<int>(a.near.z | ls.move)))};
}
__device__ __forceinline__ Jump TakeJump(const EventTargets &e, int mig, double ea, double de, int sel) {
  const uint32_t xy = static_cast<uint32_t>(ReadLaneInt(static_cast<int>(e.xy), sel));
  const uint32_t zm = static_cast<uint32_t>(ReadLaneInt(static_cast<int>(e.zm), sel));
  Jump j;
  j.site = static_cast<uint32_t>(ReadLaneInt(static_cast<int>(e.site), sel));
  j.to = {static_cast<int>(xy & 0xFFFFu), static_cast<int>(xy >> 16), static_cast<int>(zm & 0xFFFFu)};
  j.move = {static_cast<int>((zm >> 16) & 3u) - 1, static_cast<int>((zm >> 18) & 3u) - 1,
            static_cast<int>((zm >> 20) & 3u) - 1};
  j.mig = ReadLaneInt(mig, sel);
  j.ea = ea;
  j.de = de;
  return j;
}

// The first half of a step's end, before the next gather: what depends on the state before the jump
// (escape record, log, atoms; kFull), then the occupancy (kStore) and the vacancy's new position. Every
// lane holds Q; lane 0 keeps the records. energies: the log's too.
template <bool kFull, bool kStore = true>
__device__ __forceinline__ void ApplyJump(const KTables &t, const KmcDev &k, ReplicaLds &Q, uint8_t *occ,
                                          int r, const Jump &j, bool escaped, bool energies = true) {
  if constexpr (kFull) {
    const bool writer = kStore && LaneId() == 0;
    if (escaped) {
      if (writer && k.esc_time) {
        k.esc_time[r] = Q.time;
        k.esc_step[r] = Q.steps;
        k.esc_site[r] = Q.vac;
      }
      Q.esc = 1;
      Q.steps = Q.max_steps + 1;
    }
    if (writer && k.log_every && LogDue(Q.steps, k.log_every))
      LogStep(k, Q, r, static_cast<int64_t>(j.site), j.ea, j.de, energies);
    if (writer && k.atom) {  // the vacancy at Q.vac is the lhs of the reference's jump pair
      const int64_t o = k.off[r];
      const int h = Q.m2 >> 1;
      AtomJump(k.atom + o, k.shift + 3 * o, Q.vac, static_cast<int64_t>(j.site), ImageChange(j.to.X - Q.vx, h),
               ImageChange(j.to.Y - Q.vy, h), ImageChange(j.to.Z - Q.vz, h));
    }
  }
  if constexpr (kStore) {
    // Config::LatticeJump (Config.cpp:431-456): the two bytes in one store of all lanes, without a
    // branch
    const bool odd = (LaneId() & 1) != 0;
    occ[odd ? j.site : static_cast<uint32_t>(Q.vac)] = static_cast<uint8_t>(odd ? t.x_code : j.mig);
  }
  Q.vx = j.to.X;
  Q.vy = j.to.Y;
  Q.vz = j.to.Z;
  Q.vac = static_cast<int64_t>(j.site);
}

// The second half, under the next gather's loads: clock, energies, trace, displacements
// (KineticMcAbstract.cpp:147-181). energies: the trace's too.
template <bool kFull>
__device__ __forceinline__ void FinishStep(const KmcDev &k, ReplicaLds &Q, int r, uint64_t trace_index,
                                           const Jump &j, double dt, XYZ &moved, bool energies = true) {
  const XYZ &d = j.move;
  if constexpr (kFull) {
    if (trace_index < k.trace_cap && LaneId() == 0) {
      const uint64_t o = static_cast<uint64_t>(r) * k.trace_cap + trace_index;
      k.tr_sel[o] = static_cast<int64_t>(j.site);
      k.tr_ea[o] = j.ea;
      if (energies) k.tr_de[o] = j.de;
      k.tr_time[o] = Q.time + dt;
    }
    if ((Q.flags & 4) && j.mig != Q.solvent) {  // solute COM (KineticMcAbstract.cpp:163-177)
      const double wgt = k.mass[j.mig] / Q.smass;
      Q.com[0] -= d.X * kHalfLattice * wgt;
      Q.com[1] -= d.Y * kHalfLattice * wgt;
      Q.com[2] -= d.Z * kHalfLattice * wgt;
    }
  }
  Q.time += dt;
  Q.energy += j.de;
  Q.abse += j.de;
  moved.X += d.X;
  moved.Y += d.Y;
  moved.Z += d.Z;
  Q.steps += 1;
  if (Q.steps > Q.max_steps || (kFull && Q.esc)) Q.done = 1;
}

// IsEscaped (KineticMcAbstract.cpp:192-223): the 42 sites of the vacancy's three shells (sites
// 0 .. 41) hold the solvent.
__device__ __forceinline__ bool Escaped(const ReplicaLds &Q, int code0) {
  return (Q.flags & 2) && __ballot(LaneId() < 42 && code0 != Q.solvent) == 0;
}

// Event of the ordered cumulative probabilities: the first one whose sum reaches u2 of the total,
// else the last (`cum` on lanes 0 .. 10 of a row).
__device__ __forceinline__ int SelectEvent(double cum, double goal) {
  const uint64_t below = __ballot(LaneId() < 11 && cum < goal);
  return __builtin_ctzll(~below);
}

// Exchange area of a team: events' direction and migrating species, listed sites, partial sums.
struct TeamExchange {
  double part[kTeam][16][3];
  int info[16];
  int K;  // listed sites + 1 (0: the replica or the launch has ended) | choice of the step before << 8, and
          // at the end whether that step escaped << 12
  OrderedLds ordered;
  int32_t off[12][64];  // slots' offsets by direction (EnergyKeeper)
};

// The energies of a team's replica (OrderedDe), kept by one wave beside the leading wave's work, two steps
// late, so that nothing waits for them: the species of a step's slots are loaded one step later, when
// its choice is known, and summed another step later. In between the leading wave may have stored the
// next jump: of the slots that are read, that changes the target only, whose species the jump names.
// It takes 0.04 us of a step's 1.74 us (64 replicas, E0; the step without it and with one code for all
// waves: 1.82 us), and with chain steps, in a wave of its own, 0.1 us of 8.5. Batches with more replicas
// than CUs have no wave to spare and add the quadratic form's changes.
template <bool kFull>
struct EnergyKeeper {
  ReplicaLds Q;
  LaneSites ls;
  OrderedClusters clusters;
  const uint8_t *occ;
  const int32_t *off;  // offsets of the event's slots by direction
  int n, r;
  double sign;         // chain steps add the reverse event's change, negated
  uint64_t log_n, trace_base;
  XYZ c;               // the vacancy before the step to come
  uint32_t site;       // the step loaded: site and species of its slot `lane`, migrating species
  int code, mig;
  __device__ __forceinline__ void Start(const KTables &t, const KmcDev &k, int replica, int wv, const int32_t *slots,
                                        double way, uint64_t base) {
    r = replica;
    n = k.ncell[r];
    ls = LoadSites(t, wv);
    clusters = LoadOrdered(t);
    occ = k.occ + k.off[r];
    off = slots;
    sign = way;
    trace_base = base;
    LoadReplica(k, r, n, Q);
    log_n = kFull && k.log_every ? k.log_n[r] : 0;
    c = VacancyXYZ(Q);
    site = 0;
    code = mig = 0;
  }
  // The choice of step `it` of the launch (direction | migrating species << 8), whose jump is stored; the
  // next one is not before the barrier that follows. last: no step follows; escaped: in the last.
  __device__ __forceinline__ void Take(const KTables &t, const KmcDev &k, OrderedLds &D, const char *wd, int it,
                                       int choice, bool last, bool escaped) {
    const XYZ to = WrapAdd(c, PackedXYZ(ReadLaneInt(ls.pk[0], choice & 255)), Q.m2);
    const uint32_t new_site = SiteId<uint32_t>(WrapSite(c, n, off[64 * (choice & 255) + LaneId()]), n);
    const int new_code = occ[new_site];
    const uint32_t target = SiteId<uint32_t>(
        {static_cast<uint32_t>(to.X), static_cast<uint32_t>(to.Y), static_cast<uint32_t>(to.Z)}, n);
    code = site == target ? choice >> 8 : code;
    int i = it - 1;  // the last step is summed at once
#pragma nounroll
    do {
      if (i >= 0) {
        const double de = sign * OrderedDe(t, clusters, D, code, wd, mig);
        if constexpr (kFull) {
          const uint64_t steps = i == it && escaped ? Q.max_steps + 1 : Q.steps + i;
          if (k.log_every && LogDue(steps, k.log_every)) {
            if (log_n < k.log_cap && LaneId() == 0)
              LogEnergy(k.log[static_cast<uint64_t>(r) * k.log_cap + log_n], Q.energy, de);
            ++log_n;
          }
          if (trace_base + i < k.trace_cap && LaneId() == 0)
            k.tr_de[static_cast<uint64_t>(r) * k.trace_cap + (trace_base + i)] = de;
        }
        Q.energy += de;
        Q.abse += de;
      }
      code = new_code;
      mig = choice >> 8;
      ++i;
    } while (last && i <= it);
    c = to;
    site = new_site;
    asm volatile("" : "+v"(code));  // loaded before the barrier that follows
  }
};

// A helper wave of a team: its share of the sums of every step, from barrier to barrier; it ends when the
// leading wave announces no further step (X.K). The last helper also keeps the energies, after a step's
// second barrier, while the leading wave finishes the step.
template <bool kQ, bool kFull>
__device__ __forceinline__ void HelpTeam(const KTables &t, const PairShared<kQ> &G, const PairTab &T,
                                         const TeamLds &S, WaveLds &W, TeamExchange &X, char *wd,
                                         const KmcDev &k, int r, int wv, uint64_t trace_base) {
  const int lane = LaneId();
  const bool keeps = wv == kTeam - 1;
  EnergyKeeper<kFull> keeper;
  keeper.Start(t, k, r, wv, X.off[0], 1.0, trace_base);
  int before = 0;  // X.info of the step before
  for (int it = 0;; ++it) {
    __syncthreads();
    const int word = __builtin_amdgcn_readfirstlane(X.K), K = (word & 255) - 1;
    const int info = X.info[lane & 15];
    if (K >= 0) {
      const PairSums s =
          PairTerms<kQ, kTeam>(G, T, S, W, keeper.ls, K, MakeRow<kQ>(t, T, info & 255, info >> 8), wv);
      if (lane < 16) {
        double *p = X.part[wv][lane];
        p[0] = s.de;
        p[1] = s.la;
        if (kQ) p[2] = s.lb;
      }
      __syncthreads();
    }
    if (keeps && it == 0) {  // the keeper's tables, needed from the next step on
      CopyTable(reinterpret_cast<char *>(X.off), t.env_pk, sizeof(X.off), lane, 64);
      CopyTable(wd, t.wd, 8 * t.nwd, lane, 64);
      WaveFence();
    }
    if (keeps && it > 0)
      keeper.Take(t, k, X.ordered, wd, it - 1, ReadLaneInt(before, (word >> 8) & 15), K < 0, word >> 12);
    before = info;
    if (K < 0) break;
  }
  if (keeps && lane == 0) StoreEnergy(k, r, keeper.Q);
}

// Persistent KMC. kWaves 1: `group` replicas per workgroup, one wave each; the waves never meet after
// the table copy. kWaves kTeam: one replica per workgroup, a leading wave makes the step and three
// helpers share its sums, with two barriers per step (HelpTeam).
// kFull: options, schedule, trace, log and atoms are compiled in.
template <bool kQ, int kTab, int kWaves, bool kFull>
__global__ __launch_bounds__(kWaves == 1 ? 512 : 64 * kTeam) LMC_WAVES(1, 2) void KmcKernel(
    KTables t, KmcLayout lay, KmcDev k, int group, int nsteps, uint64_t trace_base) {
  __shared__ PairShared<kQ> G;
  extern __shared__ __align__(16) char dyn[];
  const int lane = LaneId(), wave = WaveIndex();
  const int first = blockIdx.x * group, mine = kWaves == 1 ? wave : 0;
  const PairTab T =
      LoadPairTables<kQ, kTab>(t, G, dyn, lay.tab, k.solvent[first], threadIdx.x, blockDim.x);
  TeamExchange &X = *reinterpret_cast<TeamExchange *>(dyn + lay.extra);
  __syncthreads();
  const int r = first + mine;
  if (mine >= group || r >= k.R) return;
  TeamLds &S = reinterpret_cast<TeamLds *>(dyn + lay.team)[mine];
  WaveLds &W = reinterpret_cast<WaveLds *>(dyn + lay.wave)[wave];
  if constexpr (kWaves > 1) {
    if (wave != 0) {
      HelpTeam<kQ, kFull>(t, G, T, S, W, X, dyn + lay.wd, k, r, wave, trace_base);
      return;
    }
  }
  const LaneSites ls = LoadSites(t, 0);
  const ExpConst E = MakeExpConst();
  uint8_t *occ = k.occ + k.off[r];
  const int n = k.ncell[r];
  ReplicaLds Q;
  LoadReplica(k, r, n, Q);
  StepDraws draws{0.0, 0.0, 0, false};
  XYZ moved{0, 0, 0};  // displacement of this launch
  StepClock clock{1.0, 0.0};
  Around<uint32_t> a;
  double u2 = 0.0, log_u1 = 0.0;
  int dir = 0, sel = 0;
  bool error = false;
  if (!Q.done) {
    GatherAround(ls, occ, n, VacancyXYZ(Q), a);
    dir = EventDirection(G, VacancyXYZ(Q), n);
    DrawStep(draws, Q, u2, log_u1);
  }
  for (int it = 0; it < nsteps; ++it) {
    if (Q.done) break;
    if (kFull) UpdateTemperature(k, Q, clock);
    const bool bad = CheckCodes(t, a, dir, k.error);
    const int M = Bpermute(dir, a.code[0]);
    const EventTargets to = MakeTargets(ls, a, dir);
    const EventRow row = MakeRow<kQ>(t, T, dir, M);
    const EventConst ec = LoadConst(t, G, M);
    const int K = ListSites<kQ>(t, G, T, S, ls, a);
    PairSums s;
    if constexpr (kWaves == 1) {
      s = PairTerms<kQ, 1>(G, T, S, W, ls, K, row, 0);
    } else {
      if (lane < 16) X.info[lane] = row.dir | (row.M << 8);
      if (lane == 0) X.K = (K + 1) | (sel << 8);
      __syncthreads();
      s = PairTerms<kQ, kWaves>(G, T, S, W, ls, K, row, 0);
      if (lane < 16) {
        double *p = X.part[0][lane];
        p[0] = s.de;
        p[1] = s.la;
        if (kQ) p[2] = s.lb;
      }
      __syncthreads();
      const double *p = X.part[0][lane & 15];
      s = {p[0], p[1], kQ ? p[2] : 0.0};
#pragma unroll
      for (int w = 1; w < kWaves; ++w) {
        s.de += p[48 * w];
        s.la += p[48 * w + 1];
        if (kQ) s.lb += p[48 * w + 2];
      }
    }
    const EventValue e = FinishEvent<kQ>(E, ec, s, bad);
    error = error || EventError(e);
    const double cum = RowScan((lane & 15) < 12 ? Exp(E, -e.ea * Q.beta) : 0.0);
    const double total = ReadLane(cum, 11);
    sel = SelectEvent(cum, u2 * total);
    const Jump j = TakeJump(to, row.M, kFull ? ReadLane(e.ea, sel) : 0.0, ReadLane(e.de, sel), sel);
    ApplyJump<kFull>(t, k, Q, occ, r, j, kFull && Escaped(Q, a.code[0]), kWaves == 1);
    WaveFence();
    GatherAround(ls, occ, n, VacancyXYZ(Q), a);
    dir = EventDirection(G, VacancyXYZ(Q), n);
    double dt = -log_u1 / (total * kPrefactor);
    if (kFull && (Q.flags & 1)) dt *= clock.corr;
    FinishStep<kFull>(k, Q, r, trace_base + it, j, dt, moved, kWaves == 1);
    DrawStep(draws, Q, u2, log_u1);
  }
  if constexpr (kWaves > 1) {  // no further step
    if (lane == 0) X.K = (sel << 8) | (kFull ? Q.esc << 12 : 0);
    __syncthreads();
  }
  if (__ballot(error) && lane == 0) atomicOr(k.error, 1);
  if (lane == 0) StoreReplica<kFull>(k, r, Q, moved, kWaves == 1);
}

// Persistent second-order (chain) KMC, KineticMcChainOmpi (KineticMcChainOmpi.cpp:56-151). Each step
// evaluates the 12 jumps out of every first neighbour i of the vacancy k in the configuration after
// the jump k -> i (12 passes: the vacancy at i, site k holding i's species), takes k -> i as the
// reverse of i -> k, and forms the second-order probabilities and the time with lane r on neighbour
// r (id order). kWaves 1: one wave makes all passes of a replica. kWaves kTeam: four waves hold the
// replica's state and make every fourth pass; one barrier per step exchanges their results, wave 0
// writes. A fifth wave, where the launch has one, keeps the energies.
struct ChainExchange {
  double res[2][12][3];  // as res below
  int choice[2];         // by step parity: direction | migrating species << 8
  int end[2];            // by step parity: 1, no such step; 3, and the step before it escaped
  OrderedLds ordered;
  int32_t off[12][64];
};
template <bool kQ, int kTab, int kWaves, bool kFull>
__global__ __launch_bounds__(kWaves == 1 ? 512 : 64 * kChainTeam) LMC_WAVES(1, 2) void KmcChainKernel(
    KTables t, KmcLayout lay, KmcDev k, int group, int nsteps, uint64_t trace_base) {
  __shared__ PairShared<kQ> G;
  extern __shared__ __align__(16) char dyn[];
  const int lane = LaneId(), wave = WaveIndex();
  const int first = blockIdx.x * group;
  const PairTab T =
      LoadPairTables<kQ, kTab>(t, G, dyn, lay.tab, k.solvent[first], threadIdx.x, blockDim.x);
  ChainExchange &X = *reinterpret_cast<ChainExchange *>(dyn + lay.extra);
  const bool kept = kWaves > 1 && blockDim.x > 64 * kWaves;  // the energies, by the wave past the last
  if (kept) {
    CopyTable(dyn + lay.wd, t.wd, 8 * t.nwd, threadIdx.x, blockDim.x);
    CopyTable(reinterpret_cast<char *>(X.off), t.env_pk + 12 * 64, sizeof(X.off), threadIdx.x, blockDim.x);
    if (threadIdx.x < 2) X.end[threadIdx.x] = 0;
  }
  __syncthreads();
  const int r = kWaves == 1 ? first + wave : first;
  if (kWaves == 1 && (wave >= group || r >= k.R)) return;
  const int wv = kWaves == 1 ? 0 : wave;
  if (kWaves > 1 && wv == kWaves) {
    EnergyKeeper<kFull> keeper;
    keeper.Start(t, k, r, 0, X.off[0], -1.0, trace_base);
    for (int it = 0;; ++it) {
      __syncthreads();
      const int end = __builtin_amdgcn_readfirstlane(X.end[it & 1]);
      if (it > 0) keeper.Take(t, k, X.ordered, dyn + lay.wd, it - 1,
                              __builtin_amdgcn_readfirstlane(X.choice[(it - 1) & 1]), end != 0, end == 3);
      if (end) break;
    }
    if (lane == 0) StoreEnergy(k, r, keeper.Q);
    return;
  }
  TeamLds &S = reinterpret_cast<TeamLds *>(dyn + lay.team)[wave];
  WaveLds &W = reinterpret_cast<WaveLds *>(dyn + lay.wave)[wave];
  // results of the passes, [step parity][neighbour rank][total rate, Ea, dE]
  double *res = reinterpret_cast<double *>(dyn + lay.extra) + (kWaves == 1 ? wave * 72 : 0);
  const LaneSites ls = LoadSites(t, 0);
  const ExpConst E = MakeExpConst();
  uint8_t *occ = k.occ + k.off[r];
  const int n = k.ncell[r];
  ReplicaLds Q;
  LoadReplica(k, r, n, Q);
  uint32_t prev = static_cast<uint32_t>(k.prev_j[r]);
  int prev_mig = -1;  // species the last jump left at prev
  bool error = false;
  StepDraws draws{0.0, 0.0, 0, false};
  XYZ moved{0, 0, 0};  // displacement of this launch
  StepClock clock{1.0, 0.0};
  int it = 0;
  for (; it < nsteps; ++it) {
    if (Q.done) break;
    if (kFull) UpdateTemperature(k, Q, clock);
    const XYZ c = VacancyXYZ(Q);
    Around<uint32_t> a;
    GatherAround(ls, occ, n, c, a);
    // the other waves may read before wave 0 has stored the jump
    if (kWaves > 1 && prev_mig >= 0) Substitute(a, prev, prev_mig);
    double u2, log_u1;
    DrawStep(draws, Q, u2, log_u1);
    const int dir = EventDirection(G, c, n);
    (void)CheckCodes(t, a, dir, k.error);
    double *x = res + (it & 1) * 36;
    for (int i = wv; i < 12; i += kWaves) {
      const int di = ReadLaneInt(dir, i);
      const XYZ ci = WrapAdd(c, PackedXYZ(ReadLaneInt(ls.pk[0], di)), Q.m2);
      Around<uint32_t> b;
      GatherAround(ls, occ, n, ci, b);
      if (kWaves > 1 && prev_mig >= 0) Substitute(b, prev, prev_mig);
      Substitute(b, static_cast<uint32_t>(Q.vac), ReadLaneInt(a.code[0], di));
      const int dirb = EventDirection(G, ci, n);
      const bool bad = CheckCodes(t, b, dirb, k.error);
      const int M = Bpermute(dirb, b.code[0]);
      const EventConst ec = LoadConst(t, G, M);
      const int K = ListSites<kQ>(t, G, T, S, ls, b);
      const PairSums s = PairTerms<kQ, 1>(G, T, S, W, ls, K, MakeRow<kQ>(t, T, dirb, M), 0);
      const EventValue e = FinishEvent<kQ>(E, ec, s, bad);
      error = error || EventError(e);
      const double cum = RowScan((lane & 15) < 12 ? Exp(E, -e.ea * Q.beta) : 0.0);
      // the jump back to k has the opposite direction, 11 - di
      const int back = __builtin_ctzll(__ballot(lane < 12 && dirb == 11 - di));
      const double ea = ReadLane(e.ea, back), de = ReadLane(e.de, back), tot = ReadLane(cum, 11);
      if (lane == 0) {
        x[3 * i] = tot;
        x[3 * i + 1] = ea;
        x[3 * i + 2] = de;
      }
    }
    if (kWaves > 1) __syncthreads();
    else WaveFence();
    // lane i: the event k -> i as the reverse of i -> k (KineticMcChainOmpi.cpp:56-91,
    // JumpEvent.cpp:25-30,51-54)
    const int ev = (lane & 15) < 12 ? lane & 15 : 11;
    const bool on = (lane & 15) < 12;
    const double total_i = x[3 * ev], barrier = x[3 * ev + 1] - x[3 * ev + 2], de = -x[3 * ev + 2];
    const double rate = on ? Exp(E, -barrier * Q.beta) : 0.0;
    const double p_ik = Exp(E, (de - barrier) * Q.beta) / total_i;
    const uint32_t sid = static_cast<uint32_t>(Bpermute(dir, static_cast<int>(a.id[0])));
    const double total = ReadLane(RowScan(rate), 11);
    const double t1 = 1 / total / kPrefactor, ti = 1 / total_i / kPrefactor;
    const double p_ki = rate / total;
    const double bb = on ? p_ki * p_ik : 0.0, b1 = on ? p_ki * (1 - p_ik) : 0.0;
    const bool was = on && sid == prev;
    auto row_total = [](double v) { return ReadLane(RowScan(v), 11); };
    const double g = row_total(bb), gb = row_total(b1);
    const double og = row_total(was ? 0.0 : bb), ob = row_total(was ? 0.0 : b1);
    const double al = row_total(was ? b1 : 0.0), ga = row_total(was ? p_ki : 0.0);
    const double tb = on ? (t1 + ti) * bb : 0.0;
    const double ts = row_total(tb) / g, ts_j = row_total(was ? 0.0 : tb) / og;
    const double inv = 1 / (1 - ga);
    double dt = inv * (ob * t1 + og * (ts_j + t1 + g / gb * ts));
    const double prob = was ? inv * (og / gb) * al : inv * (1 + og / gb) * b1;
    const double cum = RowScan(prob);
    const int sel = SelectEvent(cum, u2);
    const Jump j = TakeJump(MakeTargets(ls, a, dir), Bpermute(dir, a.code[0]), ReadLane(barrier, sel),
                            ReadLane(de, sel), sel);
    if (kept && wv == 0) X.choice[it & 1] = ReadLaneInt(dir, sel) | (j.mig << 8);
    prev = static_cast<uint32_t>(Q.vac);
    prev_mig = j.mig;
    const bool escaped = kFull && Escaped(Q, a.code[0]);
    if (wv == 0) ApplyJump<kFull>(t, k, Q, occ, r, j, escaped, !kept);
    else ApplyJump<kFull, false>(t, k, Q, occ, r, j, escaped);
    WaveFence();
    if (kFull && (Q.flags & 1)) dt *= clock.corr;
    if (wv == 0) FinishStep<kFull>(k, Q, r, trace_base + it, j, dt, moved, !kept);
    else FinishStep<kFull>(k, Q, r, ~0ull, j, dt, moved);
  }
  if (kept) {
    if (wv == 0) X.end[it & 1] = Q.esc ? 3 : 1;
    __syncthreads();
  }
  if (wv != 0) return;
  if (__ballot(error) && lane == 0) atomicOr(k.error, 1);
  if (lane == 0) {
    StoreReplica<kFull>(k, r, Q, moved, !kept);
    k.prev_j[r] = static_cast<int64_t>(prev);
  }
}

// Dynamic LDS plan for workgroups of `teams` replicas and `waves` waves: the value tables go to LDS
// when per_cu workgroups then still fit a CU, of a Quartic model also dE and MMM alone (63 of a quaternary
// one's 163 KB). Quaternary Quartic, none of them in LDS and mixed: first-order steps of equiatomic boxes 6.8
// and 4.1 us (64 replicas), 16.4 and 8.4 us (1 024); with 3 % solutes 2.58 and 2.26 us, 2.44 and 2.22 us; a scan
// of 32 000 sites of an equiatomic frame 497 and 222 us. The sums over all clusters took 7.5, 15.6 and 468.
KmcLayout PlanLds(const KTables &t, int teams, int waves, size_t extra, int per_cu, bool ordered = false) {
  const DeviceLimits &dl = CurrentDeviceLimits();
  const bool quartic = t.kind == kQuartic;
  const size_t fixed = quartic ? sizeof(PairShared<true>) : sizeof(PairShared<false>);
  const size_t share = std::min(dl.lds_block, dl.lds_cu / std::max(1, per_cu));
  KmcLayout lay{};
  size_t at = 0;
  auto add = [&](int &where, size_t bytes) {
    where = static_cast<int>(at);
    at = (at + bytes + 15) & ~size_t(15);
  };
  add(lay.team, teams * sizeof(TeamLds));
  add(lay.wave, waves * sizeof(WaveLds));
  add(lay.extra, extra);
  if (ordered) add(lay.wd, 8 * static_cast<size_t>(t.nwd));
  const size_t row = 8 * static_cast<size_t>(t.ne);
  const size_t some = row * (t.de_row + t.la_row) + 32, all = some + (quartic ? row * t.lb_row + 16 : 0);
  lay.tab.tab_lds = fixed + at + all <= share ? kShared : quartic && fixed + at + some <= share ? kMixed : kGlobal;
  if (lay.tab.tab_lds != kGlobal) {
    add(lay.tab.de, row * t.de_row);
    add(lay.tab.la, row * t.la_row);
  }
  if (quartic && lay.tab.tab_lds == kShared) add(lay.tab.lb, row * t.lb_row);
  lay.bytes = static_cast<int>(at);
  return lay;
}

template <typename K>
hipError_t AllowLds(K kernel, size_t bytes) {
  return RaiseDynamicLds(reinterpret_cast<const void *>(kernel), bytes);
}

// f(quartic, tables in LDS) with compile-time arguments.
template <typename F>
hipError_t WithModel(const KTables &t, const KmcLayout &lay, F &&f) {
  constexpr std::integral_constant<int, kGlobal> global;
  constexpr std::integral_constant<int, kShared> shared;
  constexpr std::integral_constant<int, kMixed> mixed;
  if (t.kind != kQuartic) return lay.tab.tab_lds ? f(std::false_type{}, shared) : f(std::false_type{}, global);
  if (lay.tab.tab_lds == kMixed) return f(std::true_type{}, mixed);
  return lay.tab.tab_lds ? f(std::true_type{}, shared) : f(std::true_type{}, global);
}

template <bool kScan>
hipError_t LaunchEval(const KTables &t, const uint8_t *occ, const int64_t *off, const int32_t *ncell,
                      const int64_t *vac, int32_t R, int64_t *nb, double *ea, double *de, int32_t *err,
                      hipStream_t s, uint8_t *env_out, double *ekra_out, int n, int64_t sub_site,
                      int sub_code) {
  if (R <= 0) return hipSuccess;
  const KmcLayout lay = PlanLds(t, kEvalWaves, kEvalWaves, 16, 1);
  // As many workgroups as are resident at once (one per CU for a ternary model's 92 KB; 2 where two fit), so
  // that none copies the tables again. Two per CU where one fits: 32 000 sites 73.8 us, one 71.8; 8 192
  // sites 48.7 and 45.5; Quartic 85.4 and 82.1, 52.5 and 49.0.
  const DeviceLimits &dl = CurrentDeviceLimits();
  const size_t lds = (t.kind == kQuartic ? sizeof(PairShared<true>) : sizeof(PairShared<false>)) + lay.bytes;
  // A CU to each where there is one: eight waves share the dense sums. Calls of 64 equiatomic boxes, us, from
  // Python: ternary E0 32.6, by one wave 36.0, by sums over all clusters 32.5; quaternary Quartic 33.6, 40.7
  // and 36.5.
  const bool share = R <= dl.cus;
  const int blocks = share ? R : std::min((R + kEvalWaves - 1) / kEvalWaves, (2 * lds <= dl.lds_cu ? 2 : 1) * dl.cus);
  return WithModel(t, lay, [&](auto q, auto tab) {
    constexpr bool kQ = decltype(q)::value;
    constexpr int kT = decltype(tab)::value;
    auto kernel = share ? EvalJumpsKernel<kQ, kT, kScan, true> : EvalJumpsKernel<kQ, kT, kScan, false>;
    const hipError_t e = AllowLds(kernel, lay.bytes);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(blocks), dim3(64 * kEvalWaves), lay.bytes, s, t, lay, occ, off, ncell,
                       vac, R, nb, ea, de, err, env_out, ekra_out, kScan ? sub_code : t.solvent_default, n, sub_site, sub_code);
    return hipGetLastError();
  });
}

// How a KMC batch is laid over the chip. form: 0 by the batch's size, 1 one wave per replica, 2 a team of
// four waves per replica, 3 chain steps (by the batch's size).
struct KmcPlan {
  KmcLayout lay;
  int group, blocks, threads;
  bool chain, team;
};
KmcPlan PlanKmc(const KTables &t, int32_t R, int form) {
  const int cus = CurrentDeviceLimits().cus;
  KmcPlan p;
  p.chain = form == 3;
  p.team = KmcTeam(R, form);
  // one-wave replicas: as many per workgroup as it takes to give every CU one workgroup, up to eight
  p.group = p.team ? 1 : std::min(8, std::max(1, (R + cus - 1) / cus));
  p.blocks = (R + p.group - 1) / p.group;
  const int waves = std::max(kTeam, p.group);
  // chain teams: the wave that keeps the energies only where one team has the CU; two teams of five waves
  // would not fit beside each other (400 replicas: 332 us for 30 steps, 452 with it)
  p.threads = 64 * (p.chain && p.team && R <= cus ? kChainTeam : waves);
  const size_t extra = p.team ? (p.chain ? sizeof(ChainExchange) : sizeof(TeamExchange))
                              : p.chain ? waves * 72 * sizeof(double) : 0;
  p.lay = PlanLds(t, p.chain ? waves : p.group, waves, extra, p.blocks > cus ? 2 : 1, p.team);
  return p;
}

// f(kernel) of the plan's instantiation.
template <typename F>
hipError_t WithKmcKernel(const KTables &t, const KmcPlan &p, bool full, F &&f) {
  return WithModel(t, p.lay, [&](auto q, auto tab) {
    constexpr bool kQ = decltype(q)::value;
    constexpr int kT = decltype(tab)::value;
    auto pick = [&](auto all) {
      constexpr bool kF = decltype(all)::value;
      if (p.chain) return p.team ? f(KmcChainKernel<kQ, kT, kTeam, kF>) : f(KmcChainKernel<kQ, kT, 1, kF>);
      return p.team ? f(KmcKernel<kQ, kT, kTeam, kF>) : f(KmcKernel<kQ, kT, 1, kF>);
    };
    return full ? pick(std::true_type{}) : pick(std::false_type{});
  });
}

}  // namespace

hipError_t LaunchEvalJumps(const KTables &t, const uint8_t *occ, const int64_t *off,
                           const int32_t *ncell, const int64_t *vac, int32_t R, int64_t *nb,
                           double *ea, double *de, int32_t *err, hipStream_t s, uint8_t *env_out,
                           double *ekra_out) {
  return LaunchEval<false>(t, occ, off, ncell, vac, R, nb, ea, de, err, s, env_out, ekra_out, 0, -1, 0);
}

hipError_t LaunchVacancyScan(const KTables &t, const uint8_t *occ, int32_t n, int64_t sub_site,
                             int sub_code, const int64_t *sites, int32_t K, int64_t *nb,
                             double *ea, double *de, int32_t *err, hipStream_t s) {
  return LaunchEval<true>(t, occ, nullptr, nullptr, sites, K, nb, ea, de, err, s, nullptr, nullptr, n,
                          sub_site, sub_code);
}

// Measured, us per step of batches of 12^3 cells (E0, ternary), one wave / four waves per replica:
//   replicas              1           64          256         512        1 024
//   1-5 at.% solutes   1.3 / 1.5   2.2 / 1.8   2.3 / 1.8   2.4 / 2.0   2.5 / 3.9
//   4-20 at.%          4.6 / 2.6   5.4 / 2.8   5.4 / 2.8   5.8 / 3.3   5.9 / 6.5
//   chain steps                   24.8 / 9.0  25.0 / 9.3  26.4 / 10.9  29.6 / 19.7
// Formulation 0 takes four where every replica has a CU, and chain steps where two replicas share one.
bool KmcTeam(int32_t R, int form) {
  const int cus = CurrentDeviceLimits().cus;
  return form == 2 || (form == 0 && R <= cus) || (form == 3 && R <= 2 * cus);
}

hipError_t PrepareKmc(const KTables &t, int32_t R, int form) {
  if (R <= 0) return hipSuccess;
  const KmcPlan p = PlanKmc(t, R, form);
  auto allow = [&](auto kernel) { return AllowLds(kernel, p.lay.bytes); };
  const hipError_t e = WithKmcKernel(t, p, false, allow);
  return e != hipSuccess ? e : WithKmcKernel(t, p, true, allow);
}

hipError_t LaunchKmc(const KTables &t, const KmcDev &k, uint64_t steps, uint64_t trace_base,
                     hipStream_t s, int form) {
  if (k.R <= 0 || steps == 0) return hipSuccess;
  // a launch counts its steps and displacements in 32 bits
  for (constexpr uint64_t kMost = 1u << 30; steps > kMost; steps -= kMost, trace_base += kMost) {
    const hipError_t e = LaunchKmc(t, k, kMost, trace_base, s, form);
    if (e != hipSuccess) return e;
  }
  const KmcPlan p = PlanKmc(t, k.R, form);
  const bool full = k.options || k.n_tt > 0 || k.trace_cap || k.atom || k.log_every;
  return WithKmcKernel(t, p, full, [&](auto kernel) {
    const hipError_t e = AllowLds(kernel, p.lay.bytes);
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(kernel, dim3(p.blocks), dim3(p.threads), p.lay.bytes, s, t, p.lay, k, p.group, static_cast<int>(steps),
                       trace_base);
    return hipGetLastError();
  });
}

hipError_t RaiseDynamicLds(const void *kernel, size_t bytes) {
  static std::mutex mu;
  static std::map<std::pair<int, const void *>, size_t> allowed;
  int dev = 0;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess) return e;
  std::lock_guard<std::mutex> lock(mu);
  size_t &most = allowed[{dev, kernel}];
  if (bytes <= most) return hipSuccess;
  e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(bytes));
  if (e == hipSuccess) most = bytes;
  return e;
}

const DeviceLimits &CurrentDeviceLimits() {
  static std::mutex mu;
  static std::map<int, DeviceLimits> known;  // entries are never erased: references stay valid
  static const DeviceLimits fallback{256, 65536, 65536};
  int dev = 0;
  hipDeviceProp_t p;
  if (hipGetDevice(&dev) != hipSuccess) return fallback;
  std::lock_guard<std::mutex> lock(mu);
  const auto it = known.find(dev);
  if (it != known.end()) return it->second;
  if (hipGetDeviceProperties(&p, dev) != hipSuccess) return fallback;
  DeviceLimits d;
  d.cus = p.multiProcessorCount;
  d.lds_cu = p.maxSharedMemoryPerMultiProcessor ? p.maxSharedMemoryPerMultiProcessor : 65536;
  d.lds_block = p.sharedMemPerBlock;
  return known.emplace(dev, d).first->second;
}

}  // namespace lmc
