// Device-side building blocks of the surrogate kernels (lmc_surrogate_kmc.hip): the environments of
// the 12 jumps, their cluster sums, and the KineticMcFirst step. `tid` is the thread's index in its
// replica's block.
#pragma once
#include <hip/hip_runtime.h>

#include "lmc_dev_common.h"
#include "lmc_device.h"
#include "lmc_replica.h"
#include "lmc_rng.h"

namespace lmc {
namespace {

// Element ranks of one event's environment slots, pre-scaled for the cluster tables: rank * 8
// (bytes) and rank * 8 * ne (16-bit); slots 60..63 hold 0 (slot 63 is the absent site).
struct EventRanks {
  uint8_t r8[64];
  uint16_t rn8[64];
};

struct JumpLds {
  uint16_t off[12 * kEnvSlots];  // relative offsets, 4 bits per component (+8)
  double par[kMaxSpecies * 6];
  uint8_t env[12][64];
  EventRanks er[12];
  int64_t nb[12];   // by direction
  // by rank (neighbour-id order)
  double ea[12], de[12], rate[12], ekra[12];
  int64_t snb[12];
  int dir[12];
  // random numbers of the current step (drawn by an idle lane during the gather)
  double u2, log_u1, corr;
  double prob[12];  // selection probabilities by rank
  // events whose environment holds a vacancy off the jump endpoints (no one-hot type)
  int bad;
};

// Byte offsets of the tables in dynamic LDS (computed on the host).
struct DynLayout {
  int w, b1, b2, lists, bytes;
  int b1_lds, b2_lds;
};

struct Tabs {  // resolved table pointers (LDS or global)
  const double *w, *b1, *b2;
  const uint32_t *state, *mmm, *mm2;
};

// Copies n elements from global memory to LDS with threads gtid of gsize, eight loads per thread
// in flight before their stores (the copy at a launch's start is latency-bound otherwise).
template <typename E>
__device__ __forceinline__ void CopyToLds(E *dst, const E *src, int n, int gtid, int gsize) {
  int i = gtid;
  for (; i + 7 * gsize < n; i += 8 * gsize) {
    E v[8];
#pragma unroll
    for (int u = 0; u < 8; ++u) v[u] = src[i + u * gsize];
#pragma unroll
    for (int u = 0; u < 8; ++u) dst[i + u * gsize] = v[u];
  }
  for (; i < n; i += gsize) dst[i] = src[i];
}

// Per-replica LDS tables (threads tid of this replica's block) and the workgroup's shared
// dynamic tables (threads gtid of gsize); returns the resolved table pointers.
// kBL: the barrier weight tables live in LDS (lay.b1_lds, and lay.b2_lds for the quartic model),
// known at compile time so that their reads are LDS instructions.
template <bool kBL>
__device__ Tabs LoadJumpTables(const KTables &t, JumpLds &L, char *dyn, const DynLayout &lay,
                               int tid, int lsize, int gtid, int gsize) {
  for (int i = tid; i < 12 * kEnvSlots; i += lsize) {
    int dx, dy, dz;
    Unpack(t.off[i], dx, dy, dz);
    L.off[i] = static_cast<uint16_t>((dx + 8) | ((dy + 8) << 4) | ((dz + 8) << 8));
  }
  for (int i = tid; i < 6 * t.S; i += lsize) L.par[i] = t.par[i];
  if (tid < 12 * 4) {  // slots 60..63; slot 63 is the target of every packed cluster's absent sites
    const int k = tid >> 2, j = kEnvSlots + (tid & 3);
    L.env[k][j] = 0;
    L.er[k].r8[j] = 0;
    L.er[k].rn8[j] = 0;
  }
  if (tid == 0) L.bad = 0;
  Tabs T{};
  double *w = reinterpret_cast<double *>(dyn + lay.w);
  CopyToLds(w, t.wd, t.nwd, gtid, gsize);
  T.w = w;
  if (kBL) {
    double *p = reinterpret_cast<double *>(dyn + lay.b1);
    CopyToLds(p, t.b1, t.ne * t.F1, gtid, gsize);
    T.b1 = p;
    double *q = reinterpret_cast<double *>(dyn + lay.b2);
    if (t.kind == kQuartic)
      CopyToLds(q, t.b2, t.ne * t.F2, gtid, gsize);
    T.b2 = q;
  } else {
    T.b1 = t.b1;
    T.b2 = t.b2;
  }
  {
    uint32_t *p = reinterpret_cast<uint32_t *>(dyn + lay.lists);
    CopyToLds(p, t.state, t.n_state, gtid, gsize);
    T.state = p;
    p += t.n_state;
    CopyToLds(p, t.mmm, t.n_mmm, gtid, gsize);
    T.mmm = p;
    p += t.n_mmm;
    if (t.kind == kQuartic)
      CopyToLds(p, t.mm2, t.n_mm2, gtid, gsize);
    T.mm2 = p;
  }
  return T;
}

// Element rank of a species code (a vacancy gives 0).
__device__ __forceinline__ uint32_t RankOf(const KTables &t, int code) {
  return (t.rank_lut >> (4 * code)) & 15u;
}

// Row of the dE difference table (bytes) and of an expanded barrier table for migrating
// species code M.
__device__ __forceinline__ const char *WRow(const KTables &t, const Tabs &T, int M) {
  return reinterpret_cast<const char *>(T.w) + __umul24(RankOf(t, M), 8 * t.wrow);
}
__device__ __forceinline__ const char *BRow(const double *b, int F, const KTables &t, int M) {
  return reinterpret_cast<const char *>(b) + __umul24(RankOf(t, M), 8 * F);
}

// Phase 1: species of the 12 environments; neighbour ids of the 12 jumps. 720 sites over the
// kBT threads of the replica's block: independent loads per thread, issued together. Split in
// two so that a caller can issue other loads between them.
template <int kBT = kThreads>
struct Gathered {
  static constexpr int kU = (12 * kEnvSlots + kBT - 1) / kBT;
  int64_t s[kU];
  uint8_t v[kU];
};

template <int kBT = kThreads>
__device__ __forceinline__ void GatherIssue(const JumpLds &L, const uint8_t *occ, int n,
                                            const XYZ &c, int tid, Gathered<kBT> &G) {
  constexpr int kTotal = 12 * kEnvSlots;
#pragma unroll
  for (int u = 0; u < Gathered<kBT>::kU; ++u) {
    const int i = tid + u * kBT;
    if (i < kTotal) {
      int dx, dy, dz;
      Unpack16(L.off[i], dx, dy, dz);
      G.s[u] = SiteAt(c, n, dx, dy, dz);
      G.v[u] = occ[G.s[u]];
    }
  }
}

template <int kBT = kThreads>
__device__ __forceinline__ void GatherStore(const KTables &t, JumpLds &L, int32_t *err, int tid,
                                            const Gathered<kBT> &G) {
  constexpr int kTotal = 12 * kEnvSlots;
#pragma unroll
  for (int u = 0; u < Gathered<kBT>::kU; ++u) {
    const int i = tid + u * kBT;
    if (i < kTotal) {
      const int k = i / kEnvSlots, j = i - k * kEnvSlots;
      uint8_t x = G.v[u];
      if (x >= t.S) {  // corrupt occupancy: flag it and keep every table index in range
        atomicOr(err, 4);
        x = 0;
      }
      if (x == t.x_code && j != t.v_slot) atomicOr(&L.bad, 1 << k);
      L.env[k][j] = x;
      const uint32_t rk = RankOf(t, x);
      L.er[k].r8[j] = static_cast<uint8_t>(rk << 3);
      L.er[k].rn8[j] = static_cast<uint16_t>(__umul24(rk, 8 * t.ne));
      if (j == t.n_slot) L.nb[k] = G.s[u];
    }
  }
}

// Byte offset of a packed entry's rank*8 slot (byte 1 of a state entry is the other one).
__device__ __forceinline__ uint32_t R8At(const EventRanks &er, uint32_t byte_off) {
  return er.r8[byte_off];
}
__device__ __forceinline__ uint32_t Rn8At(const EventRanks &er, uint32_t byte_off) {
  return *reinterpret_cast<const uint16_t *>(reinterpret_cast<const char *>(er.rn8) + byte_off);
}

// Sums of kU packed state clusters per lane: w(cluster | endpoint = M) - w(cluster | endpoint =
// X) from wm, the difference table's row of M (the entry's offset selects the negated copy for
// the neighbour endpoint's clusters). The loads of the kU clusters are issued level by level
// (entries, ranks, weights).
template <int kU>
__device__ __forceinline__ void StateBatch(const char *wm, const EventRanks &er,
                                           const uint32_t *list, int c, int stride, double *acc) {
  uint32_t d[kU], x1[kU], x2[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) d[u] = list[c + u * stride];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    x1[u] = R8At(er, d[u] & 0xFF);
    x2[u] = Rn8At(er, (d[u] >> 8) & 0xFF);
  }
#pragma unroll
  for (int u = 0; u < kU; ++u)
    acc[u] += *reinterpret_cast<const double *>(wm + (x1[u] + x2[u] + (d[u] >> 16)));
}

// Sum of the state clusters [c0, c1) of an event, lanes lane, lane + stride, ...
__device__ __forceinline__ double StateRange(const char *wm, const EventRanks &er,
                                             const uint32_t *list, int c0, int c1, int lane,
                                             int stride) {
  double a[4] = {0.0, 0.0, 0.0, 0.0};
  int c = c0 + lane;
  for (; c + 3 * stride < c1; c += 4 * stride) StateBatch<4>(wm, er, list, c, stride, a);
  for (; c < c1; c += stride) StateBatch<1>(wm, er, list, c, stride, a);
  return (a[0] + a[1]) + (a[2] + a[3]);
}

// Sums of kU packed orbit clusters per lane: bm[rank0 * ne + rank1] of the cluster's expanded
// weights (bm: the migrating species' row, bytes).
template <int kU>
__device__ __forceinline__ void OrbitBatch(const char *bm, const EventRanks &er,
                                           const uint32_t *list, int c, int stride, double *acc) {
  uint32_t d[kU], x0[kU], x1[kU];
#pragma unroll
  for (int u = 0; u < kU; ++u) d[u] = list[c + u * stride];
#pragma unroll
  for (int u = 0; u < kU; ++u) {
    x0[u] = Rn8At(er, d[u] & 0xFF);
    x1[u] = R8At(er, (d[u] >> 8) & 0xFF);
  }
#pragma unroll
  for (int u = 0; u < kU; ++u)
    acc[u] += *reinterpret_cast<const double *>(bm + (x0[u] + x1[u] + (d[u] >> 16)));
}

// Sum of the orbit clusters [0, n) of an event, lanes lane, lane + stride, ...
__device__ __forceinline__ double OrbitRange(const char *bm, const EventRanks &er,
                                             const uint32_t *list, int n, int lane, int stride) {
  double a[4] = {0.0, 0.0, 0.0, 0.0};
  int c = lane;
  for (; c + 3 * stride < n; c += 4 * stride) OrbitBatch<4>(bm, er, list, c, stride, a);
  for (; c < n; c += stride) OrbitBatch<1>(bm, er, list, c, stride, a);
  return (a[0] + a[1]) + (a[2] + a[3]);
}

// Ea and E_kra of event k from its cluster sums: dE, MMM logit la and MM2 logit lb.
__device__ __forceinline__ void Barrier(const KTables &t, const JumpLds &L, int k, double de,
                                        double la, double lb, double &ea, double &ekra) {
  const int M = L.env[k][t.n_slot];
  const double *p = L.par + 6 * M;
  ea = 0.0;
  ekra = 0.0;
  if (t.kind == kE0) {
    // E0 = exp(logit * sigma_e0 + mu_e0); Ea = max(0, E0 + dE/2) (...E0.cpp:147-158)
    const double e0 = exp((p[0] + la) * p[2] + p[1]);
    ea = fmax(0.0, e0 + de / 2);
    ekra = e0;
  } else if (t.kind == kQuartic) {
    // Quartic barrier (...Quartic.cpp:266-275)
    const double D = exp((p[0] + la) * p[2] + p[1]);
    const double Ks = exp((p[3] + lb) * p[5] + p[4]);
    const double b = 4 * de / (D * D * D);
    const double a = Ks / (4 * D * D);
    const double c = (9 * b * b - 16 * a * a * D * D) / (32 * a);
    const double delta = sqrt(fabs(9 * b * b - 32 * a * c));
    ea = (3 * b + delta) * (3 * b + delta) * (3 * b * b - 16 * a * c + b * delta) / (a * a * a) /
         2048;
    ekra = ea - de / 2;  // kinetically resolved barrier: Ea(i->j) - Ea(j->i) = dE
  }
}

// Stores event k (direction) at its rank among the 12 neighbour ids, with its rate
// exp(-Ea beta) (JumpEvent forward rate, JumpEvent.cpp:6-13).
__device__ __forceinline__ void StoreEvent(JumpLds &L, int k, double ea, double de, double ekra,
                                           double beta) {
  int r = 0;
  const int64_t mine = L.nb[k];
#pragma unroll
  for (int j = 0; j < 12; ++j) r += L.nb[j] < mine;
  L.ea[r] = ea;
  L.de[r] = de;
  L.ekra[r] = ekra;
  L.rate[r] = exp(-ea * beta);
  L.snb[r] = mine;
  L.dir[r] = k;
}

// Random numbers of step Q.steps (one lane, overlapping the gather): Philox u1, u2, log(u1) and
// the RateCorrector factor (KineticMcFirstOmp.cpp:79-82, RateCorrector.hpp:17-24).
__device__ void DrawStep(JumpLds &L, const ReplicaLds &Q) {
  const U4 u = Philox4x32_10(Q.seed, Q.steps, Q.rid, 0u);
  L.u2 = UnitOpenRight(Join64(u.z, u.w));
  L.log_u1 = log(UnitOpenLeft(Join64(u.x, u.y)));
  L.corr = (Q.flags & 1) ? Q.cv / (1.64 * exp(-(0.66 / kBoltzmann / Q.T - 0.7))) / (1 - 13 * Q.cs)
                         : 1.0;
}

// Phase 4 (lanes i < 12): lane i divides rate i by the total (KineticMcFirstOmp.cpp:69-77);
// lane 0 then forms the ordered cumulative probabilities and takes the first one >= u2, or event
// 11 when there is none (KineticMcAbstract.cpp:106-123), and the residence time
// (KineticMcFirstOmp.cpp:79-82). Returns true on lane 0 with the event's rank.
__device__ __forceinline__ bool ChooseEvent(JumpLds &L, const ReplicaLds &Q, int i, int &sel,
                                            double &dt) {
  double total = 0.0;
#pragma unroll
  for (int j = 0; j < 12; ++j) total += L.rate[j];
  L.prob[i] = L.rate[i] / total;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (i != 0) return false;
  const double u2 = L.u2;
  double cum = 0.0;
  sel = 11;
#pragma unroll
  for (int j = 0; j < 11; ++j) {
    cum += L.prob[j];
    if (sel == 11 && !(cum < u2)) sel = j;
  }
  dt = -L.log_u1 / total / kPrefactor;
  if (Q.flags & 1) dt *= L.corr;
  return true;
}

// One lane: advances the clock and applies a jump of the vacancy to site `jump` (offset
// dx, dy, dz; migrating species mig) with barrier ea and energy change de
// (KineticMcAbstract.cpp:147-181). `escaped`: IsEscaped of the step.
// kRecord: atom tracking and log records are compiled in (taken when k.atom / k.log_every are
// set); kernels launched without either use the variant without them.
template <bool kRecord = true>
__device__ void ApplyJump(const KTables &t, const KmcDev &k, ReplicaLds &Q, uint8_t *occ, int r,
                          uint64_t trace_index, int64_t jump, int dx, int dy, int dz, int mig,
                          double ea, double de, double dt, bool escaped) {
  if (escaped) {
    if (k.esc_time) {
      k.esc_time[r] = Q.time;
      k.esc_step[r] = Q.steps;
      k.esc_site[r] = Q.vac;
    }
    Q.esc = 1;
    Q.steps = Q.max_steps + 1;
  }
  if (kRecord && k.log_every && LogDue(Q.steps, k.log_every)) LogStep(k, Q, r, jump, ea, de);
  if (trace_index < k.trace_cap) {
    const uint64_t o = static_cast<uint64_t>(r) * k.trace_cap + trace_index;
    k.tr_sel[o] = jump;
    k.tr_ea[o] = ea;
    k.tr_de[o] = de;
    k.tr_time[o] = Q.time + dt;
  }
  Q.time += dt;
  Q.energy += de;
  Q.abse += de;
  if ((Q.flags & 4) && mig != Q.solvent) {  // solute COM (KineticMcAbstract.cpp:163-177)
    const double wgt = k.mass[mig] / Q.smass;
    Q.com[0] -= dx * kHalfLattice * wgt;
    Q.com[1] -= dy * kHalfLattice * wgt;
    Q.com[2] -= dz * kHalfLattice * wgt;
  }
  if (kRecord && k.atom) {  // the vacancy at Q.vac is the lhs of the reference's jump pair
    const int64_t o = k.off[r];
    const int m = Q.m2, h = m >> 1;
    AtomJump(k.atom + o, k.shift + 3 * o, Q.vac, jump,
             ImageChange(Wrap(Q.vx + dx, m) - Q.vx, h), ImageChange(Wrap(Q.vy + dy, m) - Q.vy, h),
             ImageChange(Wrap(Q.vz + dz, m) - Q.vz, h));
  }
  Q.disp[0] += dx;
  Q.disp[1] += dy;
  Q.disp[2] += dz;
  Q.vx = Wrap(Q.vx + dx, Q.m2);
  Q.vy = Wrap(Q.vy + dy, Q.m2);
  Q.vz = Wrap(Q.vz + dz, Q.m2);
  occ[Q.vac] = static_cast<uint8_t>(mig);  // Config::LatticeJump (Config.cpp:431-456)
  occ[jump] = static_cast<uint8_t>(t.x_code);
  Q.steps += 1;
  Q.vac = jump;
  if (Q.steps > Q.max_steps || Q.esc) Q.done = 1;
}

// One lane: applies the chosen event `sel` of the first-order step with energy change de.
template <bool kRecord = true>
__device__ void ApplyEvent(const KTables &t, const KmcDev &k, const JumpLds &L, ReplicaLds &Q,
                           uint8_t *occ, int r, uint64_t trace_index, int sel, double dt,
                           double de) {
  bool all = false;
  if (Q.flags & 2) {  // IsEscaped (KineticMcAbstract.cpp:192-223)
    // walk the set bits of the shell mask without unrolling: an unrolled loop keeps one scalar
    // predicate per slot live through the whole kernel
    all = true;
    uint64_t m = t.vac_shell_mask;
#pragma unroll 1
    while (m && all) {
      const int j = __ffsll(static_cast<unsigned long long>(m)) - 1;
      m &= m - 1;
      all = L.env[0][j] == Q.solvent;
    }
  }
  const int dir = L.dir[sel];
  int dx, dy, dz;
  Unpack16(L.off[dir * kEnvSlots + t.n_slot], dx, dy, dz);
  ApplyJump<kRecord>(t, k, Q, occ, r, trace_index, L.snb[sel], dx, dy, dz, L.env[dir][t.n_slot], L.ea[sel],
            de, dt, all);
}

}  // namespace
}  // namespace lmc
