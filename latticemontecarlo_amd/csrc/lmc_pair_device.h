// Device side of the quadratic jump evaluation (lmc_pairs.h): the 12 jumps of a vacancy from the
// non-reference sites around it.
//
//   1. Read the 134 sites of the 12 environments: three loads per lane of one wave.
//   2. List the sites that do not hold the reference species (ballots).
//   3. Add their one-site terms to the 12 events, and find the pairs of them within three shells of
//      each other (one squared distance per lane, 64 pairs at a time). Lane l works on event l % 16
//      with the list entries l / 16, l / 16 + 4, ...: the sites' slots in the event's environment,
//      the class of the slot pair, its dE and logit values.
//   4. Add the pairs' terms the same way, then the four rows of 16 lanes (permlane swaps), so that
//      every row holds the 12 sums.
// At 6 at.% solute that is 8 sites and 8 pairs of 134 sites, where summing every cluster takes
// 13 044 table reads. An environment with more than kMaxSparse non-reference sites is summed over
// the 614 slot pairs that have a term instead.
//
// Measured, 1 024 replicas of 20^3 cells (E0, 2-10 at.% solute), per step of the slowest replica: 2.4 us,
// against 6.3 us of summing every cluster with 256 threads per replica (12.6 -> 4.7 ms per 2 000 steps;
// 700 instructions and 4 700 cycles of a wave); 384 000 jumps of an exit-time scan 36 against 254 us.
// kMaxSparse: a step by the dense sums takes 5.9 us at any composition (summing every cluster: 6.6 us). The
// line at 24, 32, 40 and 48 sites gives, with one wave per replica (1 024 replicas), 5.7, 4.8, 4.1 and 4.1 us
// at 2-9 at.% of each solute and 5.8, 5.8, 5.9 and 6.8 us at 3-15 %; with four (128 replicas) 2.7, 2.3, 2.3
// and 2.3 us, and 2.7, 2.7, 2.8 and 3.0 us.
//
// One wave has a SIMD to itself in the batches of interest, so a step's time is its instruction count
// times the issue interval plus the exposed latencies: list writes go to a spare element instead of
// branching, the first batch of one-site terms and the first 64 pairs share a block of straight
// code, and rare conditions cost one scalar branch.
#pragma once
#include <hip/hip_runtime.h>

#include "lmc_dev_common.h"
#include "lmc_device.h"
#include "lmc_pairs.h"
#include "lmc_replica.h"

namespace lmc {
namespace {

constexpr int kMaxSparse = 40;
constexpr int kBatch = 4;               // list entries per lane and batch
constexpr int kSolPad = 16 * kBatch;    // blank entries after the list, for whole batches
constexpr int kEntries = 256;           // pair list of a wave; emptied when 64 more might not fit

// Working set of one replica.
struct TeamLds {
  uint2 sol[kMaxSparse + kSolPad + 2];  // packed offset; site | diagonal value offset << 8 |
                                        // q-rank << 16 | |offset|^2 << 24
  // dense sums: by site, q * q-rank | q-rank << 8 (reference: 16 | 32 << 8); the two by slot for the
  // events of three directions, a byte each; migrating rank by direction. Environment rows: species.
  uint16_t code[kPairSiteRow];
  uint32_t era[4 * kEnvSlots], erb[4 * kEnvSlots];
  uint8_t mig[12];
};
// Working set of one wave: pair entries site1 | site2 << 8 | value offset << 16; dense sums by
// direction.
struct WaveLds {
  uint32_t ent[kEntries + 64 + 4];
  double sum[12][3];
};

// Geometry tables of a workgroup, each where 16-byte copies may start.
template <bool kQ>
struct PairShared {
  alignas(16) uint32_t cls[(kNoSlot + 1) * kClsRow];
  alignas(16) uint16_t clsb[kQ ? (kNoSlot + 1) * kClsRow : 8];
  alignas(16) uint32_t one[12 * kOneRow];     // cls of a site's slot with itself
  alignas(16) uint16_t oneb[kQ ? 12 * kOneRow : 8];
  alignas(16) uint8_t slot[12 * kPairSiteRow];
  alignas(16) uint8_t order[27 * 16];         // event directions by the faces the vacancy touches
  alignas(16) uint2 dense[kMaxDense];         // slot pairs with a term: cls; 16 s1 | 16 s2 << 16
  alignas(16) uint16_t denseb[kQ ? kMaxDense : 8];
  alignas(16) uint32_t site3[4 * kEnvSlots];
  double base[5 * 3], par[kMaxSpecies * 6];
};

// Where the value tables lie in dynamic LDS (bytes). tab_lds: kGlobal none of them, kShared all, kMixed dE and MMM.
constexpr int kGlobal = 0, kShared = 1, kMixed = 2;
struct PairLayout {
  int de, la, lb, bytes, tab_lds;
};

// Resolved value tables of one reference species, [migrating rank][row].
struct PairTab {
  const char *de, *la, *lb;
  int de_row, la_row, lb_row;  // bytes
  int q;                       // non-reference elements
  uint32_t sol_mul;            // the q-rank's fields of a site's list entry
  uint32_t qlut;               // q-rank by species code, 4 bits each; 15: the reference
};

__device__ __forceinline__ int LaneId() { return static_cast<int>(threadIdx.x) & 63; }
// Number of set bits of a wave mask below this lane.
__device__ __forceinline__ int RankInMask(uint64_t m) {
  return static_cast<int>(__builtin_amdgcn_mbcnt_hi(static_cast<uint32_t>(m >> 32),
                          __builtin_amdgcn_mbcnt_lo(static_cast<uint32_t>(m), 0u)));
}

// Copies `bytes` (a multiple of 4; both sides 16-byte aligned: the blob's tables lie 256 bytes apart and
// the parts of a PairBlock start on 16 bytes) to LDS, 16 bytes per thread and
// load, four loads in flight: the copy is bound by the latency of its few rounds.
__device__ __forceinline__ void CopyTable(char *dst, const void *src, int bytes, int tid, int size) {
  const uint4 *s = reinterpret_cast<const uint4 *>(src);
  uint4 *d = reinterpret_cast<uint4 *>(dst);
  const int n = bytes >> 4;
  int i = tid;
  for (; i + 3 * size < n; i += 4 * size) {
    uint4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) v[u] = s[i + u * size];
#pragma unroll
    for (int u = 0; u < 4; ++u) d[i + u * size] = v[u];
  }
  for (; i < n; i += size) d[i] = s[i];
  for (int j = (n << 2) + tid; j < (bytes >> 2); j += size)
    reinterpret_cast<uint32_t *>(dst)[j] = reinterpret_cast<const uint32_t *>(src)[j];
}

// The workgroup's tables for reference species code `ref` into LDS (all threads; the caller
// synchronises). kTab: where the value tables go; what stays in global memory is read there.
template <bool kQ, int kTab>
__device__ __forceinline__ PairTab LoadPairTables(const KTables &t, PairShared<kQ> &G, char *dyn,
                                                  const PairLayout &lay, int ref, int tid, int size) {
  const int rr = static_cast<int>((t.rank_lut >> (4 * ref)) & 15u);
  PairTab T;
  T.q = t.ne > 1 ? t.ne - 1 : 1;
  T.sol_mul = (1u << 16) | (static_cast<uint32_t>(8 * (T.q + 1)) << 8);
  T.de_row = 8 * t.de_row;
  T.la_row = 8 * t.la_row;
  T.lb_row = 8 * t.lb_row;
  T.qlut = 0;
  for (int c = 0; c < t.S; ++c) {
    const int r = static_cast<int>((t.rank_lut >> (4 * c)) & 15u);
    T.qlut |= static_cast<uint32_t>(r == rr ? 15 : r - (r > rr ? 1 : 0)) << (4 * c);
  }
  CopyTable(reinterpret_cast<char *>(G.cls), t.cls, sizeof(G.cls), tid, size);
  CopyTable(reinterpret_cast<char *>(G.one), t.one, sizeof(G.one), tid, size);
  CopyTable(reinterpret_cast<char *>(G.slot), t.slot, sizeof(G.slot), tid, size);
  CopyTable(reinterpret_cast<char *>(G.order), t.order, sizeof(G.order), tid, size);
  CopyTable(reinterpret_cast<char *>(G.dense), t.dense, sizeof(G.dense), tid, size);
  CopyTable(reinterpret_cast<char *>(G.site3), t.site3, sizeof(G.site3), tid, size);
  if (kQ) {
    CopyTable(reinterpret_cast<char *>(G.clsb), t.clsb, sizeof(G.clsb), tid, size);
    CopyTable(reinterpret_cast<char *>(G.oneb), t.oneb, sizeof(G.oneb), tid, size);
    CopyTable(reinterpret_cast<char *>(G.denseb), t.denseb, sizeof(G.denseb), tid, size);
  }
  // the first reference's block, then the others' by rank
  const PairBlock at = PairBlockOf(t.ne, t.de_row, t.la_row, t.lb_row);
  const double *v = t.pairs + (rr == t.first_ref ? 0 : rr + (rr < t.first_ref ? 1 : 0)) * at.size;
  for (int i = tid; i < 3 * t.ne; i += size) G.base[i] = v[at.base + i];
  for (int i = tid; i < 6 * t.S; i += size) G.par[i] = t.par[i];
  const char *de = reinterpret_cast<const char *>(v);
  const char *la = reinterpret_cast<const char *>(v + at.la);
  const char *lb = reinterpret_cast<const char *>(v + at.lb);
  T.de = de;
  T.la = la;
  T.lb = lb;
  if (kTab != kGlobal) {
    CopyTable(dyn + lay.de, de, t.ne * T.de_row, tid, size);
    CopyTable(dyn + lay.la, la, t.ne * T.la_row, tid, size);
    T.de = dyn + lay.de;
    T.la = dyn + lay.la;
  }
  if (kQ && kTab == kShared) {
    CopyTable(dyn + lay.lb, lb, t.ne * T.lb_row, tid, size);
    T.lb = dyn + lay.lb;
  }
  return T;
}

// The lane's sites (lane, lane + 64, lane + 128; lanes past the last site repeat site 0, or with kOwn have
// the vacancy's own, whose species is then checked too) and the pair of list entries it tests first,
// read once per launch.
struct LaneSites {
  int32_t pk[3];
  uint32_t word[3];  // site | |offset|^2 << 24
  uint32_t move;     // lanes 0 .. 11: the jump's components plus one, two bits each, from bit 16
  int i, j;          // pair number wave * 64 + lane: i (i - 1) / 2 + j, j < i
};
// The pair of a pair number: the root is exact at every i, the half bounds its rounding.
__device__ __forceinline__ void PairOf(int p, int &i, int &j) {
  i = static_cast<int>((__builtin_amdgcn_sqrtf(8.0f * p + 1.5f) + 1.0f) * 0.5f);
  j = p - ((i * (i - 1)) >> 1);
}
template <bool kOwn = false>
__device__ __forceinline__ LaneSites LoadSites(const KTables &t, int wv) {
  LaneSites s;
  const int lane = LaneId();
#pragma unroll
  for (int u = 0; u < 3; ++u) {
    const bool in = lane + 64 * u < kPairSites;
    s.pk[u] = kOwn && !in ? 0 : t.site_pk[in ? lane + 64 * u : 0];
    const uint32_t r2 = static_cast<uint32_t>(__builtin_amdgcn_sdot4(s.pk[u], s.pk[u], 0, false));
    s.word[u] = static_cast<uint32_t>(lane + 64 * u) | (r2 << 24);
  }
  PairOf(64 * wv + lane, s.i, s.j);
  s.move = 0;
#pragma unroll
  for (int c = 0; c < 3; ++c)
    s.move |= ((static_cast<uint32_t>(s.pk[0] >> (8 * c)) + 1u) & 3u) << (16 + 2 * c);
  return s;
}
// Lanes whose third site exists.
constexpr uint64_t kThirdMask = (1ull << (kPairSites - 128)) - 1;

// v in [-m, 2m) on the periodic axis of m steps: the out-of-range candidates are huge unsigned.
__device__ __forceinline__ uint32_t WrapMin(uint32_t v, uint32_t m) { return min(min(v, v + m), v - m); }

// Wrapped coordinates of packed offset pk from c, and the site id of coordinates. Id: uint32_t for
// boxes of at most 1000^3 cells.
struct Coords {
  uint32_t x, y, z;
};
__device__ __forceinline__ Coords WrapSite(const XYZ &c, uint32_t n, int32_t pk) {
  const uint32_t m = 2 * n;
  return {WrapMin(static_cast<uint32_t>(c.X + static_cast<int8_t>(pk)), m),
          WrapMin(static_cast<uint32_t>(c.Y + static_cast<int8_t>(pk >> 8)), m),
          WrapMin(static_cast<uint32_t>(c.Z + static_cast<int8_t>(pk >> 16)), m)};
}
template <typename Id>
__device__ __forceinline__ Id SiteId(const Coords &s, uint32_t n) {
  const uint32_t m = 2 * n;
  if constexpr (sizeof(Id) == 4) return __umul24(s.x, m * n) + (__umul24(s.y, n) + (s.z >> 1));
  else return static_cast<Id>(s.x) * (static_cast<Id>(m) * n) + (static_cast<Id>(s.y) * n + (s.z >> 1));
}

// Site ids and species of the lane's sites around c (the loads are only issued here), and the
// coordinates of its first one (lanes 0 .. 11: the first neighbours).
template <typename Id>
struct Around {
  Id id[3];
  int code[3];
  Coords near;
};
template <typename Id>
__device__ __forceinline__ void GatherAround(const LaneSites &s, const uint8_t *occ, int n,
                                             const XYZ &c, Around<Id> &a) {
#pragma unroll
  for (int u = 0; u < 3; ++u) {
    const Coords w = WrapSite(c, static_cast<uint32_t>(n), s.pk[u]);
    if (u == 0) a.near = w;
    a.id[u] = SiteId<Id>(w, static_cast<uint32_t>(n));
    a.code[u] = occ[a.id[u]];
  }
}

// Replaces the species read at lattice site `site`.
template <typename Id>
__device__ __forceinline__ void Substitute(Around<Id> &a, Id site, int code) {
#pragma unroll
  for (int u = 0; u < 3; ++u) a.code[u] = a.id[u] == site ? code : a.code[u];
}

__device__ __forceinline__ int Bpermute(int lane, int v) { return __builtin_amdgcn_ds_bpermute(4 * lane, v); }
__device__ __forceinline__ uint64_t Bpermute64(int lane, uint64_t v) {
  const uint32_t lo = static_cast<uint32_t>(Bpermute(lane, static_cast<int>(v)));
  const uint32_t hi = static_cast<uint32_t>(Bpermute(lane, static_cast<int>(v >> 32)));
  return lo | (static_cast<uint64_t>(hi) << 32);
}
__device__ __forceinline__ int ReadLaneInt(int v, int lane) { return __builtin_amdgcn_readlane(v, lane); }

// Direction of the event of this lane (lane % 16, neighbour ids ascending; lanes past 11 repeat
// event 11). Directions are in (x, y, z) order, which is the id order of the neighbours unless one
// lies across a box face; the table holds the order for each case (an axis: inside, at 0, at the top).
template <bool kQ>
__device__ __forceinline__ int EventDirection(const PairShared<kQ> &G, const XYZ &c, int n) {
  const int top = 2 * n - 1;
  auto face = [&](int v) { return v == 0 ? 1 : v == top ? 2 : 0; };
  return G.order[16 * (face(c.X) + 3 * face(c.Y) + 9 * face(c.Z)) + (LaneId() & 15)];
}

// Sum over the lane's column (lanes l, l ^ 16, l ^ 32, l ^ 48), the same in all four rows.
__device__ __forceinline__ double RowsSum(double v) {
  const uint32_t lo = static_cast<uint32_t>(__double2loint(v)), hi = static_cast<uint32_t>(__double2hiint(v));
  const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  const double s = __hiloint2double(static_cast<int>(h[0]), static_cast<int>(l[0])) +
                   __hiloint2double(static_cast<int>(h[1]), static_cast<int>(l[1]));
  const uint32_t slo = static_cast<uint32_t>(__double2loint(s)), shi = static_cast<uint32_t>(__double2hiint(s));
  const auto l2 = __builtin_amdgcn_permlane32_swap(slo, slo, false, false);
  const auto h2 = __builtin_amdgcn_permlane32_swap(shi, shi, false, false);
  return __hiloint2double(static_cast<int>(h2[0]), static_cast<int>(l2[0])) +
         __hiloint2double(static_cast<int>(h2[1]), static_cast<int>(l2[1]));
}

// Inclusive sums within each row of 16 lanes.
__device__ __forceinline__ double RowScan(double v) {
  v += RowShr<1>(v);
  v += RowShr<2>(v);
  v += RowShr<4>(v);
  v += RowShr<8>(v);
  return v;
}

struct PairSums {
  double de, la, lb;
};

// Values of one batch: the loads of all its terms, then the additions.
template <bool kQ, int kN>
struct Values {
  double de[kN], la[kN], lb[kQ ? kN : 1];
  __device__ __forceinline__ void Load(int u, const char *pd, const char *pl, const char *pb) {
    de[u] = *reinterpret_cast<const double *>(pd);
    la[u] = *reinterpret_cast<const double *>(pl);
    if (kQ) lb[u] = *reinterpret_cast<const double *>(pb);
  }
};

// Per-lane views for the event the lane works on: migrating species, its value rows, slots.
struct EventRow {
  int dir, M;
  const char *de, *la, *lb;
};
template <bool kQ>
__device__ __forceinline__ EventRow MakeRow(const KTables &t, const PairTab &T, int dir, int M) {
  const int mr = static_cast<int>((t.rank_lut >> (4 * M)) & 15u);
  return {dir, M, T.de + __umul24(mr, T.de_row), T.la + __umul24(mr, T.la_row),
          kQ ? T.lb + __umul24(mr, T.lb_row) : nullptr};
}

// Lists the non-reference sites of `a` in S.sol with blanks after them; returns their number
// (uniform). With more than kMax, the inputs of DenseTerms are formed instead.
template <bool kQ, int kMax = kMaxSparse, typename Id>
__device__ __forceinline__ int ListSites(const KTables &t, const PairShared<kQ> &G, const PairTab &T, TeamLds &S,
                                         const LaneSites &ls, const Around<Id> &a) {
  const int lane = LaneId();
  uint64_t mask[3];
  int qr[3], K = 0;
#pragma unroll
  for (int u = 0; u < 3; ++u) {
    qr[u] = static_cast<int>((T.qlut >> (4 * a.code[u])) & 15u);
    mask[u] = __ballot(qr[u] != 15);
    if (u == 2) mask[u] &= kThirdMask;
    K += __builtin_popcountll(mask[u]);
  }
  if (K <= kMax) {
    int at = 0;
#pragma unroll
    for (int u = 0; u < 3; ++u) {
      const int rank = at + RankInMask(mask[u]);
      const bool on = u == 2 ? qr[u] != 15 && lane < kPairSites - 128 : qr[u] != 15;
      S.sol[on ? rank : kMaxSparse + kSolPad] =
          make_uint2(static_cast<uint32_t>(ls.pk[u]), __umul24(qr[u], T.sol_mul) + ls.word[u]);
      at += __builtin_popcountll(mask[u]);
    }
    S.sol[K + lane] = make_uint2(0u, kPairSites);  // kSolPad blanks
  } else {
#pragma unroll
    for (int u = 0; u < 3; ++u)
      if (lane + 64 * u < kPairSites)
        S.code[lane + 64 * u] = static_cast<uint16_t>(qr[u] == 15 ? 16 | (32 << 8) : T.q * qr[u] | (qr[u] << 8));
    if (lane == 0) S.code[kPairSites] = 16 | (32 << 8);
    if (lane < 12) S.mig[lane] = static_cast<uint8_t>((t.rank_lut >> (4 * a.code[0])) & 15u);
    WaveFence();
#pragma unroll
    for (int i = lane; i < 4 * kEnvSlots; i += 64) {
      const uint32_t s3 = G.site3[i];
      const uint32_t x = S.code[s3 & 255u], y = S.code[(s3 >> 8) & 255u], z = S.code[(s3 >> 16) & 255u];
      S.era[i] = (x & 255u) | ((y & 255u) << 8) | ((z & 255u) << 16);
      S.erb[i] = (x >> 8) | (y & 0xFF00u) | ((z & 0xFF00u) << 8);
    }
  }
  WaveFence();
  return K;
}

template <bool kQ, int kN>
__device__ __forceinline__ void AddValues(const Values<kQ, kN> &w, PairSums &s) {
#pragma unroll
  for (int u = 0; u < kN; ++u) {
    s.de += w.de[u];
    s.la += w.la[u];
    if (kQ) s.lb += w.lb[u];
  }
}

// A batch of one-site terms (list entries p, p + kSubs, ...) and one of pair terms (entries p, p + 4,
// ... of the wave's list), in stages: list entries, [slots,] classes, values, sums.
template <bool kQ, int kN, int kSubs>
struct SiteBatch {
  uint32_t y[kN], c[kN], cb[kQ ? kN : 1];
  Values<kQ, kN> w;
  __device__ __forceinline__ void Entries(const TeamLds &S, int p) {
#pragma unroll
    for (int u = 0; u < kN; ++u) y[u] = S.sol[p + u * kSubs].y;
  }
  __device__ __forceinline__ void Classes(const PairShared<kQ> &G, const EventRow &R) {
#pragma unroll
    for (int u = 0; u < kN; ++u) {
      const int at = R.dir * kOneRow + (y[u] & 255u);
      c[u] = G.one[at];
      if (kQ) cb[u] = G.oneb[at];
    }
  }
  __device__ __forceinline__ void Load(const EventRow &R) {
#pragma unroll
    for (int u = 0; u < kN; ++u) {
      const uint32_t v = (y[u] >> 8) & 255u;
      w.Load(u, R.de + ((c[u] & 0xFFFFu) + v), R.la + ((c[u] >> 16) + v), kQ ? R.lb + (cb[u] + v) : nullptr);
    }
  }
};
template <bool kQ>
struct PairBatch {
  uint32_t e[kBatch], s1[kBatch], s2[kBatch], c[kBatch], cb[kQ ? kBatch : 1];
  Values<kQ, kBatch> w;
  __device__ __forceinline__ void Entries(const WaveLds &W, int p) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u) e[u] = W.ent[p + 4 * u];
  }
  __device__ __forceinline__ void Slots(const uint8_t *slots) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      s1[u] = slots[e[u] & 255u];
      s2[u] = slots[(e[u] >> 8) & 255u];
    }
  }
  __device__ __forceinline__ void Classes(const PairShared<kQ> &G) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const uint32_t at = s1[u] * kClsRow + s2[u];
      c[u] = G.cls[at];
      if (kQ) cb[u] = G.clsb[at];
    }
  }
  __device__ __forceinline__ void Load(const EventRow &R) {
#pragma unroll
    for (int u = 0; u < kBatch; ++u) {
      const uint32_t v = e[u] >> 16;
      w.Load(u, R.de + ((c[u] & 0xFFFFu) + v), R.la + ((c[u] >> 16) + v), kQ ? R.lb + (cb[u] + v) : nullptr);
    }
  }
};

// The pair terms of the wave's entries [from, cnt), rows row, row + 4, ... (blanks are appended here).
template <bool kQ>
__device__ __forceinline__ void AddPairs(const PairShared<kQ> &G, WaveLds &W, int from, int cnt,
                                         const EventRow &R, PairSums &s) {
  const int lane = LaneId(), row = lane >> 4;
  W.ent[cnt + lane] = kPairSites | (kPairSites << 8);
  const uint8_t *slots = G.slot + R.dir * kPairSiteRow;
  for (int p0 = from; p0 < cnt; p0 += 4 * kBatch) {
    WaveFence();
    PairBatch<kQ> b;
    b.Entries(W, p0 + row);
    Stage();
    b.Slots(slots);
    Stage();
    b.Classes(G);
    Stage();
    b.Load(R);
    Stage();
    AddValues(b.w, s);
  }
}

// A near-pair test of list entries x and y: the pair's entry goes to the end of the wave's list.
// Returns the list's new length.
__device__ __forceinline__ int AppendPair(WaveLds &W, int q, const uint2 &x, const uint2 &y, bool on, int cnt) {
  const int r2 = static_cast<int>((x.y >> 24) + (y.y >> 24)) -
                 2 * __builtin_amdgcn_sdot4(static_cast<int>(x.x), static_cast<int>(y.x), 0, false);
  const bool hit = on && r2 <= 6;
  const uint64_t m = __ballot(hit);
  const uint32_t qx = (x.y >> 16) & 255u, qy = (y.y >> 16) & 255u;
  W.ent[hit ? cnt + RankInMask(m) : kEntries + 64] =
      (x.y & 255u) | ((y.y & 255u) << 8) | ((8 * (__umul24(qx, q) + qy)) << 16);
  return cnt + __builtin_popcountll(m);
}

// The sums over the 614 slot pairs with a term, for environments with many non-reference sites: lane l
// works on the pairs l % 16, l % 16 + 16, ... of its wave's share and the three directions 3 (l / 16)
// .. + 2, so that a pair's class and both slots are read once for three events and no lane is idle.
// The rows' sums meet in W.sum.
template <bool kQ, int kWaves>
__device__ __forceinline__ PairSums DenseTerms(const PairShared<kQ> &G, const PairTab &T, const TeamLds &S,
                                               WaveLds &W, int dir, int wv) {
  const int lane = LaneId(), g = lane >> 4;
  double de[3] = {0, 0, 0}, la[3] = {0, 0, 0}, lb[3] = {0, 0, 0};
  const char *rd[3], *rl[3], *rb[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int mr = S.mig[3 * g + i];
    rd[i] = T.de + __umul24(mr, T.de_row);
    rl[i] = T.la + __umul24(mr, T.la_row);
    rb[i] = kQ ? T.lb + __umul24(mr, T.lb_row) : nullptr;
  }
  const uint32_t zero = static_cast<uint32_t>(T.q * T.q);  // the zero after a block's values
  const char *ea = reinterpret_cast<const char *>(S.era + g), *eb = reinterpret_cast<const char *>(S.erb + g);
  constexpr int kU = 5;
  static_assert(kMaxDense % (16 * kWaves * kU) == 0, "whole batches");
  for (int p = 16 * wv + (lane & 15); p < kMaxDense; p += 16 * kWaves * kU) {
    uint2 d[kU];
    uint32_t x[kU], cb[kU];
    Values<kQ, 3 * kU> w;
#pragma unroll
    for (int u = 0; u < kU; ++u) {
      d[u] = G.dense[p + 16 * kWaves * u];
      if (kQ) cb[u] = G.denseb[p + 16 * kWaves * u];
    }
    Stage();
#pragma unroll
    for (int u = 0; u < kU; ++u)
      x[u] = *reinterpret_cast<const uint32_t *>(ea + (d[u].y & 0xFFFFu)) +
             *reinterpret_cast<const uint32_t *>(eb + (d[u].y >> 16));
    Stage();
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const uint32_t v = 8 * min((x[u] >> (8 * i)) & 255u, zero);
        w.Load(3 * u + i, rd[i] + ((d[u].x & 0xFFFFu) + v), rl[i] + ((d[u].x >> 16) + v),
               kQ ? rb[i] + (cb[u] + v) : nullptr);
      }
    Stage();
#pragma unroll
    for (int u = 0; u < kU; ++u)
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        de[i] += w.de[3 * u + i];
        la[i] += w.la[3 * u + i];
        if (kQ) lb[i] += w.lb[3 * u + i];
      }
  }
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    de[i] = RowScan(de[i]);
    la[i] = RowScan(la[i]);
    if (kQ) lb[i] = RowScan(lb[i]);
    if ((lane & 15) == 15) {
      W.sum[3 * g + i][0] = de[i];
      W.sum[3 * g + i][1] = la[i];
      W.sum[3 * g + i][2] = lb[i];
    }
  }
  WaveFence();
  return {W.sum[dir][0], W.sum[dir][1], W.sum[dir][2]};
}

// The cluster sums of the lane's event without their base: this wave's share of the K listed sites
// and their pairs (kWaves waves share them; wave `wv` of them), the same in all four rows.
template <bool kQ, int kWaves>
__device__ __forceinline__ PairSums PairTerms(const PairShared<kQ> &G, const PairTab &T, const TeamLds &S,
                                              WaveLds &W, const LaneSites &ls, int K, const EventRow &R,
                                              int wv) {
  constexpr int kSubs = 4 * kWaves, kFirst = kWaves == 1 ? kBatch : 1;
  if (K > kMaxSparse) return DenseTerms<kQ, kWaves>(G, T, S, W, R.dir, wv);
  const int lane = LaneId(), row = lane >> 4, sub = 4 * wv + row;
  PairSums s{0.0, 0.0, 0.0};
  // The first 16 sites, the first 64 pairs of the wave and the first 16 near ones in one block: the
  // sites' look-ups run under the pairs'.
  SiteBatch<kQ, kFirst, kSubs> a;
  PairBatch<kQ> b;
  a.Entries(S, sub);
  const bool on = ls.i < K;
  const uint2 x = S.sol[on ? ls.i : 0], y = S.sol[on ? ls.j : 0];
  Stage();
  a.Classes(G, R);
  int cnt = AppendPair(W, T.q, x, y, on, 0);
  W.ent[cnt + lane] = kPairSites | (kPairSites << 8);
  WaveFence();
  b.Entries(W, row);
  Stage();
  b.Slots(G.slot + R.dir * kPairSiteRow);
  a.Load(R);
  Stage();
  b.Classes(G);
  Stage();
  b.Load(R);
  AddValues(a.w, s);
  Stage();
  AddValues(b.w, s);
  // what is left of the sites, the pairs and the near ones
  for (int p = sub + kSubs * kFirst; p < K + sub; p += kSubs * kFirst) {  // uniform trip count
    SiteBatch<kQ, kFirst, kSubs> r;
    r.Entries(S, p);
    Stage();
    r.Classes(G, R);
    Stage();
    r.Load(R);
    Stage();
    AddValues(r.w, s);
  }
  int from = 4 * kBatch;
  if (K * (K - 1) / 2 > 64 * kWaves) {
    cnt = cnt > from ? cnt : from;  // entries below `from` are done, or blank
    for (int p0 = 64 * (kWaves + wv); p0 < K * (K - 1) / 2; p0 += 64 * kWaves) {
      int i, j;
      PairOf(p0 + lane, i, j);
      const bool in = i < K;
      cnt = AppendPair(W, T.q, S.sol[in ? i : 0], S.sol[in ? j : 0], in, cnt);
      if (cnt > kEntries - 64) {  // uniform
        AddPairs<kQ>(G, W, from, cnt, R, s);
        WaveFence();
        cnt = from = 0;
      }
    }
  }
  if (cnt > from) AddPairs<kQ>(G, W, from, cnt, R, s);
  WaveFence();
  s.de = RowsSum(s.de);
  s.la = RowsSum(s.la);
  if (kQ) s.lb = RowsSum(s.lb);
  return s;
}

// The energy change of one event, added cluster by cluster in the order of the state list: 84 running
// sums (of entries c, c + 84, ...), the four that are 21 apart added two and two, then the 21 results
// one after another. A trajectory whose changes cancel (a vacancy among solvent atoms, or back at its
// start) has nothing but the rounding of these sums in its energy, so that a small batch's energies keep
// this order; the quadratic form, which decides the rates, adds in another one. One wave: lanes 2 i and
// 2 i + 1 hold the four running sums i, i + 21, i + 42 and i + 63.
constexpr int kOrderedRounds = kMaxStateClusters / kClusterPad;
struct OrderedLds {  // element ranks of the event's slots, as the entries of t.state index them
  uint16_t rn8[64];  // rank * 8 * ne
  uint8_t r8[64];    // rank * 8
};
struct OrderedClusters {
  uint32_t entry[2][kOrderedRounds];  // the lane's
};
__device__ __forceinline__ OrderedClusters LoadOrdered(const KTables &t) {
  const int lane = LaneId(), half = lane < 42 ? lane : 41;  // lanes past the last sum repeat it
  const uint32_t *list = t.state + (half >> 1) + 42 * (half & 1);
  OrderedClusters o;
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int b = 0; b < kOrderedRounds; ++b) o.entry[j][b] = list[21 * j + kClusterPad * b];
  return o;
}
// The event whose slot s = lane holds species `code`; M: migrating species; w: the rows of t.wd.
__device__ __forceinline__ double OrderedDe(const KTables &t, const OrderedClusters &o, OrderedLds &D, int code,
                                            const char *w, int M) {
  const int lane = LaneId();
  const uint32_t rank = lane < kEnvSlots ? (t.rank_lut >> (4 * code)) & 15u : 0u;
  D.r8[lane] = static_cast<uint8_t>(rank << 3);
  D.rn8[lane] = static_cast<uint16_t>(__umul24(rank, 8 * t.ne));
  WaveFence();
  const char *row = w + __umul24((t.rank_lut >> (4 * M)) & 15u, 8 * t.wrow);
  uint32_t at[2][kOrderedRounds];
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int b = 0; b < kOrderedRounds; ++b) {
      const uint32_t e = o.entry[j][b];
      at[j][b] = D.r8[e & 255u] + D.rn8[(e >> 9) & 127u] + (e >> 16);
    }
  double v[2] = {0.0, 0.0};
#pragma unroll
  for (int b = 0; b < kOrderedRounds; ++b)
#pragma unroll
    for (int j = 0; j < 2; ++j) v[j] += *reinterpret_cast<const double *>(row + at[j][b]);
  double four = v[0] + v[1];
  four += PairLane(four);
  double sum = 0.0;
#pragma unroll
  for (int i = 0; i < 21; ++i) sum += ReadLane(four, 2 * i);
  WaveFence();
  return sum;
}

// exp: x = k ln 2 + r by Cody and Waite's two-part reduction, the Taylor series to r^13 (truncation below
// 2^-57 at |r| = ln 2 / 2) in even and odd halves, then the scaling by 2^k, which takes care of overflow
// and gradual underflow. NaN stays NaN. The same fused steps on 6e7 arguments up to 708 either way are at
// most 1.04 units in the last place off. The constants are made opaque so that they stay in vector
// registers: as literals each would take two scalar moves at every use.
struct ExpConst {
  double log2e, hi, lo, c[12];  // c[i] = 1 / (i + 2)!
};
__device__ __forceinline__ ExpConst MakeExpConst() {
  ExpConst e{1.4426950408889634, 0x1.62e42fefa39efp-1, 0x1.abc9e3b39803fp-56, {}};
  double f = 1.0;
#pragma unroll
  for (int i = 0; i < 12; ++i) {
    f *= i + 2;
    e.c[i] = 1.0 / f;
  }
  asm volatile("" : "+v"(e.log2e), "+v"(e.hi), "+v"(e.lo));
#pragma unroll
  for (int i = 0; i < 12; ++i) asm volatile("" : "+v"(e.c[i]));
  return e;
}
__device__ __forceinline__ double Exp(const ExpConst &E, double x) {
  double y = x > 2000.0 ? 2000.0 : x;
  y = y < -2000.0 ? -2000.0 : y;
  const double k = rint(y * E.log2e);
  const double r = fma(-k, E.lo, fma(-k, E.hi, y));
  const double r2 = r * r;
  double even = E.c[10], odd = E.c[11];
#pragma unroll
  for (int i = 8; i >= 0; i -= 2) {
    even = fma(even, r2, E.c[i]);
    odd = fma(odd, r2, E.c[i + 1]);
  }
  const double p = fma(r2, fma(odd, r, even), r) + 1.0;
  return ldexp(p, static_cast<int>(k));
}

struct EventValue {
  double ea, de, ekra, la;
};

// What an event needs besides its sums, read ahead of them: all-reference sums and barrier parameters of
// the migrating species (the quartic model's two logits in the even and odd rows of the wave).
struct EventConst {
  double b[3], p[3];
};
template <bool kQ>
__device__ __forceinline__ EventConst LoadConst(const KTables &t, const PairShared<kQ> &G, int M) {
  const double *b = G.base + 3 * static_cast<int>((t.rank_lut >> (4 * M)) & 15u);
  const double *p = G.par + 6 * M + (kQ && (LaneId() & 16) ? 3 : 0);
  return {{b[0], b[1], kQ ? b[2] : 0.0}, {p[0], p[1], p[2]}};
}

// Ea, dE and E_kra of the lane's event from its sums. bad: the environment holds a vacancy off the
// jump's endpoints (no one-hot type; the reference throws).
// E0 = exp(logit * sigma_e0 + mu_e0), Ea = max(0, E0 + dE/2) (VacancyMigrationPredictorE0.cpp:
// 147-158); the quartic barrier of VacancyMigrationPredictorQuartic.cpp:266-275, whose two
// exponentials are taken side by side in the even and odd rows of the wave.
template <bool kQ>
__device__ __forceinline__ EventValue FinishEvent(const ExpConst &E, const EventConst &c, const PairSums &s,
                                                  bool bad) {
  EventValue e;
  e.de = c.b[0] + s.de;
  const double la = bad ? __builtin_nan("") : c.b[1] + s.la;
  e.la = la;
  if (!kQ) {
    e.ekra = Exp(E, (c.p[0] + la) * c.p[2] + c.p[1]);
    e.ea = fmax(0.0, e.ekra + e.de / 2);
    return e;
  }
  const double lb = c.b[2] + s.lb;
  const double x = Exp(E, (c.p[0] + ((LaneId() & 16) ? lb : la)) * c.p[2] + c.p[1]);
  const uint32_t lo = static_cast<uint32_t>(__double2loint(x)), hi = static_cast<uint32_t>(__double2hiint(x));
  const auto l = __builtin_amdgcn_permlane16_swap(lo, lo, false, false);
  const auto h = __builtin_amdgcn_permlane16_swap(hi, hi, false, false);
  const double D = __hiloint2double(static_cast<int>(h[0]), static_cast<int>(l[0]));
  const double Ks = __hiloint2double(static_cast<int>(h[1]), static_cast<int>(l[1]));
  const double bq = 4 * e.de / (D * D * D);
  const double aq = Ks / (4 * D * D);
  const double cq = (9 * bq * bq - 16 * aq * aq * D * D) / (32 * aq);
  const double delta = sqrt(fabs(9 * bq * bq - 32 * aq * cq));
  e.ea = (3 * bq + delta) * (3 * bq + delta) * (3 * bq * bq - 16 * aq * cq + bq * delta) /
         (aq * aq * aq) / 2048;
  e.ekra = e.ea - e.de / 2;  // kinetically resolved barrier: Ea(i->j) - Ea(j->i) = dE
  return e;
}

// Whether one of the sites in the masks `vac` lies in the lane's environment (endpoint sites: the
// target counts, as any slot but the vacancy's own).
__device__ __forceinline__ bool VacancyInEvent(const KTables &t, uint64_t v0, uint64_t v1, uint64_t v2, int dir) {
  bool bad = false;
#pragma unroll 1
  for (int s = 0; s < kEnvSlots; ++s) {
    const int i = t.site_of[dir * kEnvSlots + s];
    const uint64_t m = i < 64 ? v0 : i < 128 ? v1 : v2;
    if (i < kPairSites) bad = bad || ((m >> (i & 63)) & 1);
  }
  return bad;
}

// Checks the species just read: codes past the model's set the error flag and read as 0. Returns
// whether the lane's environment holds a vacancy off the jump's origin. Both are rare; together they
// cost one scalar branch.
template <typename Id>
__device__ __forceinline__ bool CheckCodes(const KTables &t, Around<Id> &a, int dir, int32_t *err) {
  const uint64_t past = __ballot(max(max(a.code[0], a.code[1]), a.code[2]) >= t.S);
  const uint64_t v0 = __ballot(a.code[0] == t.x_code), v1 = __ballot(a.code[1] == t.x_code);
  const uint64_t v2 = __ballot(a.code[2] == t.x_code) & kThirdMask;
  if ((past | v0 | v1 | v2) == 0) return false;
  if (past) {
    if (LaneId() == 0) atomicOr(err, 4);
#pragma unroll
    for (int u = 0; u < 3; ++u) a.code[u] = a.code[u] >= t.S ? 0 : a.code[u];
  }
  // a species 0 put in for a corrupt code counts as read
  return VacancyInEvent(t, v0, v1, v2, dir);
}

// Whether the event met a model error: no one-hot type, or an unknown cluster type.
__device__ __forceinline__ bool EventError(const EventValue &e) {
  return !(e.ea == e.ea) || !(e.de == e.de) || !(e.la == e.la);
}

// Signed offset of a packed site.
__device__ __forceinline__ XYZ PackedXYZ(int32_t pk) {
  return {static_cast<int8_t>(pk), static_cast<int8_t>(pk >> 8), static_cast<int8_t>(pk >> 16)};
}
__device__ __forceinline__ XYZ WrapAdd(const XYZ &c, const XYZ &d, int m) {
  return {Wrap(c.X + d.X, m), Wrap(c.Y + d.Y, m), Wrap(c.Z + d.Z, m)};
}

}  // namespace
}  // namespace lmc
