// Replica state of the persistent KMC kernels and what they do with it besides evaluating jumps:
// temperature schedule, log records, loading and storing.
#pragma once
#include <hip/hip_runtime.h>

#include "lmc_dev_common.h"
#include "lmc_device.h"

namespace lmc {
namespace {

// Replica state of the persistent KMC kernel (in LDS, or uniform over a wave in registers).
struct ReplicaLds {
  uint64_t steps, max_steps, seed;
  double time, energy, abse, T, beta, cv, cs, smass;
  double com[3];
  int64_t vac, disp[3];
  uint32_t rid;
  int flags, esc, solvent, done;
  int vx, vy, vz, m2;  // vacancy coordinates (a/2 units) and the box edge 2n, advanced per jump
};

// Vacancy coordinates of the replica state from its site id (once per launch).
__device__ __forceinline__ void SetVacancyXYZ(ReplicaLds &Q, int n) {
  const XYZ c = ToXYZ(Q.vac, n);
  Q.vx = c.X;
  Q.vy = c.Y;
  Q.vz = c.Z;
  Q.m2 = 2 * n;
}
__device__ __forceinline__ XYZ VacancyXYZ(const ReplicaLds &Q) { return {Q.vx, Q.vy, Q.vz}; }

// TimeTemperatureInterpolator::GetTemperature (TimeTemperatureInterpolator.cpp:44-65)
__device__ double ScheduleTemperature(const double *tt, const double *tv, int n, double time) {
  int i = 0;
  while (i < n && tt[i] < time) ++i;
  if (i == n) return tv[n - 1];
  if (i == 0 && time <= tt[0]) return tv[0];
  return tv[i - 1] + ((time - tt[i - 1]) / (tt[i] - tt[i - 1])) * (tv[i] - tv[i - 1]);
}

// The dump cadence of KineticMcFirstAbstract::Dump (KineticMcAbstract.cpp:83-98): every
// log_every steps past 10 log_every; below that every 10^(floor(log10(steps + 1)) - 1) steps
// (every step below 99), at most log_every.
__device__ bool LogDue(uint64_t steps, uint64_t log_every) {
  uint64_t every = log_every;
  if (steps <= 10 * log_every) {
    uint64_t p = 1;
    for (uint64_t t = steps + 1; t >= 100; t /= 10) p *= 10;
    every = p < log_every ? p : log_every;
  }
  return steps % every == 0;
}

// The energies of a log record: before the step's jump, and the jump's change.
__device__ __forceinline__ void LogEnergy(KmcLogRecord &L, double energy, double de) {
  L.energy = energy;
  L.de = de;
}

// The kmc_log.txt record of the step about to jump the vacancy to `jump` (one lane); energies: with its
// energies.
__device__ void LogStep(const KmcDev &k, const ReplicaLds &Q, int r, int64_t jump, double ea,
                        double de, bool energies = true) {
  const uint64_t i = k.log_n[r];
  k.log_n[r] = i + 1;  // counts past the capacity too, so the host can report the loss
  if (i >= k.log_cap) return;
  KmcLogRecord &L = k.log[static_cast<uint64_t>(r) * k.log_cap + i];
  L.steps = Q.steps;
  L.time = Q.time;
  L.temperature = Q.T;
  L.ea = ea;
  if (energies) LogEnergy(L, Q.energy, de);
  const int64_t o = k.off[r];
  const int32_t *sv = nullptr;
  L.atom = -1;
  if (k.atom) {
    L.atom = k.atom[o + jump];
    sv = k.shift + 3 * (o + k.atom[o + Q.vac]);
  }
  // Config::GetUnwrappedCartesianPositionOfLattice (Config.cpp:280-291) on the cubic box
  const double m = Q.m2, edge = k.log_edge[r];
  L.vac[0] = (Q.vx / m + (sv ? sv[0] : 0)) * edge;
  L.vac[1] = (Q.vy / m + (sv ? sv[1] : 0)) * edge;
  L.vac[2] = (Q.vz / m + (sv ? sv[2] : 0)) * edge;
  L.com[0] = Q.com[0];
  L.com[1] = Q.com[1];
  L.com[2] = Q.com[2];
}

// Replica r's state (one thread, or every lane of a wave for a copy in registers).
__device__ void LoadReplica(const KmcDev &k, int r, int n, ReplicaLds &Q) {
  Q.steps = k.steps[r];
  Q.max_steps = k.max_steps[r];
  Q.seed = k.seed[r];
  Q.rid = k.rid[r];
  Q.time = k.time[r];
  Q.energy = k.energy[r];
  Q.abse = k.abs_energy[r];
  Q.T = k.temp[r];
  Q.cv = k.cv[r];
  Q.cs = k.cs[r];
  Q.smass = k.solute_mass[r];
  Q.vac = k.vac[r];
  Q.flags = k.flags[r];
  Q.esc = k.escaped[r];
  Q.solvent = k.solvent[r];
  for (int a = 0; a < 3; ++a) {
    Q.disp[a] = k.disp[3 * r + a];
    Q.com[a] = k.com[3 * r + a];
  }
  Q.done = (Q.steps > Q.max_steps || Q.esc || !ValidSite(n, Q.vac)) ? 1 : 0;
  Q.beta = 1.0 / kBoltzmann / Q.T;
  SetVacancyXYZ(Q, n);
}

// Replica r's state back to HBM (one thread); `moved`: its displacement in this launch. Without
// kFull the temperature, the escape flag and the solute displacement have not changed. energies:
// with its energies.
__device__ __forceinline__ void StoreEnergy(const KmcDev &k, int r, const ReplicaLds &Q) {
  k.energy[r] = Q.energy;
  k.abs_energy[r] = Q.abse;
}
template <bool kFull>
__device__ void StoreReplica(const KmcDev &k, int r, const ReplicaLds &Q, const XYZ &moved, bool energies = true) {
  k.steps[r] = Q.steps;
  k.time[r] = Q.time;
  if (energies) StoreEnergy(k, r, Q);
  k.vac[r] = Q.vac;
  k.disp[3 * r] += moved.X;
  k.disp[3 * r + 1] += moved.Y;
  k.disp[3 * r + 2] += moved.Z;
  if constexpr (kFull) {
    k.temp[r] = Q.T;
    k.escaped[r] = Q.esc;
    for (int a = 0; a < 3; ++a) k.com[3 * r + a] = Q.com[a];
  }
}

}  // namespace
}  // namespace lmc
