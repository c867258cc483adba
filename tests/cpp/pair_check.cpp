// Checks the quadratic form of the jump sums against the sums over every cluster, on random
// environments: pair_check MODEL.json KIND ELEMENT... prints the largest relative difference.
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include <stdexcept>
#include <string>
#include <vector>

#include "lmc_pairs.h"

namespace lmc {
Model::~Model() {}  // no device tables here
}  // namespace lmc
using namespace lmc;

namespace {

struct Sums {
  long double v[3] = {0, 0, 0}, size[3] = {0, 0, 0};
  void Add(int i, long double x) {
    v[i] += x;
    size[i] += std::fabs(x);
  }
};

// Every cluster of the environment env[60] (element ranks; env[n_slot] the migrating rank).
Sums Clusters(const Model &m, const JumpTables &jt, const std::vector<int> &code, const int *env) {
  Sums s;
  const int S = m.S, M = code[env[jt.n_slot]];
  auto state = [&](const std::vector<StateCluster> &cl, int endpoint, double sign) {
    for (const auto &c : cl) {
      int o[2] = {0, 0}, n = 0;
      for (int i = 0; i < c.size; ++i)
        if (c.slots[i] != endpoint) o[n++] = code[env[c.slots[i]]];
      auto w = [&](int x) {
        if (c.label == 0) return m.w[x];
        if (c.label < 4) return m.w[S + (c.label - 1) * S * S + x * S + o[0]];
        return m.w[S + 3 * S * S + (c.label - 4) * S * S * S + (x * S + o[0]) * S + o[1]];
      };
      s.Add(0, sign * (static_cast<long double>(w(M)) - w(m.x_code)));
    }
  };
  state(jt.state_v_only, jt.v_slot, 1.0);
  state(jt.state_n_only, jt.n_slot, -1.0);
  auto orbits = [&](const OrbitTable &ot, const std::vector<double> &b, int F, const std::vector<int> &base,
                    int out, bool mirror) {
    for (const auto &c : ot.clusters) {
      const int kind = ot.orbit_kind[c.orbit];
      auto at = [&](int slot) { return code[env[mirror ? jt.mirror[slot] : slot]]; };
      const int ty = m.type_tab[(kind * S + at(c.s0)) * S + (kind == 0 ? code[0] : at(c.s1))];
      s.Add(out, b[static_cast<size_t>(M) * F + base[c.orbit] + ty]);
    }
  };
  orbits(jt.mmm, m.b_mmm, m.F_mmm, m.base_mmm, 1, false);
  if (m.kind == kQuartic) {
    orbits(jt.mm2, m.b_mm2, m.F_mm2, m.base_mm2, 2, false);
    orbits(jt.mm2, m.b_mm2, m.F_mm2, m.base_mm2, 2, true);
  }
  return s;
}

}  // namespace

int main(int argc, char **argv) {
  const std::vector<std::string> els(argv + 3, argv + argc);
  Model *m = LoadModel(argv[1], els, std::atoi(argv[2]));
  const JumpTables &jt = GetJumpTables();
  const PairGeometry &g = GetPairGeometry();
  const PairTables &t = GetPairTables(m->ne, m->kind == kQuartic);
  const int ne = m->ne, q = std::max(1, ne - 1);
  std::vector<int> code;
  for (int c = 0; c < m->S; ++c)
    if (c != m->x_code) code.push_back(c);
  // the parts of a block can be copied 16 bytes at a time and do not overlap
  const PairBlock bl = PairBlockOf(ne, t.de_row, t.la_row, t.lb_row);
  if (bl.la % 2 || bl.lb % 2 || bl.base % 2 || bl.size % 2 || bl.la < ne * t.de_row || bl.lb < bl.la + ne * t.la_row ||
      bl.base < bl.lb + ne * t.lb_row || bl.size < bl.base + 3 * ne)
    return std::puts("parts of a block"), 1;
  // geometry: slots and sites name the same offsets, and pairs with a term are near
  for (int d = 0; d < 12; ++d)
    for (int i = 0; i < kPairSites; ++i) {
      const int s = g.slot[d][i];
      if (s != kNoSlot && g.site_of[d][s] != i) return std::puts("slot and site_of differ"), 1;
      for (int j = 0; j < kPairSites; ++j) {
        const int u = g.slot[d][j];
        const size_t at = static_cast<size_t>(s) * kClsRow + u;
        if (s == u || !(t.cls[at] | (t.clsb.size() > 8 ? t.clsb[at] : 0))) continue;
        const I3 &a = g.site[i], &b = g.site[j];
        const int r2 = (a.x - b.x) * (a.x - b.x) + (a.y - b.y) * (a.y - b.y) + (a.z - b.z) * (a.z - b.z);
        if (r2 > 6) return std::puts("a far pair has a term"), 1;
      }
    }
  // the event order is that of the neighbour ids, for vacancies at and away from every face
  for (int n : {4, 5, 7})
    for (int64_t v = 0; v < 4ll * n * n * n; ++v) {
      const I3 c = SiteXYZ(n, v);
      auto face = [&](int x) { return x == 0 ? 1 : x == 2 * n - 1 ? 2 : 0; };
      const auto &o = g.order[face(c.x) + 3 * face(c.y) + 9 * face(c.z)];
      for (int e = 0; e < 11; ++e)
        if (SiteAdd(n, v, g.site[o[e]]) >= SiteAdd(n, v, g.site[o[e + 1]])) return std::puts("event order"), 1;
      for (int e = 11; e < 16; ++e)
        if (o[e] != o[11]) return std::puts("event order past the last"), 1;
    }
  for (int s = 0; s < kEnvSlots; ++s)
    for (int d = 0; d < 12; ++d)
      if (((g.site3[s][d / 3] >> (8 * (d % 3))) & 255u) != g.site_of[d][s]) return std::puts("site3"), 1;
  // one direction is the reverse of the direction 11 - d
  for (int d = 0; d < 12; ++d)
    if (g.site[d].x != -g.site[11 - d].x || g.site[d].y != -g.site[11 - d].y || g.site[d].z != -g.site[11 - d].z)
      return std::puts("directions are not in opposite order"), 1;
  std::mt19937 rng(7);
  double worst = 0;
  for (int ref = 0; ref < ne; ++ref) {
    const std::vector<double> v = BuildPairValues(*m, ref);
    if (v.size() != static_cast<size_t>(bl.size)) return std::puts("size of the values"), 1;
    for (int trial = 0; trial < 200; ++trial) {
      int env[kEnvSlots], none[kEnvSlots];
      const double fill = trial % 4 == 3 ? 1.0 : 0.15 * (1 + trial % 4);
      for (int s = 0; s < kEnvSlots; ++s) {
        env[s] = std::uniform_real_distribution<>(0, 1)(rng) < fill ? static_cast<int>(rng() % ne) : ref;
        none[s] = ref;
      }
      none[jt.n_slot] = env[jt.n_slot];
      env[jt.v_slot] = none[jt.v_slot] = ref;
      const Sums want = Clusters(*m, jt, code, env), base = Clusters(*m, jt, code, none);
      const int M = env[jt.n_slot];
      double sparse[3], dense[3];
      for (int i = 0; i < 3; ++i) {
        sparse[i] = dense[i] = v[bl.base + 3 * M + i];
        const double size = static_cast<double>(base.size[i]) + 1e-300;
        worst = std::max(worst, std::fabs(sparse[i] - static_cast<double>(base.v[i])) / size);
      }
      auto rank = [&](int s) { return env[s] - (env[s] > ref ? 1 : 0); };
      auto add = [&](double *sum, uint32_t c, uint32_t cb, int a, int b) {
        sum[0] += v[M * t.de_row + (c & 0xFFFF) / 8 + a * q + b];
        sum[1] += v[bl.la + M * t.la_row + (c >> 16) / 8 + a * q + b];
        if (m->kind == kQuartic) sum[2] += v[bl.lb + M * t.lb_row + cb / 8 + a * q + b];
      };
      auto other = [&](int s) { return s != jt.v_slot && s != jt.n_slot && env[s] != ref; };
      for (int a = 0; a < kEnvSlots; ++a)
        for (int b = 0; b <= a; ++b)
          if (other(a) && other(b)) {  // either order of a pair
            const int x = trial & 1 ? a : b, y = trial & 1 ? b : a;
            const size_t at = static_cast<size_t>(x) * kClsRow + y;
            add(sparse, t.cls[at], m->kind == kQuartic ? t.clsb[at] : 0, rank(x), rank(y));
          }
      for (int i = 0; i < kMaxDense; ++i) {
        const int a = (t.dense[2 * i + 1] & 0xFFFF) / 16, b = (t.dense[2 * i + 1] >> 16) / 16;
        const bool on = other(a) && other(b);  // else the zero after the block
        add(dense, t.dense[2 * i], t.denseb[i], on ? rank(a) : q, on ? rank(b) : 0);
      }
      for (int i = 0; i < 3; ++i) {
        const double scale = static_cast<double>(want.size[i]) + 1e-300;
        worst = std::max(worst, std::fabs(sparse[i] - static_cast<double>(want.v[i])) / scale);
        worst = std::max(worst, std::fabs(dense[i] - static_cast<double>(want.v[i])) / scale);
      }
    }
  }
  std::printf("%.3e\n", worst);
  return 0;
}
