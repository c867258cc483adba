// Host construction of the pair tables (lmc_pairs.h).
#include "lmc_pairs.h"

#include <algorithm>
#include <stdexcept>
#include <tuple>

namespace lmc {

namespace {

std::tuple<int, int, int> Key(const I3 &o) { return {o.x, o.y, o.z}; }

PairGeometry BuildPairGeometry() {
  const JumpTables &jt = GetJumpTables();
  PairGeometry g;
  std::array<int, 12> dir{};  // direction order -> kNN1 index
  for (int k = 0; k < 12; ++k) dir[k] = k;
  std::sort(dir.begin(), dir.end(), [](int a, int b) { return Key(kNN1[a]) < Key(kNN1[b]); });
  std::vector<I3> sites;
  auto add = [&](const I3 &o) {
    if (Key(o) == Key(I3{0, 0, 0})) return;
    for (const I3 &s : sites)
      if (Key(s) == Key(o)) return;
    sites.push_back(o);
  };
  for (int k : dir) add(kNN1[k]);
  for (const I3 &o : kNN2) add(o);
  for (const I3 &o : kNN3) add(o);
  for (int k : dir)
    for (const I3 &o : jt.off[k]) add(o);
  if (sites.size() != kPairSites) throw std::logic_error("jump environments do not cover 134 sites");
  std::copy(sites.begin(), sites.end(), g.site.begin());
  for (int d = 0; d < 12; ++d) {
    g.slot[d].fill(kNoSlot);
    for (int s = 0; s < kEnvSlots; ++s) {
      const I3 &o = jt.off[dir[d]][s];
      g.site_of[d][s] = kPairSites;
      for (int i = 0; i < kPairSites; ++i)
        if (Key(g.site[i]) == Key(o)) {
          g.site_of[d][s] = static_cast<uint8_t>(i);
          if (s != jt.v_slot && s != jt.n_slot) g.slot[d][i] = static_cast<uint8_t>(s);
        }
    }
  }
  for (int d = 0; d < 12; ++d)  // the direction back is 11 - d
    for (int s = 0; s < kEnvSlots; ++s) {
      const I3 &o = jt.off[dir[11 - d]][s];
      g.back[d][s] = I3{g.site[d].x + o.x, g.site[d].y + o.y, g.site[d].z + o.z};
    }
  for (int d = 0; d < 12; ++d)
    for (int s = 0; s < kEnvSlots; ++s)
      g.site3[s][d / 3] |= static_cast<uint32_t>(g.site_of[d][s]) << (8 * (d % 3));
  for (int f = 0; f < 27; ++f) {
    auto wrapped = [](int v, int face) { return face == 1 && v < 0 ? 2 : face == 2 && v > 0 ? -2 : v; };
    auto key = [&](int d) {
      const I3 &o = g.site[d];
      return Key(I3{wrapped(o.x, f % 3), wrapped(o.y, f / 3 % 3), wrapped(o.z, f / 9)});
    };
    std::array<int, 12> ev{};
    for (int k = 0; k < 12; ++k) ev[k] = k;
    std::sort(ev.begin(), ev.end(), [&](int a, int b) { return key(a) < key(b); });
    for (int k = 0; k < 16; ++k) g.order[f][k] = static_cast<uint8_t>(ev[std::min(k, 11)]);
  }
  return g;
}

}  // namespace

const PairGeometry &GetPairGeometry() {
  static const PairGeometry g = BuildPairGeometry();
  return g;
}

namespace {

// What the clusters of a slot pair (or of one slot, with its pairs to reference sites) look like: a
// cluster kind, its label or orbit, which of its sites is the pair's first, and how often.
enum { kVacancyState, kNeighbourState, kMmm, kMm2, kMm2Backward };
struct Member {
  int kind, id, role, count;
  bool operator<(const Member &o) const {
    return std::tie(kind, id, role) < std::tie(o.kind, o.id, o.role);
  }
  bool operator==(const Member &o) const {
    return kind == o.kind && id == o.id && role == o.role && count == o.count;
  }
};
struct PairClass {
  bool single;
  std::vector<Member> members;
};
// The classes of one sum (dE, MMM logit, MM2 logit) and the class of every ordered slot pair (0: none,
// else index + 1). The same for every model.
struct ClassTable {
  std::vector<PairClass> classes;
  std::vector<int> of;  // [60][60]
};

ClassTable BuildClasses(int sum) {
  const JumpTables &jt = GetJumpTables();
  struct Term {
    int s0, s1, kind, id;  // sites in the cluster's own order (second -1: one site)
    bool symmetric;
  };
  std::vector<Term> terms;
  auto state = [&](const std::vector<StateCluster> &cl, int endpoint, int kind) {
    for (const auto &c : cl) {
      int o[2] = {-1, -1}, n = 0;
      for (int i = 0; i < c.size; ++i)
        if (c.slots[i] != endpoint) o[n++] = c.slots[i];
      if (n) terms.push_back({o[0], o[1], kind, c.label, true});
    }
  };
  auto orbits = [&](const OrbitTable &ot, int kind, bool mirror) {
    auto slot = [&](int s) { return s < 0 ? -1 : mirror ? jt.mirror[s] : s; };
    for (const auto &c : ot.clusters)
      terms.push_back({slot(c.s0), slot(c.s1), kind, c.orbit, ot.orbit_kind[c.orbit] != 1});
  };
  if (sum == 0) {
    state(jt.state_v_only, jt.v_slot, kVacancyState);
    state(jt.state_n_only, jt.n_slot, kNeighbourState);
  } else if (sum == 1) {
    orbits(jt.mmm, kMmm, false);
  } else {
    orbits(jt.mm2, kMm2, false);
    orbits(jt.mm2, kMm2Backward, true);
  }
  std::vector<std::vector<Member>> mem(kEnvSlots * kEnvSlots);
  auto put = [&](int s1, int s2, const Term &e, int role) {
    mem[s1 * kEnvSlots + s2].push_back({e.kind, e.id, e.symmetric ? 0 : role, 1});
  };
  for (const Term &e : terms) {
    if (e.s1 < 0) {
      mem[e.s0 * kEnvSlots + e.s0].push_back({e.kind, e.id, 2, 1});
      continue;
    }
    put(e.s0, e.s0, e, 0);
    put(e.s1, e.s1, e, 1);
    put(e.s0, e.s1, e, 0);
    put(e.s1, e.s0, e, 1);
  }
  ClassTable t;
  t.of.assign(kEnvSlots * kEnvSlots, 0);
  for (int s = 0; s < kEnvSlots * kEnvSlots; ++s) {
    if (mem[s].empty()) continue;
    std::sort(mem[s].begin(), mem[s].end());
    std::vector<Member> merged;
    for (const Member &m : mem[s]) {
      if (!merged.empty() && !(merged.back() < m)) ++merged.back().count;
      else merged.push_back(m);
    }
    const bool single = s / kEnvSlots == s % kEnvSlots;
    int at = -1;
    for (size_t i = 0; i < t.classes.size() && at < 0; ++i)
      if (t.classes[i].single == single && t.classes[i].members == merged) at = static_cast<int>(i);
    if (at < 0) {
      at = static_cast<int>(t.classes.size());
      t.classes.push_back({single, merged});
    }
    t.of[s] = at + 1;
  }
  return t;
}

const ClassTable &Classes(int sum) {
  static const ClassTable t[3] = {BuildClasses(0), BuildClasses(1), BuildClasses(2)};
  return t[sum];
}

}  // namespace

PairTables BuildPairTables(const Model &m) {
  const JumpTables &jt = GetJumpTables();
  const int S = m.S, ne = m.ne, q = std::max(1, ne - 1), block = q * q + 1;
  const bool quartic = m.kind == kQuartic;
  PairTables t;
  if (m.kind != kE0 && m.kind != kQuartic) return t;
  std::vector<int> code;  // element rank -> species code
  for (int c = 0; c < S; ++c)
    if (c != m.x_code) code.push_back(c);
  // value of a cluster of each kind and label or orbit: [id][M][a][b] over ranks
  const size_t row = static_cast<size_t>(ne) * ne * ne;
  std::vector<long double> values[5];
  auto each = [&](std::vector<long double> &v, int ids, auto &&f) {
    v.resize(ids * row);
    size_t i = 0;
    for (int id = 0; id < ids; ++id)
      for (int M = 0; M < ne; ++M)
        for (int a = 0; a < ne; ++a)
          for (int b = 0; b < ne; ++b) v[i++] = f(id, M, a, b);
  };
  auto w = [&](int label, int x, int a, int b) -> long double {
    if (label == 0) return m.w[x];
    if (label < 4) return m.w[S + (label - 1) * S * S + x * S + code[a]];
    return m.w[S + 3 * S * S + (label - 4) * S * S * S + (x * S + code[a]) * S + code[b]];
  };
  each(values[kVacancyState], 8, [&](int id, int M, int a, int b) {
    return w(id, code[M], a, b) - w(id, m.x_code, a, b);
  });
  values[kNeighbourState] = values[kVacancyState];
  for (long double &x : values[kNeighbourState]) x = -x;
  auto orbit = [&](const OrbitTable &ot, const std::vector<double> &bw, int F, const std::vector<int> &base) {
    return [&, F](int id, int M, int a, int b) -> long double {
      const int kind = ot.orbit_kind[id];
      const int ty = m.type_tab[(kind * S + code[a]) * S + (kind == 0 ? code[0] : code[b])];
      return bw[static_cast<size_t>(code[M]) * F + base[id] + ty];
    };
  };
  each(values[kMmm], static_cast<int>(jt.mmm.orbit_kind.size()), orbit(jt.mmm, m.b_mmm, m.F_mmm, m.base_mmm));
  if (quartic) {
    each(values[kMm2], static_cast<int>(jt.mm2.orbit_kind.size()), orbit(jt.mm2, m.b_mm2, m.F_mm2, m.base_mm2));
    values[kMm2Backward] = values[kMm2];
  }
  std::vector<uint16_t> offs[3];
  std::vector<double> *out[3] = {&t.de, &t.la, &t.lb};
  int *rows[3] = {&t.de_row, &t.la_row, &t.lb_row};
  for (int x = 0; x < (quartic ? 3 : 2); ++x) {
    const ClassTable &ct = Classes(x);
    *rows[x] = static_cast<int>(ct.classes.size() + 1) * block;
    if (*rows[x] * 8 > 65535) throw std::invalid_argument("pair classes exceed the packed tables");
    offs[x].assign((kNoSlot + 1) * kClsRow, 0);
    for (int s = 0; s < kEnvSlots * kEnvSlots; ++s)
      offs[x][s / kEnvSlots * kClsRow + s % kEnvSlots] = static_cast<uint16_t>(ct.of[s] * block * 8);
    std::vector<double> &tab = *out[x];
    const size_t stride = PairStride(ne, *rows[x]);
    tab.assign(ne * stride, 0.0);
    for (int ref = 0; ref < ne; ++ref) {
      std::vector<int> rank;  // non-reference ranks
      for (int r = 0; r < ne; ++r)
        if (r != ref) rank.push_back(r);
      const int nr = static_cast<int>(rank.size());  // 0 with one element: every term is zero
      for (int M = 0; M < ne; ++M)
        for (size_t c = 0; c < ct.classes.size(); ++c) {
          const PairClass &pc = ct.classes[c];
          double *val = tab.data() + ref * stride + static_cast<size_t>(M) * *rows[x] + (c + 1) * block;
          for (int i = 0; i < nr; ++i)
            for (int j = 0; j < nr; ++j) {
              if (pc.single && i != j) continue;
              const int a = rank[i], b = rank[j];
              long double sum = 0;
              for (const Member &e : pc.members) {
                const long double *v = values[e.kind].data() + e.id * row + static_cast<size_t>(M) * ne * ne;
                auto at = [&](int p, int r) { return v[p * ne + r]; };
                if (pc.single)  // role 2: a singlet, whose value ignores the second rank
                  sum += e.count * ((e.role == 1 ? at(ref, a) : at(a, ref)) - at(ref, ref));
                else
                  sum += e.count * ((e.role ? at(b, a) - at(b, ref) - at(ref, a)
                                            : at(a, b) - at(a, ref) - at(ref, b)) + at(ref, ref));
              }
              val[i * q + j] = static_cast<double>(sum);
            }
        }
    }
  }
  t.cls.resize(offs[0].size());
  for (size_t i = 0; i < t.cls.size(); ++i)
    t.cls[i] = static_cast<uint32_t>(offs[0][i]) | (static_cast<uint32_t>(offs[1][i]) << 16);
  t.clsb = quartic ? offs[2] : std::vector<uint16_t>(8, 0);
  for (int s1 = 0; s1 < kEnvSlots; ++s1)
    for (int s2 = s1; s2 < kEnvSlots; ++s2) {
      const size_t i = static_cast<size_t>(s1) * kClsRow + s2;
      if (!t.cls[i] && !(quartic && t.clsb[i])) continue;
      t.dense.push_back(t.cls[i]);
      t.dense.push_back(static_cast<uint32_t>(16 * s1 | (16 * s2) << 16));
      t.denseb.push_back(quartic ? t.clsb[i] : 0);
    }
  if (t.denseb.size() > kMaxDense) throw std::logic_error("more slot pairs than the list holds");
  t.dense.resize(2 * kMaxDense, 0);  // a blank's class is block 0
  t.denseb.resize(kMaxDense, 0);
  const PairGeometry &g = GetPairGeometry();
  for (int d = 0; d < 12; ++d)
    for (int i = 0; i < kOneRow; ++i) {
      const size_t at = static_cast<size_t>(g.slot[d][std::min(i, kPairSiteRow - 1)]) * (kClsRow + 1);
      t.one.push_back(t.cls[at]);
      t.oneb.push_back(quartic ? t.clsb[at] : 0);
    }
  return t;
}

}  // namespace lmc
