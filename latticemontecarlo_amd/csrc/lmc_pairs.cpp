// Host construction of the pair tables (lmc_pairs.h).
#include "lmc_pairs.h"

#include <algorithm>
#include <map>
#include <memory>
#include <mutex>
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
  uint8_t at[9][9][9];  // site at an offset, every component of which is within four
  std::fill_n(&at[0][0][0], 9 * 9 * 9, static_cast<uint8_t>(kPairSites));
  auto site_at = [&](const I3 &o) -> uint8_t & { return at[o.x + 4][o.y + 4][o.z + 4]; };
  auto add = [&](const I3 &o) {
    if (Key(o) == Key(I3{0, 0, 0}) || site_at(o) != kPairSites) return;
    site_at(o) = static_cast<uint8_t>(sites.size());
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
      const int i = site_at(jt.off[dir[d]][s]);
      g.site_of[d][s] = static_cast<uint8_t>(i);
      if (s != jt.v_slot && s != jt.n_slot) g.slot[d][i] = static_cast<uint8_t>(s);
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
  // cluster kind, id and role of every slot pair's members
  constexpr int kPairs = kEnvSlots * kEnvSlots;
  std::vector<std::pair<int, uint32_t>> all;
  std::vector<int> start(kPairs + 1, 0);
  all.reserve(4 * terms.size());
  auto put = [&](int s1, int s2, const Term &e, int role) {
    const int s = s1 * kEnvSlots + s2;
    ++start[s + 1];
    all.emplace_back(s, static_cast<uint32_t>(e.kind << 24 | e.id << 2 | role));
  };
  for (const Term &e : terms) {
    if (e.s1 < 0) {
      put(e.s0, e.s0, e, 2);
      continue;
    }
    const int second = e.symmetric ? 0 : 1;
    put(e.s0, e.s0, e, 0);
    put(e.s1, e.s1, e, second);
    put(e.s0, e.s1, e, 0);
    put(e.s1, e.s0, e, second);
  }
  for (int s = 0; s < kPairs; ++s) start[s + 1] += start[s];
  std::vector<uint32_t> members(all.size());
  std::vector<int> end(start.begin(), start.end() - 1);
  for (const auto &[s, m] : all) members[end[s]++] = m;
  ClassTable t;
  t.of.assign(kEnvSlots * kEnvSlots, 0);
  std::map<std::vector<uint32_t>, int> known;  // the members of a class, each followed by its count
  std::vector<uint32_t> key;
  for (int s = 0; s < kPairs; ++s) {
    if (start[s] == end[s]) continue;
    std::sort(members.begin() + start[s], members.begin() + end[s]);
    const bool single = s / kEnvSlots == s % kEnvSlots;
    key.assign(1, single);
    for (int i = start[s]; i < end[s]; ++i) {
      if (key.size() > 1 && key[key.size() - 2] == members[i]) ++key.back();
      else key.insert(key.end(), {members[i], 1u});
    }
    auto at = known.find(key);
    if (at == known.end()) {
      at = known.emplace(key, static_cast<int>(t.classes.size())).first;
      PairClass c{single, {}};
      for (size_t k = 1; k < key.size(); k += 2)
        c.members.push_back({static_cast<int>(key[k] >> 24), static_cast<int>(key[k] >> 2) & 0x3FFFFF,
                             static_cast<int>(key[k] & 3), static_cast<int>(key[k + 1])});
      t.classes.push_back(std::move(c));
    }
    t.of[s] = at->second + 1;
  }
  return t;
}

template <int kSum>
const ClassTable &ClassesOf() {
  static const ClassTable t = BuildClasses(kSum);
  return t;
}
const ClassTable &Classes(int sum) {
  return sum == 0 ? ClassesOf<0>() : sum == 1 ? ClassesOf<1>() : ClassesOf<2>();
}

PairTables BuildPairTables(int ne, bool quartic) {
  const int q = std::max(1, ne - 1), block = q * q + 1;
  PairTables t;
  std::vector<uint16_t> offs[3];
  int *rows[3] = {&t.de_row, &t.la_row, &t.lb_row};
  for (int x = 0; x < (quartic ? 3 : 2); ++x) {
    const ClassTable &ct = Classes(x);
    *rows[x] = static_cast<int>(ct.classes.size() + 1) * block;
    if (*rows[x] * 8 > 65535) throw std::invalid_argument("pair classes exceed the packed tables");
    offs[x].assign((kNoSlot + 1) * kClsRow, 0);
    for (int s = 0; s < kEnvSlots * kEnvSlots; ++s)
      offs[x][s / kEnvSlots * kClsRow + s % kEnvSlots] = static_cast<uint16_t>(ct.of[s] * block * 8);
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

}  // namespace

const PairTables &GetPairTables(int ne, bool quartic) {
  static std::mutex mu;
  static std::unique_ptr<const PairTables> known[kMaxSpecies + 1][2];
  std::lock_guard<std::mutex> lock(mu);
  auto &t = known[std::clamp(ne, 0, kMaxSpecies)][quartic];
  if (!t) t = std::make_unique<const PairTables>(BuildPairTables(ne, quartic));
  return *t;
}

std::vector<double> BuildPairValues(const Model &m, int ref) {
  const JumpTables &jt = GetJumpTables();
  const int S = m.S, ne = m.ne, q = std::max(1, ne - 1), block = q * q + 1;
  const bool quartic = m.kind == kQuartic;
  const PairTables &t = GetPairTables(ne, quartic);
  const PairBlock at = PairBlockOf(ne, t.de_row, t.la_row, t.lb_row);
  std::vector<double> out(at.size, 0.0);
  std::vector<int> code;  // element rank -> species code
  for (int c = 0; c < S; ++c)
    if (c != m.x_code) code.push_back(c);
  // weight of a cluster of a label or orbit over element ranks: [label][M, or ne: the vacancy][a][b] and
  // [orbit][M][a][b]
  const size_t cells = static_cast<size_t>(ne) * ne, state_row = cells * (ne + 1), row = cells * ne;
  std::vector<double> state(8 * state_row), mmm(jt.mmm.orbit_kind.size() * row), mm2(quartic ? jt.mm2.orbit_kind.size() * row : 0);
  size_t i = 0;
  for (int label = 0; label < 8; ++label)
    for (int M = 0; M <= ne; ++M) {
      const int x = M < ne ? code[M] : m.x_code;
      for (int a = 0; a < ne; ++a)
        for (int b = 0; b < ne; ++b)
          state[i++] = label == 0  ? m.w[x]
                       : label < 4 ? m.w[S + (label - 1) * S * S + x * S + code[a]]
                                   : m.w[S + 3 * S * S + (label - 4) * S * S * S + (x * S + code[a]) * S + code[b]];
    }
  std::vector<int> type(3 * cells);  // one-hot type by orbit kind and ranks
  for (int kind = 0; kind < 3; ++kind)
    for (int a = 0; a < ne; ++a)
      for (int b = 0; b < ne; ++b) type[kind * cells + a * ne + b] = m.type_tab[(kind * S + code[a]) * S + (kind == 0 ? code[0] : code[b])];
  auto orbits = [&](std::vector<double> &v, const OrbitTable &ot, const std::vector<double> &bw, int F, const std::vector<int> &base) {
    for (size_t id = 0, at = 0; id < ot.orbit_kind.size(); ++id)
      for (int M = 0; M < ne; ++M) {
        const double *w = bw.data() + static_cast<size_t>(code[M]) * F + base[id];
        const int *ty = type.data() + ot.orbit_kind[id] * cells;
        for (size_t k = 0; k < cells; ++k) v[at++] = w[ty[k]];
      }
  };
  orbits(mmm, jt.mmm, m.b_mmm, m.F_mmm, m.base_mmm);
  if (quartic) orbits(mm2, jt.mm2, m.b_mm2, m.F_mm2, m.base_mm2);
  // the weights that a class adds, for one migrating rank; sums in 64-bit mantissas
  struct Weights {
    const double *v;
    long double count;
    int da, db;  // strides of the first site's rank and the second's
  };
  std::vector<Weights> terms;
  const int rows[3] = {t.de_row, t.la_row, t.lb_row}, part[3] = {0, at.la, at.lb};
  for (int x = 0; x < (quartic ? 3 : 2); ++x) {
    const ClassTable &ct = Classes(x);
    for (size_t c = 0; c < ct.classes.size(); ++c)
      for (int M = 0; M < ne; ++M) {
        const PairClass &pc = ct.classes[c];
        terms.clear();
        for (const Member &e : pc.members) {
          const int da = e.role == 1 ? 1 : ne, db = e.role == 1 ? ne : 1;
          if (e.kind <= kNeighbourState) {  // the endpoint's change from a vacancy to M, or back
            const double *v = state.data() + e.id * state_row;
            const long double count = e.kind == kVacancyState ? e.count : -e.count;
            terms.push_back({v + M * cells, count, da, db});
            terms.push_back({v + ne * cells, -count, da, db});
          } else {
            terms.push_back({(e.kind == kMmm ? mmm : mm2).data() + e.id * row + M * cells, static_cast<long double>(e.count), da, db});
          }
        }
        double *val = out.data() + part[x] + static_cast<size_t>(M) * rows[x] + (c + 1) * block;
        for (int k = 0, a = 0; a < ne; ++a) {  // with one element there is none but the reference: zeros
          if (a == ref) continue;
          if (pc.single) {  // its pairs are with reference sites; a singlet's weight ignores the second rank
            long double f1 = 0;
            for (const Weights &w : terms) {
              const double *v = w.v + ref * w.db;
              f1 += w.count * (static_cast<long double>(v[a * w.da]) - v[ref * w.da]);
            }
            val[k * q + k] = static_cast<double>(f1);
          } else {
            for (int l = 0, b = 0; b < ne; ++b) {
              if (b == ref) continue;
              long double f2 = 0;
              for (const Weights &w : terms) {
                const double *va = w.v + a * w.da, *vr = w.v + ref * w.da;
                f2 += w.count * ((static_cast<long double>(va[b * w.db]) - va[ref * w.db]) - (static_cast<long double>(vr[b * w.db]) - vr[ref * w.db]));
              }
              val[k * q + l++] = static_cast<double>(f2);
            }
          }
          ++k;
        }
      }
  }
  // all-reference sums: every cluster of a label or orbit has the same weight
  const size_t same = static_cast<size_t>(ref) * ne + ref;
  int of_label[8] = {};
  for (const auto &c : jt.state_v_only) ++of_label[c.label];
  for (const auto &c : jt.state_n_only) --of_label[c.label];
  for (int M = 0; M < ne; ++M) {
    long double de = 0, la = 0, lb = 0;
    for (int label = 0; label < 8; ++label)
      de += of_label[label] * (static_cast<long double>(state[label * state_row + M * cells + same]) - state[label * state_row + ne * cells + same]);
    for (size_t o = 0; o < jt.mmm.orbit_size.size(); ++o) la += jt.mmm.orbit_size[o] * static_cast<long double>(mmm[o * row + M * cells + same]);
    if (quartic)
      for (size_t o = 0; o < jt.mm2.orbit_size.size(); ++o) lb += 2 * jt.mm2.orbit_size[o] * static_cast<long double>(mm2[o * row + M * cells + same]);
    double *o = out.data() + at.base + 3 * M;
    o[0] = static_cast<double>(de);
    o[1] = static_cast<double>(la);
    o[2] = static_cast<double>(lb);
  }
  return out;
}

}  // namespace lmc
