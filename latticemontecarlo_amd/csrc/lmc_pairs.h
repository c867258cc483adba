// The jump evaluation as a quadratic form over the non-reference sites of an environment.
//
// Every cluster of a jump's dE (one endpoint and at most two other sites) and of its barrier logits
// (at most two sites) touches at most two of the 58 non-endpoint slots, so each sum is, exactly,
//   base[M] + sum_j f1[M][j][r_j] + sum_{j<k} f2[M][j,k][r_j, r_k]
// over the slots that do not hold the reference species s (usually the solvent), with
//   f1[j][a]    = sum over clusters containing j of value(a, rest s) - value(all s),
//   f2[j,k][a,b] = sum over clusters containing both of v(a,b) - v(a,s) - v(s,b) + v(s,s).
// f2 vanishes unless j and k are within three shells of each other: 556 pairs, which fall into
// few classes of equal values (the orbits of the barrier encodings, the triplet labels of dE).
#pragma once
#include <array>
#include <cstdint>
#include <vector>

#include "lmc_model.h"

namespace lmc {

constexpr int kPairSites = 134;   // sites of the 12 environments, without the vacancy's own
constexpr int kPairSiteRow = 136; // row length of the site tables
constexpr int kNoSlot = 60;       // slot of a site outside an environment, or at an endpoint
constexpr int kOneRow = kPairSiteRow + 1;  // odd, so that a site's 12 entries lie in 12 banks
constexpr int kClsRow = 64;
constexpr int kMaxDense = 640;    // list of the 614 slot pairs with a term, with blanks

// Geometry shared by all models. Directions are in ascending (x, y, z) order of the jump vector,
// which is the order of the neighbour ids away from the box faces.
struct PairGeometry {
  std::array<I3, kPairSites> site{};  // offsets: the 12 first neighbours in direction order, the
                                      // other sites within three shells, the rest
  std::array<std::array<uint8_t, kPairSiteRow>, 12> slot{};   // [direction][site]
  std::array<std::array<uint8_t, kEnvSlots>, 12> site_of{};   // [direction][slot]; vacancy: kPairSites
  // offsets from the vacancy of the slots of the reverse event, from the neighbour in a direction back
  std::array<std::array<I3, kEnvSlots>, 12> back{};
  // sites of a slot for the directions 3 g .. 3 g + 2, a byte each: [slot][g]
  std::array<std::array<uint32_t, 4>, kEnvSlots> site3{};
  // directions by ascending neighbour id for a vacancy inside the box (0), at coordinate 0 (1) or at
  // the top coordinate (2) of each axis: [x + 3 y + 9 z][event]; entries past 11 repeat event 11
  std::array<std::array<uint8_t, 16>, 27> order{};
};
const PairGeometry &GetPairGeometry();

// Class lists of the models with one number of elements. A class is a block of q * q values (q = ne - 1 non-reference ranks) and
// one zero after them, block 0 all zero. cls[s1 * 64 + s2] holds the byte offsets of the blocks of the ordered slot pair
// (s1 == s2: the one-site term, on the block's diagonal) within a row: dE in the low half-word,
// the MMM logit in the high one; clsb the MM2 logit's. A block is indexed by the rank at s1 times q
// plus the rank at s2, ranks numbered without the reference's.
struct PairTables {
  std::vector<uint32_t> cls;       // [61][64]
  std::vector<uint16_t> clsb;      // [61][64], quartic only
  std::vector<uint32_t> one;       // [12][137] cls of a site's slot with itself, by direction
  std::vector<uint16_t> oneb;
  // slot pairs with a term: cls, then 16 s1 | 16 s2 << 16, and clsb; blanks after them
  std::vector<uint32_t> dense;
  std::vector<uint16_t> denseb;
  int de_row = 0, la_row = 0, lb_row = 0;  // rows of the values, in doubles
};
const PairTables &GetPairTables(int ne, bool quartic);  // ne: the model's elements

// The values of one reference species, in doubles: [migrating rank][row] of the dE, MMM and MM2 classes and
// the all-reference sums [migrating rank][dE, MMM, MM2 logit]. Each part starts on 16 bytes, as does the
// next reference's block.
struct PairBlock {
  int la, lb, base, size;  // where the parts start (dE: at 0), and the length of all
};
constexpr PairBlock PairBlockOf(int ne, int de_row, int la_row, int lb_row) {
  const int la = (ne * de_row + 1) & ~1, lb = la + ((ne * la_row + 1) & ~1), base = lb + ((ne * lb_row + 1) & ~1);
  return {la, lb, base, base + ((3 * ne + 1) & ~1)};
}
// The block of reference rank ref. The engine forms a species' block when a batch first has it as its
// solvent: all of a five-element Quartic model's take 1 ms.
std::vector<double> BuildPairValues(const Model &m, int ref);

}  // namespace lmc
