// Plan of the LDS-resident factorization: the levels of the elimination tree
// below the dense tail cut into parts whose factor blocks fit one workgroup's
// LDS, so that every product of the elimination reads its operands there.
#pragma once
#include <cstdint>
#include <vector>

#include "symbolic.hpp"

namespace bpf {

// What a lane group of a round forms (RES_* in the descriptor's kind bits).
// With the slot (k, r) holding L(r, k) and U(k, r), and the slot (k, rhs)
// holding the pivot inverse and y_k, every sum is over words {a, b}:
//   sumU += L(a) U(b),  sumL += L(b) U(a).
enum {
  RES_NONE = 0,
  RES_PIVOT = 1,      // pivot inverse of (L part - sumU), into the L part
  RES_PAIR = 2,       // U part - sumU; (L part - sumL) times the pivot inverse
  RES_RHS = 3,        // U part - sumU
  RES_UPD_PAIR = 4,   // sums for a slot of a later part: sumL and sumU
  RES_UPD_DIAG = 5,   // sumU for a later pivot, into the update's L block
  RES_UPD_RHS = 6     // sumU for a later right-hand side, into its U block
};
// The last part (the top of the tree, then the dense tail) has a workgroup of
// 1024 lanes and a compute unit's LDS to itself; the others take workgroups of
// RES_SMALL_LANES lanes, several to a compute unit.
constexpr int RES_TOP_LANES = 1024, RES_TOP_LDS = 158 * 1024;
constexpr int RES_SMALL_LANES = 256, RES_SMALL_LDS = 32 * 1024 - 64;
constexpr int RES_J = 8;               // words per lane and round, at most
// a wave's flags of a round: words per lane (0, 1, 2, 4 or 8) | log2 lane group
// << 4 | runs | the round's barriers, before its pivots are used and after its
// results
constexpr int RES_RUN = 1 << 7, RES_MID = 1 << 8, RES_END = 1 << 9;
constexpr int RES_PIV = 1 << 10, RES_UPD = 1 << 11;  // all its tasks: pivots; updates
// descriptor: kind << 29 | pivot slot << 13 | slot, or kind << 29 | update
constexpr int RES_KIND_SHIFT = 29, RES_SLOT_BITS = 13;
constexpr int RES_SLOT_MASK = (1 << RES_SLOT_BITS) - 1;
constexpr int RES_KEEP = 1 << 30;      // slot_pos .x: finished by the Jacobian fill
constexpr int RES_FILL = 1 << 29;      // slot_pos and tail .x: fill-in, starts from zero
constexpr int RES_POS = RES_FILL - 1;

struct ResidentPlan {
  bool ok = false;
  int nslots = 0, nupd = 0;            // slots of all parts, updates
  // parts of one stage depend only on those of earlier stages; the last
  // stage is one part, the workgroup that goes on to the dense tail
  std::vector<int> stage;              // first part of each stage, then the count
  // per part two int4: {first slot, end slot, first entry of the wave table,
  // the first after level 0 (when the fill finished it)}, {end entry, first
  // word, first descriptor, waves of its workgroup}; words and descriptors of
  // a part end where the next starts (one more entry closes the list)
  std::vector<int> part;
  // per slot {position of the L part, of the U part} in the factor storage,
  // -1 where there is none; the pivot's slot (k, rhs): {diagonal, rhs of k}
  std::vector<int> slot_pos;
  // per slot its updates from earlier parts
  std::vector<int> upd_ptr, upd;
  // per part, round and wave {first word, first descriptor, flags, 0}; word j
  // of lane l is word[first + (words per lane) l + j]
  std::vector<int> wave;
  std::vector<uint32_t> word;          // slots a | b << 16 (0: the zero slot)
  std::vector<uint32_t> desc;          // per lane; a group's first lane has its task
  // dense tail: per entry pair (r <= c) {L position, U position, r, c} and
  // its updates (the diagonal: the L block)
  std::vector<int> tail, tail_ptr, tail_upd;
};

// slots that fit `lds` bytes with factors of `scalar` bytes (after a zero slot)
constexpr int resident_cap(int lds, int scalar) { return lds / (8 * scalar) - 1; }

// cap_top, cap: slots of the last part and of the others, at most (the zero
// slot not counted); R.ok = false when the tree does not divide that way
void build_resident(const Symbolic &S, int cap_top, int cap, ResidentPlan &R);

}  // namespace bpf
