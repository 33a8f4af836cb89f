// Plan of an expectation value sum_t c_t <psi|P_t|psi>: which Pauli strings are evaluated together
// from one LDS tile of the state (energy.hip).  Plain fixed-size records and no allocation, so the
// no-allocation entry point can build one on its stack.
#pragma once

#include <complex>
#include <cstddef>
#include <cstdint>
#include <vector>

#include "layout.hpp"

namespace qs {

// Pauli strings of one plan; a longer operator is evaluated plan by plan.
constexpr int kEnergyMaxStrings = 128;
constexpr int kEnergyMaxGens = 8;
constexpr int kEnergyLaneBits = 8;  // tile-local bits [0, 8) are the thread index

// One string at the amplitudes i of a tile, partner j = i ^ x: its contribution is
// w (-1)^{popcount(base & z) + popcount(l & zloc)} times Re (kind 0) or Im (kind 1) of
// conj(psi_i) psi_j, base the tile's first index and l the tile-local index.
struct EnergyString {
  uint64_t z;
  double w;
  uint32_t zloc, pad;
};

// Strings with the same x and the same kind: tile-local XOR mask `mask`.  The first string is in the
// record (most x have one string, and a kernel then waits for one scalar load, not two); the others
// are strings [next, next + more).
struct EnergyGroup {
  EnergyString head;
  uint32_t mask, kind, next, more;
};

// A pass over the state in tiles of 2^t amplitudes: the low L index bits (contiguous) and the span
// of `gen` (one generator per tile-local bit L .. t-1, low L bits zero).  `pivot` holds the
// positions, ascending, that enumerate the tiles: tile k starts at k << L with a zero inserted at
// every pivot.
struct EnergyPass {
  uint64_t gen[kEnergyMaxGens];
  uint32_t first_group, n_groups;
  uint8_t pivot[kEnergyMaxGens];
};

struct EnergyPlan {
  uint32_t t, L, h;             // tile bits, contiguous bits, generators (t = L + h)
  uint32_t n_passes, n_groups, n_strings;
  EnergyPass passes[kEnergyMaxStrings];
  EnergyGroup groups[kEnergyMaxStrings + 1];  // one spare: kernels load one group ahead
  EnergyString strings[kEnergyMaxStrings];
};

// The used records of a plan, packed for one upload: passes, then groups, then strings.
constexpr size_t kEnergyRecordBytes =
    size_t(kEnergyMaxStrings) * (sizeof(EnergyPass) + sizeof(EnergyString)) + (kEnergyMaxStrings + 1) * sizeof(EnergyGroup);
struct EnergyRecords {
  size_t groups, strings, bytes;  // byte offsets, and the size
};
EnergyRecords pack_energy(const EnergyPlan &plan, char *out);

// One string omega X^x Z^z with coefficient c, encoded as in encode_pauli (planner.hpp).
struct EnergyTerm {
  uint64_t x, z;
  std::complex<double> omega;
  double c;
};

// Plans `count` <= kEnergyMaxStrings terms on a state of n qubits.  Terms that are not Hermitian
// are left out: the real part of their expectation value is zero.  workgroups: where the state has few
// tiles, the strings are spread over more passes until about that many workgroups have work.
void plan_energy(const EnergyTerm *terms, int count, unsigned n, bool c64, uint64_t workgroups, EnergyPlan &plan);
constexpr uint64_t kEnergyWorkgroups = 1024;  // fills the chip: for a plan that runs alone

// ---- sum_t c_t P_t applied to a state (qubit operators and the terms of a time evolution) ----------

// Strings with the same x and kind, the first in the record as in EnergyGroup: each contributes
// w (-1)^{popcount(i & z)} psi_{i ^ x}, kind 1 times the imaginary unit (the sign (-1)^{popcount(x & z)} is
// folded into w).  The partner is in the tile, at tile-local index ^ mask (inside), or read from memory.
struct SumGroup {
  EnergyString head;
  uint64_t x;
  uint32_t mask, kind, inside, next, more, pad;
};

constexpr uint32_t kSumTileBits = 10;
struct SumPlan {
  uint32_t t, L, h;  // the tile, as in EnergyPlan
  uint64_t gen[kEnergyMaxGens];
  uint8_t pivot[kEnergyMaxGens];
  std::vector<SumGroup> groups;  // and one spare: kernels load one group ahead
  std::vector<EnergyString> strings;
};
// c may be complex; the strings need not be Hermitian.
struct SumTerm {
  uint64_t x, z;
  std::complex<double> c;  // with the string's phase
};
void plan_sum(const std::vector<SumTerm> &terms, unsigned n, bool c64, SumPlan &plan);

}  // namespace qs
