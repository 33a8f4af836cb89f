// Plan of an expectation value sum_t c_t <psi|P_t|psi>: which Pauli strings are evaluated together
// from one LDS tile of the state (energy.hip).  Plain fixed-size records and no allocation, so the
// no-allocation entry point can build one on its stack.
#pragma once

#include <complex>
#include <cstddef>
#include <cstdint>

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

// Strings with the same x: tile-local XOR mask `mask`; strings [first, first + n_re) are of kind 0
// and the n_im after them of kind 1.
struct EnergyGroup {
  uint32_t mask, first, n_re, n_im;
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
  EnergyGroup groups[kEnergyMaxStrings];
  EnergyString strings[kEnergyMaxStrings];
};

// The used records of a plan, packed for one upload: passes, then groups, then strings.
constexpr size_t kEnergyRecordBytes =
    size_t(kEnergyMaxStrings) * (sizeof(EnergyPass) + sizeof(EnergyGroup) + sizeof(EnergyString));
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
// are left out: the real part of their expectation value is zero.
void plan_energy(const EnergyTerm *terms, int count, unsigned n, bool c64, EnergyPlan &plan);

}  // namespace qs
