// Launchers of the expectation-value kernels (energy.hip).
#pragma once

#include "common.hpp"
#include "energy_plan.hpp"

namespace qs {
namespace dev {

constexpr int kEnergyThreads = 256;

// Partial sums a plan may leave, at most: the workgroups of the launch.
constexpr uint32_t kEnergyPartials = 4096;

// *out <- the plan's expectation value on psi (n qubits).  d_records: pack_energy's buffer in device
// memory, rec its offsets; partials: kEnergyPartials doubles; out may be pinned host memory.
template <typename R>
void energy(const amp_t<R> *psi, unsigned n, const EnergyPlan &plan, const char *d_records, const EnergyRecords &rec,
            double *partials, double *out, hipStream_t s);

// ---- batches of circuits (batch_energy.hip) ----
// One pass of one circuit's plan over its tiles: group and string indices are batch-wide.
struct BatchEnergyPass {
  uint64_t state_off, n_amps;  // the circuit's amplitudes
  uint32_t L, h;
  EnergyPass pass;
};
// One workgroup: tiles [tile, tile + tiles) of pass `pass`, its sum to partials[slot]; kNoPass marks an idle
// workgroup (the launch pads every XCD's share of workgroups to the same length).
constexpr uint32_t kNoPass = 0xffffffffu;
struct BatchEnergyBlock {
  uint32_t pass, tile, tiles, slot;
};
// partials of the workgroups, all of whose passes have tiles of 2^t amplitudes, or of any size (kMixedTiles)
constexpr uint32_t kMixedTiles = 0;
template <typename R>
void batch_energy(const amp_t<R> *psi, uint32_t t, const BatchEnergyPass *passes, const BatchEnergyBlock *blocks,
                  uint32_t n_blocks, const EnergyGroup *groups, const EnergyString *strings, double *partials, hipStream_t s);
// energies[c] <- sum of partials [first[c], first[c + 1]) in a fixed order
void batch_energy_finish(const uint32_t *first, int n_circuits, const double *partials, double *energies, hipStream_t s);

}  // namespace dev
}  // namespace qs
