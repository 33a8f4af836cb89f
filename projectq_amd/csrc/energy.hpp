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

}  // namespace dev
}  // namespace qs
