// Launchers of the measurement kernels (measure.hip).
#pragma once

#include "common.hpp"
#include "math_map.hpp"

namespace qs {
namespace dev {

// What one measurement leaves on the device for its collapse: the picked index and the factor of the
// amplitudes that stay.
struct Measurement {
  unsigned long long pick;
  double scale;
};

// Chunks of a measurement's first pass, at most.
constexpr uint32_t kMeasureChunks = 32768;
// Subspaces up to this size are measured by one workgroup in one launch.
constexpr uint64_t kMeasureSmall = 4096;

struct MeasureArgs {
  uint64_t n_amps, n_sub;  // amplitudes of the state, and of the subspace outside which they are zero
  BitRuns free;            // the subspace's free bits: compact index -> index
  uint64_t sval, zmask;    // the values of the fixed bits, and their mask
  uint64_t mask;           // index bits of the measured qubits
  uint64_t n_kept;         // of another number of qubits than one: amplitudes of the subspace with one outcome of them
  BitRuns kept;            // their free bits
  double rnd;              // the draw; 0: the reference's loop never runs and the pick is all ones
};

// Pick (the first index whose running norm reaches the draw), projection and renormalisation.  m: one
// record in device memory; pick: pinned, written before `picked` is recorded; sums: 2 kMeasureChunks
// doubles; partials: kReduceGrid doubles.
template <typename R>
void measure(amp_t<R> *psi, const MeasureArgs &a, Measurement *m, unsigned long long *pick, double *sums, double *partials,
             hipEvent_t picked, hipStream_t s);

// *flags (pinned) <- bit 0: an amplitude > tol with index bit p clear, bit 1: one with it set, over the
// subspace.  count: two ints of device memory.
template <typename R>
void classical(const amp_t<R> *psi, uint64_t n_sub, const BitRuns &free, uint64_t sval, int p, double tol, int *count,
               int *flags, hipStream_t s);

}  // namespace dev
}  // namespace qs
