// Expectation value of Pauli strings on a caller-owned device state without any allocation.
//
// The same computation as Engine::get_expectation_value (the same kernels, in the same order, with
// the same host-side combination), for callers that cannot allocate.  Its uploaded strings,
// partial sums and per-string results live in `scratch`, one file-scope device array per GPU,
// whose address on each device is looked up once (hipGetSymbolAddress) with that device current.
// Host-side work uses fixed-size stack chunks: no device or heap allocation happens in a call.
// Calls that overlap on one GPU share that GPU's array and race.
#include "noalloc.hpp"

#include <hip/hip_runtime.h>

#include <algorithm>
#include <complex>
#include <mutex>

#include "energy.hpp"
#include "planner.hpp"

namespace qs {

namespace {

// scratch layout (byte offsets, 256-byte aligned)
constexpr size_t kRecordsOff = 0;                                                            // one plan's records
constexpr size_t kPartialsOff = kRecordsOff + ((kEnergyRecordBytes + 255) & ~size_t(255));  // double[kEnergyPartials]
constexpr size_t kResultsOff = kPartialsOff + sizeof(double) * dev::kEnergyPartials;        // double[plans]
constexpr size_t kPlans = kNoAllocMaxTerms / kEnergyMaxStrings;
constexpr size_t kScratchBytes = kResultsOff + sizeof(double) * kPlans;
static_assert(kPartialsOff % 256 == 0 && kResultsOff % 256 == 0, "scratch regions stay 256-byte aligned");
static_assert(kScratchBytes <= kNoAllocScratchBytes, "scratch size as declared in noalloc.hpp");

}  // namespace

static __device__ __align__(256) unsigned char scratch[kScratchBytes];

namespace {

constexpr int kMaxDevices = 64;
std::mutex g_mutex;
char *g_scratch[kMaxDevices] = {};

// This GPU's copy of `scratch`, looked up on the first call with the device current.  The name
// `scratch` is a host-side stand-in: only the looked-up address may reach kernels and copies.
char *scratch_on_current_device() {
  int dev = 0;
  QS_HIP(hipGetDevice(&dev));
  if (dev < 0 || dev >= kMaxDevices) throw DeviceError("expectation_noalloc: device index out of range");
  std::lock_guard<std::mutex> lock(g_mutex);
  if (!g_scratch[dev]) {
    void *p = nullptr;
    QS_HIP(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) throw DeviceError("expectation_noalloc: no device address for the scratch array");
    g_scratch[dev] = static_cast<char *>(p);
  }
  return g_scratch[dev];
}

// String t as  omega * X^x Z^z  (the engine's encoding), with its local indices mapped.
void encode(size_t t, const uint32_t *term_idx, const uint8_t *term_ops, const size_t *term_offsets,
            const uint32_t *positions, size_t n_positions, EnergyTerm *out) {
  PauliEncoder e;
  for (size_t j = term_offsets[t]; j < term_offsets[t + 1]; ++j) {
    if (term_idx[j] >= n_positions) throw ValueError("qubit_operator acts on more qubits than contained in the qureg.");
    const char op = (char)term_ops[j];
    if (op != 'X' && op != 'Y' && op != 'Z') throw ValueError("Pauli operator must be X, Y or Z");
    e.add(positions[term_idx[j]], op);
  }
  out->x = e.x;
  out->z = e.z;
  out->omega = e.omega;
}

}  // namespace

double expectation_noalloc(const void *state, unsigned n_qubits, bool c64, const uint32_t *term_idx,
                           const uint8_t *term_ops, const size_t *term_offsets, size_t n_terms, const double *coeffs,
                           const uint32_t *positions, size_t n_positions) {
  if (n_terms > kNoAllocMaxTerms)
    throw ValueError("expectation_noalloc: at most 4096 Pauli strings per call (the scratch capacity)");
  if (n_qubits > 40) throw ValueError("expectation_noalloc: at most 40 qubits");
  if (!state) throw ValueError("expectation_noalloc: the state pointer is null");
  for (size_t l = 0; l < n_positions; ++l)
    if (positions[l] >= n_qubits) throw ValueError("expectation_noalloc: a qubit position lies outside the state");
  // validate every string before any device work
  for (size_t t = 0; t < n_terms; ++t) {
    EnergyTerm e;
    encode(t, term_idx, term_ops, term_offsets, positions, n_positions, &e);
  }
  if (n_terms == 0) return 0.0;
  char *base = scratch_on_current_device();
  double *d_partials = reinterpret_cast<double *>(base + kPartialsOff);
  double *d_results = reinterpret_cast<double *>(base + kResultsOff);
  const hipStream_t s = nullptr;  // the null stream; the call returns when its work is done
  QS_HIP(hipStreamSynchronize(s));
  EnergyTerm terms[kEnergyMaxStrings];
  EnergyPlan plan;
  char records[kEnergyRecordBytes];
  size_t plans = 0;
  for (size_t t0 = 0; t0 < n_terms; t0 += kEnergyMaxStrings, ++plans) {
    const size_t m = std::min<size_t>(kEnergyMaxStrings, n_terms - t0);
    for (size_t i = 0; i < m; ++i) {
      encode(t0 + i, term_idx, term_ops, term_offsets, positions, n_positions, &terms[i]);
      terms[i].c = coeffs[t0 + i];
    }
    plan_energy(terms, (int)m, n_qubits, c64, kEnergyWorkgroups, plan);
    const EnergyRecords rec = pack_energy(plan, records);
    // in stream order: the previous plan's kernels have read their records
    if (rec.bytes) QS_HIP(hipMemcpy(base + kRecordsOff, records, rec.bytes, hipMemcpyHostToDevice));
    if (c64)
      dev::energy<float>(static_cast<const float2 *>(state), n_qubits, plan, base + kRecordsOff, rec, d_partials,
                         d_results + plans, s);
    else
      dev::energy<double>(static_cast<const double2 *>(state), n_qubits, plan, base + kRecordsOff, rec, d_partials,
                          d_results + plans, s);
  }
  double res[kPlans];
  QS_HIP(hipMemcpy(res, d_results, plans * sizeof(double), hipMemcpyDeviceToHost));
  double total = 0.0;
  for (size_t k = 0; k < plans; ++k) total += res[k];
  return total;
}

}  // namespace qs
