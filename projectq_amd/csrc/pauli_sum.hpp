// Launchers of the Pauli-sum kernels (pauli_sum.hip).
#pragma once

#include "common.hpp"
#include "energy_plan.hpp"

namespace qs {
namespace dev {

constexpr uint32_t kSumPartials = 4096;

// The Taylor terms of one step of a time evolution: how many ran, and whether the last one was small
// enough to stop.  Kernels of terms after that do nothing.
struct EvolveState {
  int done, terms;
};

// The operator's records in device memory.
struct SumRecords {
  const SumGroup *groups;
  const EnergyString *strings;
};

// dst_i <- f sum_t c_t (P_t src)_i.  With `evolve`, unless evolve->done: also, on entries with
// (i & cmask) == cmask, out_i += dst_i, and partials <- sums of |dst_i|^2 there (kSumPartials doubles at
// most).  first: the step's first term, out_i <- g src_i + dst_i on those entries and src_i elsewhere.
template <typename R>
void pauli_sum(const amp_t<R> *src, amp_t<R> *dst, amp_t<R> *out, unsigned n, const SumPlan &plan, const SumRecords &rec,
               std::complex<double> f, bool first, std::complex<double> g, uint64_t cmask, const EvolveState *evolve,
               double *partials, hipStream_t s);
// Operators that need no tile: a few strings on a small state, one or two strings with one x on any.  The terms
// travel in the kernel arguments.
bool pauli_few(const std::vector<SumTerm> &terms, unsigned n);
template <typename R>
void pauli_map(const amp_t<R> *src, amp_t<R> *dst, uint64_t n_amps, const std::vector<SumTerm> &terms, hipStream_t s);
// state->terms += 1, state->done <- the norm of the last term is at most 1e-12; mirrored to `host`
// (pinned).  Does nothing once done.
void evolve_check(const double *partials, unsigned n, const SumPlan &plan, EvolveState *state, EvolveState *host, hipStream_t s);
void evolve_reset(EvolveState *state, hipStream_t s);

}  // namespace dev
}  // namespace qs
