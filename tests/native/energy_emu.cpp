// Test-only CPU model of the expectation-value kernel (projectq_amd/csrc/energy.hip): the product's
// plan evaluated tile by tile as the kernel does, and each pass's tiles checked to cover the state.
#include <vector>

#include "energy_plan.hpp"

using namespace qs;

static int odd(uint64_t v) { return __builtin_popcountll(v) & 1; }

// psi: 2^n interleaved complex doubles.  Returns the number of passes, -1 where a pass does not visit
// every amplitude exactly once, -2 where the records break a limit.
extern "C" int energy_emu(const double *psi, unsigned n, int c64, const unsigned long long *x, const unsigned long long *z,
                          const double *omega, const double *c, int count, double *out) {
  std::vector<EnergyTerm> terms(count);
  for (int t = 0; t < count; ++t) terms[t] = EnergyTerm{x[t], z[t], {omega[2 * t], omega[2 * t + 1]}, c[t]};
  static EnergyPlan plan;
  plan_energy(terms.data(), count, n, c64 != 0, kEnergyWorkgroups, plan);
  if (plan.t != plan.L + plan.h || plan.h > kEnergyMaxGens || plan.n_passes > (uint32_t)kEnergyMaxStrings) return -2;
  const uint64_t tiles = n > plan.t ? uint64_t(1) << (n - plan.t) : 1, N = uint64_t(1) << n;
  const uint32_t size = 1u << plan.t;
  double total = 0.0;
  for (uint32_t p = 0; p < plan.n_passes; ++p) {
    const EnergyPass &pass = plan.passes[p];
    std::vector<int> seen(N, 0);
    for (uint64_t k = 0; k < tiles; ++k) {
      uint64_t base = k << plan.L;
      for (uint32_t b = 0; b < plan.h; ++b) {
        const uint32_t q = pass.pivot[b];
        base = ((base >> q) << (q + 1)) | (base & ((uint64_t(1) << q) - 1));
      }
      std::vector<double> re(size, 0.0), im(size, 0.0);
      for (uint32_t l = 0; l < size; ++l) {
        uint64_t i = base ^ (l & ((1u << plan.L) - 1));
        for (uint32_t b = 0; b < plan.h; ++b)
          if ((l >> (plan.L + b)) & 1) i ^= pass.gen[b];
        if (i >= N) {
          if (n >= 8) return -1;
          continue;
        }
        ++seen[i];
        re[l] = psi[2 * i];
        im[l] = psi[2 * i + 1];
      }
      for (uint32_t g = pass.first_group; g < pass.first_group + pass.n_groups; ++g) {
        const EnergyGroup &gr = plan.groups[g];
        const uint32_t above = gr.mask >> kEnergyLaneBits;
        const uint32_t skip = above ? (1u << (31 - __builtin_clz(above))) << kEnergyLaneBits : 0;
        for (uint32_t s = 0; s <= gr.more; ++s) {
          const EnergyString &st = s ? plan.strings[gr.next + s - 1] : gr.head;
          for (uint32_t l = 0; l < size; ++l) {
            if (l & skip) continue;
            const uint32_t m = l ^ gr.mask;
            const double v = gr.kind == 0 ? re[l] * re[m] + im[l] * im[m] : re[l] * im[m] - im[l] * re[m];
            total += (odd(base & st.z) ^ odd(l & st.zloc)) ? -st.w * v : st.w * v;
          }
        }
      }
    }
    for (int v : seen)
      if (v != 1) return -1;
  }
  *out = total;
  return (int)plan.n_passes;
}

// sum_t c_t (-1)^{popcount(j & z_t)} psi_j, j = i ^ x_t, for every i, through the Pauli-sum plan
// (projectq_amd/csrc/pauli_sum.hip).  Returns the number of groups read from memory, negative as above.
extern "C" int sum_emu(const double *psi, unsigned n, int c64, const unsigned long long *x, const unsigned long long *z,
                       const double *c, int count, double *out) {
  std::vector<SumTerm> terms(count);
  for (int t = 0; t < count; ++t) terms[t] = SumTerm{x[t], z[t], {c[2 * t], c[2 * t + 1]}};
  SumPlan plan;
  plan_sum(terms, n, c64 != 0, plan);
  if (plan.t != plan.L + plan.h || plan.h > kEnergyMaxGens) return -2;
  const uint64_t tiles = n > plan.t ? uint64_t(1) << (n - plan.t) : 1, N = uint64_t(1) << n;
  const uint32_t size = 1u << plan.t;
  std::vector<int> seen(N, 0);
  auto index = [&](uint64_t base, uint32_t l) {
    uint64_t i = base ^ (l & ((1u << plan.L) - 1));
    for (uint32_t b = 0; b < plan.h; ++b)
      if ((l >> (plan.L + b)) & 1) i ^= plan.gen[b];
    return i;
  };
  int outside = 0;
  plan.groups.pop_back();  // the spare
  for (const SumGroup &g : plan.groups) outside += !g.inside;
  for (uint64_t k = 0; k < tiles; ++k) {
    uint64_t base = k << plan.L;
    for (uint32_t b = 0; b < plan.h; ++b) {
      const uint32_t q = plan.pivot[b];
      base = ((base >> q) << (q + 1)) | (base & ((uint64_t(1) << q) - 1));
    }
    for (uint32_t l = 0; l < size; ++l) {
      const uint64_t i = index(base, l);
      if (i >= N) {
        if (n >= 8) return -1;
        continue;
      }
      ++seen[i];
      std::complex<double> u = 0.0;
      for (const SumGroup &g : plan.groups) {
        const uint64_t j = g.inside ? index(base, l ^ g.mask) : i ^ g.x;
        if (j != (i ^ g.x)) return -3;
        const std::complex<double> b(psi[2 * j], psi[2 * j + 1]);
        for (uint32_t s = 0; s <= g.more; ++s) {
          const EnergyString &st = s ? plan.strings[g.next + s - 1] : g.head;
          const double w = (odd(base & st.z) ^ odd(l & st.zloc)) ? -st.w : st.w;
          u += g.kind == 0 ? w * b : std::complex<double>(0.0, w) * b;
        }
      }
      out[2 * i] = u.real();
      out[2 * i + 1] = u.imag();
    }
  }
  for (int v : seen)
    if (v != 1) return -1;
  return outside;
}
