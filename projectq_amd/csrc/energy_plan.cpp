// Host side of the expectation value (see energy_plan.hpp): grouping Pauli strings into passes.
#include "energy_plan.hpp"

#include <algorithm>
#include <cstring>

namespace qs {

namespace {

int top_bit(uint64_t v) { return 63 - __builtin_clzll(v); }
uint32_t parity(uint64_t v) { return (uint32_t)__builtin_popcountll(v) & 1u; }

// Row echelon basis of the x parts above the contiguous bits, each row with the set of generators
// that add up to it.
struct Span {
  uint64_t row[kEnergyMaxGens];
  uint32_t combo[kEnergyMaxGens];
  int n = 0;

  // subtracts the rows from v; what is left, and the generators used so far
  uint64_t reduce(uint64_t v, uint32_t *combo_out) const {
    uint32_t c = 0;
    for (int i = 0; i < n; ++i)
      if ((v >> top_bit(row[i])) & 1) {
        v ^= row[i];
        c ^= combo[i];
      }
    *combo_out = c;
    return v;
  }
  // a new generator (number n) whose reduced form is `left`
  void add(uint64_t left, uint32_t combo_left) {
    const int p = top_bit(left);
    const uint32_t mine = combo_left ^ (1u << n);
    for (int i = 0; i < n; ++i)
      if ((row[i] >> p) & 1) {
        row[i] ^= left;
        combo[i] ^= mine;
      }
    row[n] = left;
    combo[n] = mine;
    ++n;
  }
};

}  // namespace

void plan_energy(const EnergyTerm *terms, int count, unsigned n, bool c64, EnergyPlan &plan) {
  // Tile: 32 KiB of LDS, 256 threads with 16 (complex64) or 8 (complex128) amplitudes each; 256
  // contiguous bytes.  Small states take the tile that holds them.
  const uint32_t tmax = c64 ? 12u : 11u, lmin = c64 ? 5u : 4u;
  plan.t = std::max(8u, std::min(tmax, n));
  plan.L = std::min(lmin, n);
  if (n <= plan.t) plan.L = plan.t;
  plan.h = plan.t - plan.L;
  plan.n_passes = plan.n_groups = plan.n_strings = 0;

  // order by x, real kinds first
  int order[kEnergyMaxStrings], m = 0;
  for (int i = 0; i < count; ++i) {
    const EnergyTerm &e = terms[i];
    const double sigma = parity(e.x & e.z) ? -1.0 : 1.0;
    if ((e.omega * e.omega).real() * sigma > 0.0) order[m++] = i;
  }
  std::sort(order, order + m, [&](int a, int b) {
    const uint64_t xa = terms[a].x, xb = terms[b].x;
    const uint32_t ka = parity(xa & terms[a].z), kb = parity(xb & terms[b].z);
    return xa != xb ? xa < xb : ka != kb ? ka < kb : a < b;
  });
  // groups of equal x, in that order
  struct Group {
    int first, n_re, n_im;
    uint64_t hi;
  };
  Group g[kEnergyMaxStrings];
  int n_groups = 0;
  const uint64_t low = plan.L >= 64 ? ~uint64_t(0) : (uint64_t(1) << plan.L) - 1;
  for (int i = 0; i < m;) {
    int e = i, re = 0;
    while (e < m && terms[order[e]].x == terms[order[i]].x) {
      re += !parity(terms[order[e]].x & terms[order[e]].z);
      ++e;
    }
    g[n_groups++] = Group{i, re, e - i - re, terms[order[i]].x & ~low};
    i = e;
  }
  // At least about 1024 workgroups where the state has few tiles: the strings are spread over more
  // passes (the state is in the caches then).
  const uint64_t tiles = n > plan.t ? uint64_t(1) << (n - plan.t) : 1;
  const uint64_t want = (1024 + tiles - 1) / tiles;  // passes that fill the chip
  const int most = std::max<int>(1, (int)((uint64_t)(m + (int)want - 1) / want));

  const uint32_t lanes_h = kEnergyLaneBits > (int)plan.L ? std::min(kEnergyLaneBits - plan.L, plan.h) : 0;  // generators on thread bits
  const uint32_t top_h = plan.h - lanes_h;                                                          // on the bits above
  bool used[kEnergyMaxStrings] = {};
  for (int left = n_groups; left > 0;) {
    EnergyPass &pass = plan.passes[plan.n_passes++];
    pass = EnergyPass{};
    pass.first_group = plan.n_groups;
    Span span;
    uint64_t gen[kEnergyMaxGens];
    uint32_t alpha[kEnergyMaxStrings];  // generators of each group taken
    int taken[kEnergyMaxStrings], k = 0, strings = 0;
    for (int i = 0; i < n_groups; ++i) {
      if (used[i] || (k > 0 && strings + g[i].n_re + g[i].n_im > most)) continue;
      uint32_t combo;
      const uint64_t rest = span.reduce(g[i].hi, &combo);
      if (rest) {
        if (span.n == (int)plan.h) continue;
        gen[span.n] = g[i].hi;
        alpha[k] = 1u << span.n;
        span.add(rest, combo);
      } else {
        alpha[k] = combo;
      }
      taken[k++] = i;
      strings += g[i].n_re + g[i].n_im;
      used[i] = true;
      --left;
    }
    // Generators 0 .. top_h-1 go to the tile-local bits above the thread bits, where the kernel
    // visits each pair once; a string whose x lies in the others alone would visit both members.  So
    // each of the others carries one of the first ones: gen_k ^ gen_{k mod top_h}.
    const int from_strings = span.n;
    for (uint32_t p = plan.L; span.n < (int)plan.h; ++p) {
      uint32_t combo;
      const uint64_t rest = span.reduce(uint64_t(1) << p, &combo);
      if (!rest) continue;
      gen[span.n] = uint64_t(1) << p;
      span.add(rest, combo);
    }
    for (uint32_t b = 0; b < plan.h; ++b) {
      uint8_t p = (uint8_t)top_bit(span.row[b]);
      uint32_t at = b;
      for (; at > 0 && pass.pivot[at - 1] > p; --at) pass.pivot[at] = pass.pivot[at - 1];
      pass.pivot[at] = p;
    }
    uint32_t local[kEnergyMaxGens];  // tile-local mask of generator b as a string has it
    for (uint32_t b = 0; b < plan.h; ++b) {
      const uint32_t bit = b < top_h ? plan.L + lanes_h + b : plan.L + (b - top_h);
      local[b] = 1u << bit;
      pass.gen[bit - plan.L] = gen[b];
      if (b >= top_h && top_h > 0 && (int)b < from_strings) {
        const uint32_t a = (b - top_h) % top_h;
        pass.gen[bit - plan.L] ^= gen[a];
        local[b] |= 1u << (plan.L + lanes_h + a);
      }
    }
    for (int q = 0; q < k; ++q) {
      const Group &src = g[taken[q]];
      EnergyGroup &dst = plan.groups[plan.n_groups++];
      const EnergyTerm &lead = terms[order[src.first]];
      dst.mask = (uint32_t)(lead.x & low);
      for (uint32_t b = 0; b < plan.h; ++b)
        if ((alpha[q] >> b) & 1) dst.mask ^= local[b];
      dst.first = plan.n_strings;
      dst.n_re = (uint32_t)src.n_re;
      dst.n_im = (uint32_t)src.n_im;
      const bool once = (dst.mask >> kEnergyLaneBits) != 0;  // each pair visited once: twice the weight
      for (int s = src.first; s < src.first + src.n_re + src.n_im; ++s) {
        const EnergyTerm &e = terms[order[s]];
        EnergyString &o = plan.strings[plan.n_strings++];
        // Re(omega (pr + i pi)): omega = +-1 takes +-pr, omega = +-i takes -+pi
        const bool im = parity(e.x & e.z);
        double w = e.c * (im ? -e.omega.imag() : e.omega.real());
        if (parity(e.x & e.z)) w = -w;  // popcount(j & z) = popcount(i & z) + popcount(x & z)
        o.w = once ? 2.0 * w : w;
        o.z = e.z;
        o.zloc = (uint32_t)(e.z & low);
        for (uint32_t b = 0; b < plan.h; ++b) o.zloc |= parity(pass.gen[b] & e.z) << (plan.L + b);
        o.pad = 0;
      }
    }
    pass.n_groups = plan.n_groups - pass.first_group;
  }
}

EnergyRecords pack_energy(const EnergyPlan &plan, char *out) {
  EnergyRecords r;
  r.groups = plan.n_passes * sizeof(EnergyPass);
  r.strings = r.groups + plan.n_groups * sizeof(EnergyGroup);
  r.bytes = r.strings + plan.n_strings * sizeof(EnergyString);
  std::memcpy(out, plan.passes, r.groups);
  std::memcpy(out + r.groups, plan.groups, r.strings - r.groups);
  std::memcpy(out + r.strings, plan.strings, r.bytes - r.strings);
  return r;
}

}  // namespace qs
