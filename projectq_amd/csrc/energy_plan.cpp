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

namespace {

// The tile of an n-qubit state: at most 2^tmax amplitudes, 256 contiguous bytes.  Small states take
// the tile that holds them.
void tile_of(unsigned n, bool c64, uint32_t tmax, uint32_t *t, uint32_t *L, uint32_t *h) {
  const uint32_t lmin = c64 ? 5u : 4u;
  *t = std::max(8u, std::min(tmax, n));
  *L = n <= *t ? *t : lmin;
  *h = *t - *L;
}

// fills the span up to h generators with the lowest positions it lacks; its pivots, ascending
void complete(Span &span, uint64_t *gen, uint32_t L, uint32_t h, uint8_t *pivot) {
  for (uint32_t p = L; span.n < (int)h; ++p) {
    uint32_t combo;
    const uint64_t rest = span.reduce(uint64_t(1) << p, &combo);
    if (!rest) continue;
    gen[span.n] = uint64_t(1) << p;
    span.add(rest, combo);
  }
  for (uint32_t b = 0; b < h; ++b) {
    const uint8_t p = (uint8_t)top_bit(span.row[b]);
    uint32_t at = b;
    for (; at > 0 && pivot[at - 1] > p; --at) pivot[at] = pivot[at - 1];
    pivot[at] = p;
  }
}

}  // namespace

void plan_energy(const EnergyTerm *terms, int count, unsigned n, bool c64, uint64_t workgroups, EnergyPlan &plan) {
  tile_of(n, c64, c64 ? 12u : 11u, &plan.t, &plan.L, &plan.h);
  // One generator more for segments of 128 bytes: an eighth string per read of the state.  It pays where
  // the state is beyond the caches (from 128 MiB on) and the strings need a second read: 27 qubits complex128,
  // 30 random strings 2.00 -> 1.82 ms, 28 qubits complex64, 40 random strings 3.09 -> 2.91 ms (6 -> 5
  // reads); six strings, one read either way, 0.54 and 0.56 ms; 22 qubits the same.
  if (n >= (c64 ? 24u : 23u) && count > (int)plan.h) {
    --plan.L;
    ++plan.h;
  }
  // 32 KiB of LDS, 256 threads with 16 (complex64) or 8 (complex128) amplitudes each
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
  // fewer strings to a pass where the state has few tiles (it is in the caches then)
  const uint64_t tiles = n > plan.t ? uint64_t(1) << (n - plan.t) : 1;
  const uint64_t want = std::max<uint64_t>(1, (workgroups + tiles - 1) / tiles);
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
    complete(span, gen, plan.L, plan.h, pass.pivot);
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
      const EnergyTerm &lead = terms[order[src.first]];
      uint32_t mask = (uint32_t)(lead.x & low);
      for (uint32_t b = 0; b < plan.h; ++b)
        if ((alpha[q] >> b) & 1) mask ^= local[b];
      const bool once = (mask >> kEnergyLaneBits) != 0;  // each pair visited once: twice the weight
      auto string = [&](int s) {
        const EnergyTerm &e = terms[order[s]];
        // Re(omega (pr + i pi)): omega = +-1 takes +-pr, omega = +-i takes -+pi
        const bool im = parity(e.x & e.z);
        double w = e.c * (im ? -e.omega.imag() : e.omega.real());
        if (im) w = -w;  // popcount(j & z) = popcount(i & z) + popcount(x & z)
        EnergyString o{e.z, once ? 2.0 * w : w, (uint32_t)(e.z & low), 0};
        for (uint32_t b = 0; b < plan.h; ++b) o.zloc |= parity(pass.gen[b] & e.z) << (plan.L + b);
        return o;
      };
      for (uint32_t kind = 0, s = (uint32_t)src.first; kind < 2; ++kind) {
        const uint32_t count = (uint32_t)(kind ? src.n_im : src.n_re);
        if (count == 0) continue;
        plan.groups[plan.n_groups++] = EnergyGroup{string((int)s), mask, kind, plan.n_strings, count - 1};
        for (uint32_t i = 1; i < count; ++i) plan.strings[plan.n_strings++] = string((int)(s + i));
        s += count;
      }
    }
    pass.n_groups = plan.n_groups - pass.first_group;
  }
}

EnergyRecords pack_energy(const EnergyPlan &plan, char *out) {
  EnergyRecords r;
  r.groups = plan.n_passes * sizeof(EnergyPass);
  r.strings = r.groups + (plan.n_groups + 1) * sizeof(EnergyGroup);
  r.bytes = r.strings + plan.n_strings * sizeof(EnergyString);
  std::memcpy(out, plan.passes, r.groups);
  std::memcpy(out + r.groups, plan.groups, plan.n_groups * sizeof(EnergyGroup));
  std::memset(out + r.strings - sizeof(EnergyGroup), 0, sizeof(EnergyGroup));
  std::memcpy(out + r.strings, plan.strings, r.bytes - r.strings);
  return r;
}

void plan_sum(const std::vector<SumTerm> &terms, unsigned n, bool c64, SumPlan &plan) {
  tile_of(n, c64, kSumTileBits, &plan.t, &plan.L, &plan.h);
  plan.groups.clear();
  plan.strings.clear();
  const uint64_t low = (uint64_t(1) << plan.L) - 1;
  // highest x first: the generators take the far partners, and those left to memory are near, in
  // the L2 of the workgroup's XCD
  std::vector<uint32_t> order(terms.size());
  for (size_t i = 0; i < order.size(); ++i) order[i] = (uint32_t)i;
  std::stable_sort(order.begin(), order.end(), [&](uint32_t a, uint32_t b) { return terms[a].x > terms[b].x; });
  Span span;
  std::vector<uint32_t> alpha;
  for (size_t i = 0; i < order.size();) {
    const uint64_t x = terms[order[i]].x;
    size_t e = i;
    while (e < order.size() && terms[order[e]].x == x) ++e;
    SumGroup g{};
    g.x = x;
    bool any = false;
    uint32_t combo = 0;
    for (uint32_t kind = 0; kind < 2; ++kind) {
      g.kind = kind;
      g.next = (uint32_t)plan.strings.size();
      g.more = 0;
      bool head = false;
      for (size_t s = i; s < e; ++s) {
        const SumTerm &t = terms[order[s]];
        double w = kind ? t.c.imag() : t.c.real();
        if (w == 0.0) continue;
        if (parity(x & t.z)) w = -w;  // popcount(j & z) = popcount(i & z) + popcount(x & z)
        const EnergyString o{t.z, w, 0, 0};
        if (head) {
          plan.strings.push_back(o);
          ++g.more;
        } else {
          g.head = o;
          head = true;
        }
      }
      if (!head) continue;
      if (!any) {
        any = true;
        const uint64_t rest = span.reduce(x & ~low, &combo);
        g.inside = 1;
        if (rest) {
          if (span.n < (int)plan.h) {
            plan.gen[span.n] = x & ~low;
            span.add(rest, combo);
            combo = 1u << (span.n - 1);
          } else {
            g.inside = 0;
          }
        }
      }
      alpha.push_back(combo);
      plan.groups.push_back(g);
    }
    i = e;
  }
  complete(span, plan.gen, plan.L, plan.h, plan.pivot);
  auto place = [&](EnergyString &o) {
    o.zloc = (uint32_t)(o.z & low);
    for (uint32_t b = 0; b < plan.h; ++b) o.zloc |= parity(plan.gen[b] & o.z) << (plan.L + b);
  };
  for (size_t k = 0; k < plan.groups.size(); ++k) {
    SumGroup &g = plan.groups[k];
    if (g.inside) g.mask = (uint32_t)(g.x & low) | alpha[k] << plan.L;
    place(g.head);
  }
  for (EnergyString &o : plan.strings) place(o);
  plan.groups.push_back(SumGroup{});
}

}  // namespace qs
