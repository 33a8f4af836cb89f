// Test-only CPU model of the emulate_math gather (projectq_amd/csrc/math.hip): the sources of every
// destination, computed from the plan as the kernel does.
#include "math_map.hpp"

using namespace qs;

// Returns 0 where the plan does not cover the call.  Else first[i] .. first[i + 1] are the places in
// `sources` of destination i's sources, in the order they are added; visited[c] is the destination
// of counter c.
extern "C" int math_emu(int opcode, long long a, long long N, const unsigned *qubits, const unsigned *widths, int n_regs,
                        unsigned long long cmask, unsigned n, int c64, unsigned *first, unsigned *sources, unsigned *visited) {
  std::vector<std::vector<unsigned>> regs;
  for (int r = 0; r < n_regs; ++r) {
    regs.emplace_back(qubits, qubits + widths[r]);
    qubits += widths[r];
  }
  MathGather G;
  if (!plan_math_gather(opcode, a, N, regs, cmask, n, c64 != 0, &G)) return 0;
  unsigned at = 0;
  for (uint64_t i = 0; i < (uint64_t(1) << n); ++i) {
    first[i] = at;
    if ((i & cmask) != cmask) {
      sources[at++] = (unsigned)i;
      continue;
    }
    uint64_t x[3] = {0, 0, 0};
    for (int r = 0; r < G.n_regs; ++r) x[r] = gather_bits(i, G.reg[r]);
    bool any = false;
    switch (G.source) {
      case kSrcAddConstant: any = math_source<kSrcAddConstant>(G, x[0], x[1], x[2]); break;
      case kSrcSubtract: any = math_source<kSrcSubtract>(G, x[0], x[1], x[2]); break;
      case kSrcAdd: any = math_source<kSrcAdd>(G, x[0], x[1], x[2]); break;
      case kSrcCompare: any = math_source<kSrcCompare>(G, x[0], x[1], x[2]); break;
      case kSrcMulSubtract: any = math_source<kSrcMulSubtract>(G, x[0], x[1], x[2]); break;
      case kSrcMulAdd: any = math_source<kSrcMulAdd>(G, x[0], x[1], x[2]); break;
      case kSrcAddMod: any = math_source<kSrcAddMod>(G, x[0], x[1], x[2]); break;
      case kSrcMulMod: any = math_source<kSrcMulMod>(G, x[0], x[1], x[2]); break;
    }
    if (!any) continue;
    const bool mod = G.source == kSrcAddMod || G.source == kSrcMulMod;
    do {
      uint64_t s = i & ~G.changed;
      for (int r = 0; r < G.n_regs; ++r)
        if (G.moves[r]) s |= scatter_bits(x[r], G.reg[r]);
      sources[at++] = (unsigned)s;
      x[0] += G.N;
    } while (mod && x[0] >> G.width[0] == 0);
  }
  first[uint64_t(1) << n] = at;
  for (uint64_t c = 0; c < (uint64_t(1) << n); ++c) {
    uint64_t i = scatter_bits(c & 255, G.order) | scatter_bits(c >> 12 << 12, G.order);
    for (int b = 0; b < kMathThreadBits; ++b)
      if ((c >> (8 + b)) & 1) {
        i |= G.step[b];
        for (int r = 0; r < G.n_regs; ++r)
          if (gather_bits(G.step[b], G.reg[r]) != G.reg_step[b][r]) return -1;
      }
    visited[c] = (unsigned)i;
  }
  return 1;
}
