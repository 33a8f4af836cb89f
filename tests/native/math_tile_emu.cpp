// Test-only CPU model of emulate_math in place through tiles (k_math_tile): every destination's sources,
// against those of the gather plan of the same call.
#include <cstddef>

#include "math_map.hpp"

using namespace qs;

namespace {
template <int S>
bool same(const MathGather &G, const MathTile &T, unsigned n) {
  constexpr bool mod = S == kSrcAddMod || S == kSrcMulMod;
  std::vector<char> seen(size_t(1) << n, 0);
  for (uint64_t id = 0; id < uint64_t(1) << T.outside; ++id) {
    const uint64_t base = scatter_bits(id, T.tile_id) | T.fixed;
    for (uint32_t l = 0; l < (1u << T.m); ++l) {
      uint64_t i = base | scatter_bits(l & 255u, T.tile);
      for (int b = 0; b < kMathThreadBits; ++b)
        if ((l >> (8 + b)) & 1) {
          i |= T.step[b];
          for (int r = 0; r < G.n_regs; ++r)
            if (gather_bits(T.step[b], G.reg[r]) != T.reg_step[b][r]) return false;
        }
      if (i != (base | scatter_bits(l, T.tile))) return false;
      if (i >> n || seen[i]) return false;
      seen[i] = 1;
      if ((i & G.cmask) != G.cmask) continue;  // keeps its amplitude
      uint64_t x[3] = {0, 0, 0};
      for (int r = 0; r < G.n_regs; ++r) x[r] = gather_bits(i, G.reg[r]);
      if (mod && x[0] < G.N) {  // the kernel's 32-bit form
        uint64_t y[3] = {x[0], 0, 0};
        if (!math_source<S>(G, y[0], y[1], y[2])) return false;
        if (residue_source32<S>((uint32_t)x[0], (uint32_t)G.a, (uint32_t)G.N, (uint32_t)(G.magic >> 32)) != y[0]) return false;
      }
      if (!math_source<S>(G, x[0], x[1], x[2])) continue;
      do {
        uint64_t s = i & ~G.changed;
        uint32_t sl = l & ~T.changed;
        for (int r = 0; r < G.n_regs; ++r)
          if (G.moves[r]) {
            s |= scatter_bits(x[r], G.reg[r]);
            sl |= scatter_bits32((uint32_t)x[r], T.local[r]);
          }
        if (sl >> T.m || (base | scatter_bits(sl, T.tile)) != s) return false;
        x[0] += G.N;
      } while (mod && x[0] >> G.width[0] == 0);
    }
  }
  for (uint64_t i = 0; i < (uint64_t(1) << n); ++i)
    if (!seen[i] && (i & G.cmask) == G.cmask) return false;
  return true;
}
}  // namespace

// 0: no gather plan, 1: no tile plan, 2: the same sources, 3: not the same
extern "C" int math_tile_emu(int opcode, long long a, long long N, const unsigned *qubits, const unsigned *widths, int n_regs,
                         unsigned long long cmask, unsigned n, int c64) {
  std::vector<std::vector<unsigned>> regs;
  for (int r = 0; r < n_regs; ++r) {
    regs.emplace_back(qubits, qubits + widths[r]);
    qubits += widths[r];
  }
  MathGather G;
  MathTile T;
  if (!plan_math_gather(opcode, a, N, regs, cmask, n, c64 != 0, &G)) return 0;
  if (!plan_math_tile(G, n, c64 != 0, &T)) return 1;
  if (T.m > (c64 ? kMathTileBits64 : kMathTileBits128)) return 3;
  bool ok = false;
  switch (G.source) {
    case kSrcAddConstant: ok = same<kSrcAddConstant>(G, T, n); break;
    case kSrcSubtract: ok = same<kSrcSubtract>(G, T, n); break;
    case kSrcAdd: ok = same<kSrcAdd>(G, T, n); break;
    case kSrcCompare: ok = same<kSrcCompare>(G, T, n); break;
    case kSrcMulSubtract: ok = same<kSrcMulSubtract>(G, T, n); break;
    case kSrcMulAdd: ok = same<kSrcMulAdd>(G, T, n); break;
    case kSrcAddMod: ok = same<kSrcAddMod>(G, T, n); break;
    case kSrcMulMod: ok = same<kSrcMulMod>(G, T, n); break;
  }
  return ok ? 2 : 3;
}
