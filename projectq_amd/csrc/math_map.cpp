// Which emulate_math calls the gather kernel takes (see math_map.hpp).
#include "math_map.hpp"

#include <algorithm>

namespace qs {

BitRuns runs_of(const std::vector<unsigned> &positions) {
  BitRuns r{};
  for (size_t b = 0; b < positions.size(); ++b) {
    if (r.n > 0 && r.pos[r.n - 1] + r.len[r.n - 1] == (int)positions[b]) {
      ++r.len[r.n - 1];
    } else {
      r.pos[r.n] = (uint8_t)positions[b];
      r.bit[r.n] = (uint8_t)b;
      r.len[r.n] = 1;
      ++r.n;
    }
  }
  return r;
}

namespace {

// x with a x = 1 (mod N), 0 if there is none
uint64_t inverse_mod(uint64_t a, uint64_t N) {
  int64_t r0 = (int64_t)N, r1 = (int64_t)(a % N), t0 = 0, t1 = 1;
  while (r1) {
    const int64_t q = r0 / r1, r2 = r0 - q * r1, t2 = t0 - q * t1;
    r0 = r1, r1 = r2, t0 = t1, t1 = t2;
  }
  return r0 == 1 ? (uint64_t)((t0 % (int64_t)N + (int64_t)N) % (int64_t)N) : 0;
}

}  // namespace

bool plan_math_gather(int opcode, int64_t a, int64_t N, const std::vector<std::vector<unsigned>> &regs, uint64_t cmask,
                      unsigned n, bool c64, MathGather *out) {
  MathGather &G = *out;
  G = MathGather{};
  const size_t k = regs.size();
  if (k < 1 || k > 3 || n > (unsigned)kMaxBits) return false;
  uint64_t seen = cmask, mask[3] = {0, 0, 0};
  for (size_t r = 0; r < k; ++r) {
    if (regs[r].empty() || regs[r].size() > 30) return false;  // register values are then plain ints
    for (unsigned p : regs[r]) {
      if ((seen >> p) & 1) return false;  // a qubit named twice, or a control inside a register
      seen |= uint64_t(1) << p;
      mask[r] |= uint64_t(1) << p;
    }
    G.width[r] = (uint32_t)regs[r].size();
    G.reg[r] = runs_of(regs[r]);
  }
  G.n_regs = (int32_t)k;
  G.cmask = cmask;
  const uint64_t w0 = G.width[0], w1 = G.width[1], w2 = G.width[2];
  const int64_t int_max = 0x7fffffff;
  switch (opcode) {
    case 0:  // x + a wraps modulo 2^width on every register
      G.source = kSrcAddConstant;
      G.a = (uint64_t)a;
      G.changed = mask[0] | mask[1] | mask[2];
      break;
    case 3:  // v + u modulo 2^w0: one to one in v while v is no wider than u
      if (k < 2 || w1 > w0) return false;
      G.source = kSrcSubtract;
      G.carry = k == 3;
      G.changed = mask[1] | mask[2];
      break;
    case 4:
      if (k != 2) return false;
      G.source = kSrcAdd;
      G.changed = mask[1];
      break;
    case 5:
      if (k < 2) return false;
      G.source = kSrcAdd;
      G.carry = k == 3;
      G.changed = mask[1] | mask[2];
      break;
    case 6:  // the third register becomes 0 or 1: one to one on a single qubit
      if (k != 3 || w2 != 1) return false;
      G.source = kSrcCompare;
      G.changed = mask[2];
      break;
    case 7:
    case 8: {  // results outside a C++ int are an error, which the general path finds
      if (k != 3 || w0 + w1 > 31) return false;
      const int64_t most = ((int64_t(1) << w0) - 1) * ((int64_t(1) << w1) - 1) + (int64_t(1) << w2) - 1;
      if (most > int_max) return false;
      G.source = opcode == 7 ? kSrcMulSubtract : kSrcMulAdd;
      G.changed = mask[2];
      break;
    }
    case 1:
    case 2: {  // residues: sources N apart, added in increasing index order as the reference does
      const int64_t top = (int64_t(1) << w0) - 1;
      if (k != 1 || N < 2 || N > int_max || N > top + 1 || a < 0 || a > int_max) return false;
      if (opcode == 1 ? top + a > int_max : a > int_max / top) return false;  // no wrap of the C++ int
      const bool ordered = std::is_sorted(regs[0].begin(), regs[0].end());
      if (!ordered && 2 * N < top + 1) return false;  // three sources or more: their order matters
      G.N = (uint64_t)N;
      G.magic = (uint64_t)((((unsigned __int128)1) << 64) / (unsigned __int128)N);
      if (opcode == 1) {
        G.source = kSrcAddMod;
        G.a = (uint64_t)(a % N);
      } else {
        G.source = kSrcMulMod;
        G.a = inverse_mod((uint64_t)a, (uint64_t)N);
        if (G.a == 0) return false;  // not a unit: classes of sources other than x + kN
      }
      G.changed = mask[0];
      break;
    }
    default:
      return false;
  }
  for (size_t r = 0; r < k; ++r) G.moves[r] = (G.changed & mask[r]) != 0;
  // Traversal: 256 contiguous bytes, then the lowest bits of the registers that change, then the rest
  // in memory order.  An addition moves neighbours in the first register to neighbouring values of
  // the second, whole rows apart in memory; with both in one workgroup every cache line it reads is
  // used in full.
  std::vector<unsigned> order;
  uint64_t in = 0;
  auto take = [&](unsigned p) {
    if (p < n && !((in >> p) & 1)) {
      in |= uint64_t(1) << p;
      order.push_back(p);
    }
  };
  for (unsigned p = 0; p < (c64 ? 5u : 4u); ++p) take(p);
  for (size_t b = 0; b < 12 && order.size() < 12; ++b)
    for (size_t r = 0; r < k; ++r)
      if ((G.changed & mask[r]) && b < regs[r].size() && order.size() < 12) take(regs[r][b]);
  for (unsigned p = 0; p < n; ++p) take(p);
  G.order = runs_of(order);
  for (int b = 0; b < kMathThreadBits; ++b) {
    G.step[b] = 8u + b < n ? uint64_t(1) << order[8 + b] : 0;
    for (size_t r = 0; r < k; ++r) G.reg_step[b][r] = (uint32_t)gather_bits(G.step[b], G.reg[r]);
  }
  return true;
}

bool plan_math_add(const MathGather &G, MathAdd *out) {
  MathAdd &A = *out;
  A = MathAdd{};
  if (G.source != kSrcAddConstant) return false;
  A.n_regs = G.n_regs;
  A.cmask = G.cmask;
  for (int r = 0; r < G.n_regs; ++r) {
    std::vector<unsigned> at(G.width[r]);
    for (uint32_t b = 0; b < G.width[r]; ++b) at[b] = (unsigned)__builtin_ctzll(scatter_bits(uint64_t(1) << b, G.reg[r]));
    const bool up = std::is_sorted(at.begin(), at.end()), down = std::is_sorted(at.rbegin(), at.rend());
    if (!up && !down) return false;
    if (!up) A.reversed |= 1u << r;
    for (uint32_t b = 0; b < G.width[r]; ++b) {
      const uint64_t bit = uint64_t(1) << (up ? at[b] : 63 - at[b]);
      A.mask[r] |= bit;
      if ((G.a >> b) & 1) A.sub[r] |= bit;
    }
  }
  return true;
}

bool plan_math_tile(const MathGather &G, unsigned n, bool c64, MathTile *out) {
  MathTile &T = *out;
  T = MathTile{};
  const unsigned most = c64 ? kMathTileBits64 : kMathTileBits128;
  // the changing bits and 256 contiguous bytes; then the lowest positions that are no controls
  uint64_t in = G.changed;
  for (unsigned p = 0; p < (c64 ? 5u : 4u) && p < n; ++p) in |= uint64_t(1) << p;
  if ((unsigned)__builtin_popcountll(in) > most) return false;
  for (unsigned p = 0; p < n && (unsigned)__builtin_popcountll(in) < most; ++p)
    if (!((G.cmask >> p) & 1)) in |= uint64_t(1) << p;
  T.fixed = G.cmask & ~in;
  std::vector<unsigned> at, rest;
  for (unsigned p = 0; p < n; ++p) {
    if ((in >> p) & 1) at.push_back(p);
    else if (!((T.fixed >> p) & 1)) rest.push_back(p);
  }
  T.m = (uint32_t)at.size();
  T.outside = (uint32_t)rest.size();
  T.tile = runs_of(at);
  T.tile_id = runs_of(rest);
  for (int b = 0; b < kMathThreadBits; ++b) {
    T.step[b] = 8u + b < T.m ? uint64_t(1) << at[8 + b] : 0;
    for (int r = 0; r < G.n_regs; ++r) T.reg_step[b][r] = (uint32_t)gather_bits(T.step[b], G.reg[r]);
  }
  T.changed = (uint32_t)gather_bits(G.changed, T.tile);
  for (int r = 0; r < G.n_regs; ++r) {
    if (!G.moves[r]) continue;
    std::vector<unsigned> local(G.width[r]);
    for (uint32_t b = 0; b < G.width[r]; ++b)
      local[b] = (unsigned)__builtin_ctzll(gather_bits(scatter_bits(uint64_t(1) << b, G.reg[r]), T.tile));
    T.local[r] = runs_of(local);
  }
  return true;
}

}  // namespace qs
