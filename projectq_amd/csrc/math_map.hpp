// Host-side reading of an emulate_math call: whether the map on basis states is known to be one to
// one without looking at it, and its inverse in a form the gather kernel (math.hip) evaluates per
// amplitude.  No HIP dependency, so host-only tools can include it.
#pragma once

#include <cstdint>
#include <vector>

#include "layout.hpp"

namespace qs {

// Bits moved between a compact value and an index, run by run of consecutive positions: value bits
// [bit, bit + len) <-> index bits [pos, pos + len).
struct BitRuns {
  uint32_t n;
  uint8_t pos[kMaxBits], bit[kMaxBits], len[kMaxBits];
};

#ifdef __HIPCC__
#define QS_HD __host__ __device__
#else
#define QS_HD
#endif

QS_HD inline uint64_t gather_bits(uint64_t index, const BitRuns &r) {
  uint64_t v = 0;
  for (uint32_t k = 0; k < r.n; ++k) v |= ((index >> r.pos[k]) & ((uint64_t(1) << r.len[k]) - 1)) << r.bit[k];
  return v;
}
QS_HD inline uint64_t scatter_bits(uint64_t value, const BitRuns &r) {
  uint64_t i = 0;
  for (uint32_t k = 0; k < r.n; ++k) i |= ((value >> r.bit[k]) & ((uint64_t(1) << r.len[k]) - 1)) << r.pos[k];
  return i;
}

QS_HD inline uint32_t scatter_bits32(uint32_t value, const BitRuns &r) {  // positions below 32
  uint32_t i = 0;
  for (uint32_t k = 0; k < r.n; ++k) i |= ((value >> r.bit[k]) & ((1u << r.len[k]) - 1)) << r.pos[k];
  return i;
}

// What the gather kernel computes per destination: the register values (u, v, w) of the one source,
// or, modulo N, of the first of a few sources.
enum MathSource : int32_t {
  kSrcAddConstant = 0,  // every register: x - a
  kSrcSubtract = 1,     // v <- v - u; with `carry`, w ^= (u + v overflows the first register)
  kSrcAdd = 2,          // v <- v + u; with `carry`, w ^= 1
  kSrcCompare = 3,      // w ^= (v < u)
  kSrcMulSubtract = 4,  // w <- w - u v
  kSrcMulAdd = 5,       // w <- w + u v
  kSrcAddMod = 6,       // u <- (u - a) mod N, + N, + 2N, ...; none from N on
  kSrcMulMod = 7        // u <- (u / a) mod N, + N, + 2N, ...; none from N on
};

constexpr int kMathThreadBits = 4;
struct MathGather {
  MathSource source;
  int32_t n_regs;       // 1..3
  int32_t carry;        // the third register takes part in kSrcSubtract / kSrcAdd
  uint32_t width[3];
  uint64_t cmask;       // controls: other indices keep their amplitude
  int32_t moves[3];     // registers whose value changes
  uint64_t changed;     // their index bits
  uint64_t a, N;        // kSrcAddConstant, kSrcAddMod: a; kSrcMulMod: the inverse of a modulo N
  uint64_t magic;       // floor(2^64 / N) (N > 1)
  BitRuns reg[3];
  BitRuns order;        // amplitude counter -> index: the order of the traversal
  // index and register values of counter bits 8..11 (the 16 amplitudes of one thread)
  uint64_t step[kMathThreadBits];
  uint32_t reg_step[kMathThreadBits][3];
};

// Positions in the order of the value's bits.
BitRuns runs_of(const std::vector<unsigned> &positions);

// Registers as bit positions, ascending significance.  true: `out` describes the call, whose sources
// are found from the destination.  false: nothing is known about the map (a shared qubit, a width
// or constant outside what the rules below cover), and the general path decides.
bool plan_math_gather(int opcode, int64_t a, int64_t N, const std::vector<std::vector<unsigned>> &regs, uint64_t cmask,
                      unsigned n, bool c64, MathGather *out);

// The same call in place, where every index bit that changes fits one LDS tile (the destinations of a tile
// then have all their sources in it).
struct MathTile {
  uint32_t m;         // tile bits
  uint32_t changed;   // tile bits that change
  uint64_t fixed;     // controls outside the tile: only the indices that have them set are visited
  uint32_t outside;   // index bits of the tile number
  BitRuns tile_id;    // tile number -> index bits
  BitRuns tile;       // tile-local index <-> index bits
  BitRuns local[3];   // register value <-> tile-local index (registers that change)
  // index and register values of tile-local bits 8..11 (the amplitudes of one thread)
  uint64_t step[kMathThreadBits];
  uint32_t reg_step[kMathThreadBits][3];
};
constexpr unsigned kMathTileBits64 = 12, kMathTileBits128 = 11;  // 32 KiB
bool plan_math_tile(const MathGather &G, unsigned n, bool c64, MathTile *out);

// x -> x + a on registers whose qubits ascend or descend in position.  The subtraction that finds the source runs on
// the register's bits where they are: with zeros between them a borrow passes through the gaps.  A descending
// register ascends in the index read backwards.
struct MathAdd {
  int32_t n_regs;
  uint32_t reversed;  // bit r: register r descends
  uint64_t cmask;
  uint64_t mask[3], sub[3];  // the register's bits, and a on them (of the index read backwards where reversed)
};
bool plan_math_add(const MathGather &G, MathAdd *out);

QS_HD inline uint64_t reverse_bits(uint64_t v) {
#ifdef __HIPCC__
  return __builtin_bitreverse64(v);
#else
  uint64_t r = 0;
  for (int b = 0; b < 64; ++b) r |= ((v >> b) & 1) << (63 - b);
  return r;
#endif
}
QS_HD inline uint64_t add_source(const MathAdd &A, uint64_t i) {
  if ((i & A.cmask) != A.cmask) return i;
  uint64_t s = i;
  for (int r = 0; r < 3; ++r) {
    if (r >= A.n_regs) break;
    const bool back = (A.reversed >> r) & 1;
    uint64_t t = back ? reverse_bits(s) : s;
    t = (t & ~A.mask[r]) | (((t & A.mask[r]) - A.sub[r]) & A.mask[r]);
    s = back ? reverse_bits(t) : t;
  }
  return s;
}

// Source values (u, v, w) of one destination under the rule S = G.source; returns false where there is
// no source (modulo N only).
template <int S>
QS_HD inline bool math_source(const MathGather &G, uint64_t &u, uint64_t &v, uint64_t &w) {
  switch (S) {
    case kSrcAddConstant:
      u -= G.a;
      v -= G.a;
      w -= G.a;
      return true;
    case kSrcSubtract:
      v = (v - u) & ((uint64_t(1) << G.width[1]) - 1);
      if (G.carry) w ^= ((u + v) >> G.width[0]) ? 1u : 0u;
      return true;
    case kSrcAdd:
      v += u;
      if (G.carry) w ^= 1u;
      return true;
    case kSrcCompare:
      w ^= v < u ? 1u : 0u;
      return true;
    case kSrcMulSubtract:
      w -= u * v;
      return true;
    case kSrcMulAdd:
      w += u * v;
      return true;
    case kSrcAddMod:
      if (u >= G.N) return false;
      u = u >= G.a ? u - G.a : u + G.N - G.a;
      return true;
    default: {  // kSrcMulMod: u a^-1 mod N, the quotient from the reciprocal (one too small at most)
      if (u >= G.N) return false;
      const uint64_t p = u * G.a;
      const uint64_t q = (uint64_t)(((unsigned __int128)p * G.magic) >> 64);
      uint64_t r = p - q * G.N;
      if (r >= G.N) r -= G.N;
      u = r;
      return true;
    }
  }
}

// The residue rules on registers of at most 16 bits, in 32-bit arithmetic (64-bit products are a dozen
// quarter-rate instructions): the first source of destination u < N, magic = floor(2^32 / N).
template <int S>
QS_HD inline uint32_t residue_source32(uint32_t u, uint32_t a, uint32_t N, uint32_t magic) {
  if (S == kSrcAddMod) return u >= a ? u - a : u + N - a;
  const uint32_t p = u * a;  // below 2^32; the quotient is one or two too small at most
  const uint32_t q = (uint32_t)(((uint64_t)p * magic) >> 32);
  uint32_t r = p - q * N;
  if (r >= N) r -= N;
  if (r >= N) r -= N;
  return r;
}

}  // namespace qs
