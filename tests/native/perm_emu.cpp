// Test-only CPU run of the layout permutation: the planned tile (plan_permutation) replayed with the
// kernel's index rules (k_permute_tiles), every index checked against its buffer.
#include "planner.hpp"

// dst[i'] <- src[i] for 2^n indices; returns 0, or which check failed
extern "C" int perm_run(unsigned n, const uint32_t *to, int c64, const uint32_t *src, uint32_t *dst, uint32_t *conflicts) {
  const qs::PermTile P = qs::plan_permutation(std::vector<unsigned>(to, to + n), c64 != 0);
  const uint32_t most = c64 ? 12 : 11, vn = c64 ? 2 : 1, v = c64 ? 1 : 0, w = c64 ? 5 : 4;
  if (P.m != (n < most ? n : most) || P.m + P.n_outer != n) return 1;
  if (P.src_pos[0] != 0 || P.dst_pos[0] != 0 || (vn == 2 && P.slot_src[0] != 1)) return 2;
  const uint32_t size = 1u << P.m;
  auto slot = [&](uint32_t x, const uint16_t *bits) {
    uint32_t s = 0;
    for (uint32_t r = 0; r < P.m; ++r)
      if ((x >> r) & 1) s ^= bits[r];
    return s;
  };
  auto index = [&](uint32_t x, const uint8_t *pos) {
    uint64_t i = 0;
    for (uint32_t r = 0; r < P.m; ++r) i |= uint64_t((x >> r) & 1) << pos[r];
    return i;
  };
  std::vector<uint32_t> tile(size);
  for (uint64_t id = 0; id < (uint64_t(1) << P.n_outer); ++id) {
    uint64_t sb = 0, db = 0;
    for (uint32_t i = 0; i < P.n_outer; ++i) {
      sb |= ((id >> i) & 1) << P.outer_src[i];
      db |= ((id >> i) & 1) << P.outer_dst[i];
    }
    std::vector<char> taken(size, 0);
    for (uint32_t x = 0; x < size; ++x) {
      const uint32_t s = slot(x, P.slot_src);
      if (s >= size || taken[s]) return 3;
      taken[s] = 1;
      const uint64_t i = sb | index(x, P.src_pos);
      if (i >> n) return 4;
      tile[s] = src[i];
    }
    for (uint32_t y = 0; y < size; ++y) {
      const uint32_t s = slot(y, P.slot_dst);
      const uint64_t i = db | index(y, P.dst_pos);
      if (s >= size || (i >> n)) return 5;
      dst[i] = tile[s];
    }
  }
  // accesses of 2^w lanes that meet in a bank, on the write and the read side
  for (int side = 0; side < 2; ++side) {
    std::vector<uint32_t> lanes(1u << w, 0);
    for (uint32_t l = 0; l < (1u << w) && (l << v) < size; ++l)
      ++lanes[slot(l << v, side ? P.slot_dst : P.slot_src) & ((1u << w) - 1)];
    conflicts[side] = 0;
    for (uint32_t c : lanes) conflicts[side] = c > conflicts[side] ? c : conflicts[side];
  }
  return 0;
}
