// The software-pipelined tile pass (complex64, four register bits): definitions included by tile_pf.hip
// and tile_c64_phase.hip.
#pragma once

#define QS_TILE_KERNELS
#include "tile.hpp"

namespace qs {
namespace dev {
namespace {

// Software-pipelined tile pass: while the stages of tile i run out of LDS, the loads of the
// workgroup's next tile are already in flight into registers, so HBM traffic overlaps the in-tile
// arithmetic.  Used when a thread's share of a tile is exactly kStreamChunk 16-byte vectors
// (2^t = kStreamChunk * NT * VN), so all streaming is unguarded straight-line code.  NT = 256
// serves 2^12-amplitude complex64 tiles (32 KiB of LDS, four workgroups per CU), NT = 512 tiles of
// 2^13 (64 KiB, two workgroups per CU): the same per-thread work and the same waves per CU.
template <typename R, int RB, int NT, bool TWO, bool PH = false>
__global__ __launch_bounds__(NT) __attribute__((amdgpu_waves_per_eu(4))) void k_tile_pass_pf(amp_t<R> *__restrict__ psi, uint64_t n_tiles,
                                                         TilePass P, const TileStage *__restrict__ stages,
                                                         const RegOp *__restrict__ rops,
                                                         const TileOp *__restrict__ tops,
                                                         const amp_t<R> *__restrict__ mats) {
  using V = typename Vec16<R>::type;
  constexpr int VN = Vec16<R>::n;
  constexpr uint32_t kStep = NT * VN;
  extern __shared__ __align__(16) unsigned char smem[];
  // the tile starts at LDS address 0 (no static LDS), so tile offsets need no base add;
  // the 2^h segment offsets follow the tile
  amp_t<R> *tile = reinterpret_cast<amp_t<R> *>(smem);
  uint64_t *seg = reinterpret_cast<uint64_t *>(smem + (sizeof(amp_t<R>) << P.t));
  fill_segments<NT>(P, seg);
  uint64_t tix = blockIdx.x;
  if (tix >= n_tiles) return;  // uniform over the workgroup
  const uint32_t t = P.t, L = P.L;
  const uint32_t segmask = (1u << L) - 1;
  const uint32_t l0 = threadIdx.x * VN;
  const uint32_t s0 = lds_address(tile) + slot_bytes<R>(l0);  // l0 shares no bit with j * kStep
  // the store reads the computed tile through the relabelling of P.sperm (identity: s0, j * kStep)
  const uint32_t ss0 = lds_address(tile) + slot_bytes<R>(store_source(l0, P));
  const uint32_t spair = slot_bytes<R>(store_source(1, P));
  // j * kStep for j < 8 spans three bits: its source is the XOR of theirs
  const uint32_t sbit0 = slot_bytes<R>(store_source(kStep, P)), sbit1 = slot_bytes<R>(store_source(2 * kStep, P)),
                 sbit2 = slot_bytes<R>(store_source(4 * kStep, P));
  static_assert(kStreamChunk == 8, "three step bits");
  // Each turn of the loop runs the stages of the resident tile and stores it, then moves the
  // registers holding the next tile (loaded during those stages) into LDS and starts loading the
  // tile after.  At that wait only the older loads must be complete, not the stores just issued.
  uint64_t base = tile_base(tix, P);
  V v[kStreamChunk];
#pragma unroll
  for (int j = 0; j < kStreamChunk; ++j) {
    const uint32_t l = l0 + j * kStep;
    v[j] = stream_load(reinterpret_cast<const V *>(psi + (base | seg[l >> L] | (l & segmask))));
  }
#pragma unroll
  for (int j = 0; j < kStreamChunk; ++j) tile_put16<R>(s0 ^ slot_bytes<R>(j * kStep), v[j]);
  __syncthreads();
  uint64_t next = tix + gridDim.x;
  uint64_t nbase = tile_base(next < n_tiles ? next : tix, P);
  auto prefetch = [&](uint64_t from) {
    // the segment offsets are re-read from LDS for every tile rather than kept live across the
    // stages (the empty asm keeps the compiler from hoisting them into registers)
    uint32_t lq = l0;
    asm volatile("" : "+v"(lq));
#pragma unroll
    for (int j = 0; j < kStreamChunk; ++j) {
      const uint32_t l = lq + j * kStep;
      v[j] = stream_load(reinterpret_cast<const V *>(psi + (from | seg[l >> L] | (l & segmask))));
    }
  };
  if (next < n_tiles) prefetch(nbase);
  while (true) {
    run_stages<R, RB, 2, NT, TWO, PH>(tile, t, base, P.n_stages, stages, rops, tops, mats);
    uint32_t ls = l0;
    asm volatile("" : "+v"(ls));
#pragma unroll
    for (int j = 0; j < kStreamChunk; ++j) {
      const uint32_t l = ls + j * kStep;
      stream_store(reinterpret_cast<V *>(psi + (base | seg[l >> L] | (l & segmask))),
                   tile_get16p<R>(ss0 ^ ((j & 1) ? sbit0 : 0u) ^ ((j & 2) ? sbit1 : 0u) ^ ((j & 4) ? sbit2 : 0u), spair));
    }
    __syncthreads();
    if (next >= n_tiles) break;  // uniform over the workgroup
#pragma unroll
    for (int j = 0; j < kStreamChunk; ++j) tile_put16<R>(s0 ^ slot_bytes<R>(j * kStep), v[j]);
    __syncthreads();
    base = nbase;
    const uint64_t cur = next;
    next = cur + gridDim.x;
    nbase = tile_base(next < n_tiles ? next : cur, P);
    if (next < n_tiles) prefetch(nbase);
  }
}

}  // namespace

}  // namespace dev
}  // namespace qs
