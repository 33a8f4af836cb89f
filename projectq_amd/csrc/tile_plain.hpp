// Plain and batched tile kernels of one (state precision, register bits) combination: definitions
// included by the tile_c*_rb*.hip files.
#pragma once

#define QS_TILE_KERNELS
#include "tile.hpp"

namespace qs {
namespace dev {
namespace {

// TWO = false: the instantiation for passes without 2-qubit register ops (see reg_op)
// PH = true: the one for passes with phase ops
template <typename R, int RB, bool FULL, bool TWO = true, bool PH = false>
__global__ __launch_bounds__(kBlock) void k_tile_pass(amp_t<R> *__restrict__ psi, uint64_t n_tiles,
                                                      TilePass P, const TileStage *__restrict__ stages,
                                                      const RegOp *__restrict__ rops,
                                                      const TileOp *__restrict__ tops,
                                                      const amp_t<R> *__restrict__ mats) {
  extern __shared__ __align__(16) unsigned char smem[];
  // the tile starts at LDS address 0 (no static LDS), so tile offsets need no base add;
  // the 2^h segment offsets follow the tile
  amp_t<R> *tile = reinterpret_cast<amp_t<R> *>(smem);
  uint64_t *seg = reinterpret_cast<uint64_t *>(smem + (sizeof(amp_t<R>) << P.t));
  fill_segments(P, seg);
  for (uint64_t tix = blockIdx.x; tix < n_tiles; tix += gridDim.x)
    tile_body<R, RB, FULL, TWO, PH>(psi, tix, P, seg, tile, stages, rops, tops, mats);
}

// Many circuits at once: workgroup b runs tile (b - job.first_block) of job block_job[b]; every
// job is one pass of one circuit whose state starts at psi + job.state_off.
template <typename R, int RB, bool TWO = true>
__global__ __launch_bounds__(kBlock) void k_batch_tile_pass(amp_t<R> *__restrict__ psi,
                                                            const BatchJob *__restrict__ jobs,
                                                            const uint32_t *__restrict__ block_job,
                                                            const TileStage *__restrict__ stages,
                                                            const RegOp *__restrict__ rops,
                                                            const TileOp *__restrict__ tops,
                                                            const amp_t<R> *__restrict__ mats) {
  extern __shared__ __align__(16) unsigned char smem[];
  const BatchJob *job = jobs + block_job[blockIdx.x];
  const TilePass &P = job->P;
  amp_t<R> *tile = reinterpret_cast<amp_t<R> *>(smem);
  uint64_t *seg = reinterpret_cast<uint64_t *>(smem + (sizeof(amp_t<R>) << P.t));
  fill_segments(P, seg);
  tile_body<R, RB, false, TWO>(psi + job->state_off, blockIdx.x - job->first_block, P, seg, tile, stages + job->stage_off,
                   rops + job->rop_off, tops + job->top_off, mats + job->mat_off);
}
}  // namespace

template <typename R, int RB>
void launch_tile_pass(amp_t<R> *psi, uint64_t n_tiles, const TilePass &P, const TileStage *d_stages,
                      const RegOp *d_rops, const TileOp *d_tops, const amp_t<R> *d_mats, TileForms forms,
                      hipStream_t s) {
  prepare_tile_kernels();
  const size_t lds = (sizeof(amp_t<R>) << P.t) + (sizeof(uint64_t) << P.h);
  // workgroups per launch: each loops over n_tiles / grid tiles.  About 16 tiles per workgroup
  // measured best at 2^20 tiles (18.5 ms per pass against 19.1 ms at 128 per workgroup and 19.8
  // ms at one), never fewer than 8192 workgroups; PROJECTQ_AMD_TILE_GRID fixes the count.
  static const uint64_t cap = [] {
    const char *e = std::getenv("PROJECTQ_AMD_TILE_GRID");
    return e ? std::max<uint64_t>(1, std::strtoull(e, nullptr, 10)) : uint64_t(0);
  }();
  const uint64_t grid = std::min<uint64_t>(n_tiles, cap ? cap : std::max<uint64_t>(8192, n_tiles / 16));
  const uint64_t chunk = uint64_t(kStreamChunk) * kBlock * Vec16<R>::n;  // amplitudes streamed per round
  const uint64_t tsize = uint64_t(1) << P.t;
  const bool two_qubit_ops = forms == kFormsAll;
  if (forms == kFormsPhases) {
    if (RB != 4 || tsize % chunk != 0) throw ValueError("tile pass: phase ops need full tiles and 4 register bits");
    launch_tile_pass_phase(psi, n_tiles, P, d_stages, d_rops, d_tops, d_mats, (unsigned)grid, lds, s);
    return;
  }
  if constexpr (RB == 4 && sizeof(R) == 4) {  // the only instantiations of the pipelined kernel
    if (launch_tile_pass_pf(psi, n_tiles, P, d_stages, d_rops, d_tops, d_mats, two_qubit_ops, (unsigned)grid, lds, s))
      return;
  }
  if constexpr (RB == 4) {  // passes without 2-qubit register ops: the kernel without those forms
    if (tsize % chunk == 0 && !two_qubit_ops) {
      hipLaunchKernelGGL((k_tile_pass<R, RB, true, false>), dim3((unsigned)grid), dim3(kBlock), lds, s, psi,
                         n_tiles, P, d_stages, d_rops, d_tops, d_mats);
      QS_HIP(hipGetLastError());
      return;
    }
  }
  if (tsize % chunk == 0)
    hipLaunchKernelGGL((k_tile_pass<R, RB, true>), dim3((unsigned)grid), dim3(kBlock), lds, s, psi, n_tiles, P,
                       d_stages, d_rops, d_tops, d_mats);
  else
    hipLaunchKernelGGL((k_tile_pass<R, RB, false>), dim3((unsigned)grid), dim3(kBlock), lds, s, psi, n_tiles, P,
                       d_stages, d_rops, d_tops, d_mats);
  QS_HIP(hipGetLastError());
}

template <typename R, int RB>
void launch_batch_tile_pass(amp_t<R> *psi, const BatchJob *jobs, const uint32_t *block_job, uint32_t n_blocks,
                            uint32_t max_t, const TileStage *stages, const RegOp *rops, const TileOp *tops,
                            const amp_t<R> *mats, bool two_qubit_ops, hipStream_t s) {
  prepare_tile_kernels();
  const size_t lds = (sizeof(amp_t<R>) << max_t) + (sizeof(uint64_t) << kTileMaxHigh);
  bool done = false;
  if constexpr (RB == 4) {
    if (!two_qubit_ops) {
      hipLaunchKernelGGL((k_batch_tile_pass<R, RB, false>), dim3(n_blocks), dim3(kBlock), lds, s, psi, jobs,
                         block_job, stages, rops, tops, mats);
      done = true;
    }
  }
  if (!done)
    hipLaunchKernelGGL((k_batch_tile_pass<R, RB>), dim3(n_blocks), dim3(kBlock), lds, s, psi, jobs, block_job, stages,
                       rops, tops, mats);
  QS_HIP(hipGetLastError());
}

template <typename R, int RB>
void prepare_tile_kernels_of() {
  allow_lds(k_tile_pass<R, RB, true>, kTileLdsMax<R>);
  allow_lds(k_tile_pass<R, RB, false>, kTileLdsMax<R>);
  allow_lds(k_batch_tile_pass<R, RB>, kTileLdsMax<R>);
  if constexpr (RB == 4) {
    allow_lds(k_tile_pass<R, RB, true, false>, kTileLdsMax<R>);
    allow_lds(k_batch_tile_pass<R, RB, false>, kTileLdsMax<R>);
  }
}

#define QS_INSTANTIATE_TILE(R, RB)                                                                              \
  template void launch_tile_pass<R, RB>(amp_t<R> *, uint64_t, const TilePass &, const TileStage *,             \
                                        const RegOp *, const TileOp *, const amp_t<R> *, TileForms, hipStream_t); \
  template void launch_batch_tile_pass<R, RB>(amp_t<R> *, const BatchJob *, const uint32_t *, uint32_t,        \
                                              uint32_t, const TileStage *, const RegOp *, const TileOp *,      \
                                              const amp_t<R> *, bool, hipStream_t);                            \
  template void prepare_tile_kernels_of<R, RB>();

}  // namespace dev
}  // namespace qs
