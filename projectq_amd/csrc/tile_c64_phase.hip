// Tile passes with phase ops: complex64 states.
#include "tile_pf.hpp"

namespace qs {
namespace dev {

void launch_tile_pass_phase(float2 *psi, uint64_t n_tiles, const TilePass &P, const TileStage *d_stages,
                            const RegOp *d_rops, const TileOp *d_tops, const float2 *d_mats, unsigned grid, size_t lds,
                            hipStream_t s) {
  const int threads = P.t == 13 ? 2 * kBlock : kBlock;  // full tiles of complex64: 2^12 or 2^13 amplitudes
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), lds, s, psi, n_tiles, P, d_stages, d_rops, d_tops, d_mats);
    QS_HIP(hipGetLastError());
  };
  if (P.t == 13) go(k_tile_pass_pf<float, 4, 2 * kBlock, false, true>);
  else go(k_tile_pass_pf<float, 4, kBlock, false, true>);
}

void prepare_tile_kernels_phase_c64() {
  allow_lds(k_tile_pass_pf<float, 4, kBlock, false, true>, kTileLdsMax<float>);
  allow_lds(k_tile_pass_pf<float, 4, 2 * kBlock, false, true>, kTileLdsMax<float>);
}

}  // namespace dev
}  // namespace qs
