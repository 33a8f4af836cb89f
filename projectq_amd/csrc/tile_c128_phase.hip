// Tile passes with phase ops: complex128 states.
#include "tile_plain.hpp"

namespace qs {
namespace dev {

void launch_tile_pass_phase(double2 *psi, uint64_t n_tiles, const TilePass &P, const TileStage *d_stages,
                            const RegOp *d_rops, const TileOp *d_tops, const double2 *d_mats, unsigned grid, size_t lds,
                            hipStream_t s) {
  hipLaunchKernelGGL((k_tile_pass<double, 4, true, false, true>), dim3(grid), dim3(kBlock), lds, s, psi, n_tiles, P,
                     d_stages, d_rops, d_tops, d_mats);
  QS_HIP(hipGetLastError());
}

void prepare_tile_kernels_phase_c128() {
  allow_lds(k_tile_pass<double, 4, true, false, true>, kTileLdsMax<double>);
}

}  // namespace dev
}  // namespace qs
