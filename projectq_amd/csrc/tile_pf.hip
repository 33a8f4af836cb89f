// The software-pipelined tile pass (complex64, four register bits).
#include "tile_pf.hpp"

namespace qs {
namespace dev {

bool launch_tile_pass_pf(float2 *psi, uint64_t n_tiles, const TilePass &P, const TileStage *d_stages,
                         const RegOp *d_rops, const TileOp *d_tops, const float2 *d_mats, bool two_qubit_ops,
                         unsigned grid, size_t lds, hipStream_t s) {
  // the pipelined kernel is the default where it applies; PROJECTQ_AMD_TILE_PREFETCH=0 turns it off
  static const bool prefetch = [] {
    const char *e = std::getenv("PROJECTQ_AMD_TILE_PREFETCH");
    return !e || std::atoi(e) != 0;
  }();
  const uint64_t chunk = uint64_t(kStreamChunk) * kBlock * Vec16<float>::n;  // amplitudes streamed per round
  const uint64_t tsize = uint64_t(1) << P.t;
  if (!prefetch || (tsize != chunk && tsize != 2 * chunk)) return false;
  auto go = [&](auto kernel, int threads) {
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(threads), lds, s, psi, n_tiles, P, d_stages, d_rops, d_tops, d_mats);
    QS_HIP(hipGetLastError());
  };
  if (tsize == chunk) go(two_qubit_ops ? k_tile_pass_pf<float, 4, kBlock, true> : k_tile_pass_pf<float, 4, kBlock, false>, kBlock);
  else go(two_qubit_ops ? k_tile_pass_pf<float, 4, 2 * kBlock, true> : k_tile_pass_pf<float, 4, 2 * kBlock, false>, 2 * kBlock);
  return true;
}

void prepare_tile_kernels_pf() {
  allow_lds(k_tile_pass_pf<float, 4, kBlock, true>, kTileLdsMax<float>);
  allow_lds(k_tile_pass_pf<float, 4, 2 * kBlock, true>, kTileLdsMax<float>);
  allow_lds(k_tile_pass_pf<float, 4, kBlock, false>, kTileLdsMax<float>);
  allow_lds(k_tile_pass_pf<float, 4, 2 * kBlock, false>, kTileLdsMax<float>);
}

}  // namespace dev
}  // namespace qs
