// Energies of a batch of circuits: <psi_c| H_c |psi_c> for every circuit c, H_c a sum of Pauli strings,
// FP64 sums whatever the state precision.
//
// The strings of a circuit are evaluated from LDS tiles as on one state (energy.hip): both members of a
// pair come from LDS, so a state is read once per 7 strings instead of fetching every partner of every
// string from the caches.  The host orders the workgroups so that all workgroups of one circuit run on
// one XCD (workgroup w runs on XCD w mod 8): the passes of a circuit of up to 4 MiB after the first read
// its state from that XCD's L2.
//
// What bounds it: FP64 issue and LDS reads.  160 circuits of 10 to 18 qubits, 100 strings each, complex64:
// 0.62 ms with partners from the caches, 0.30 ms now (whole run 1.20 -> 0.78 ms).  Tiles kept in LDS as FP64,
// which saves the conversions, fit half the amplitudes and measured slower (0.90 ms).
// A launch per tile size costs 1.5 us each, most of what a batch of short operators takes (64 circuits of 8 to 12
// qubits, one string each: run 61 us with one launch, 68 with five): sizes with too few workgroups to fill the chip
// share one launch (56 us).
#include "energy_device.hpp"

#include <type_traits>

namespace qs {
namespace dev {
namespace {

template <typename R, int LJ>
__device__ __forceinline__ void batch_tiles(const amp_t<R> *__restrict__ psi, const BatchEnergyPass &bp, const BatchEnergyBlock &eb,
                                            const EnergyGroup *__restrict__ groups, const EnergyString *__restrict__ strings,
                                            amp_t<R> *__restrict__ tile, Compensated &acc) {
  uint64_t step[LJ > 0 ? LJ : 1];
  const uint64_t mine = energy_offsets<LJ>(bp.pass, bp.L, step);
  for (uint32_t k = eb.tile; k < eb.tile + eb.tiles; ++k)
    energy_tile<R, LJ>(psi + bp.state_off, bp.n_amps, energy_base(bp.pass, bp.L, bp.h, k), mine, step,
                       groups + bp.pass.first_group, bp.pass.n_groups, strings, tile, acc);
}

template <typename R>
constexpr int kMaxTile = sizeof(R) == 4 ? 12 : 11;

// LJ >= 0: every pass has tiles of 2^(8 + LJ); -1: each workgroup looks up its own
template <typename R, int LJ>
__global__ __launch_bounds__(kEnergyThreads) void k_batch_energy(const amp_t<R> *__restrict__ psi,
                                                                 const BatchEnergyPass *__restrict__ passes,
                                                                 const BatchEnergyBlock *__restrict__ blocks,
                                                                 const EnergyGroup *__restrict__ groups,
                                                                 const EnergyString *__restrict__ strings,
                                                                 double *__restrict__ partials) {
  __shared__ amp_t<R> tile[LJ < 0 ? 1 << kMaxTile<R> : 256 << (LJ < 0 ? 0 : LJ)];
  __shared__ double sums[kEnergyThreads / 64];
  const BatchEnergyBlock eb = blocks[blockIdx.x];
  if (eb.pass == kNoPass) return;  // uniform over the workgroup
  const BatchEnergyPass &bp = passes[eb.pass];
  Compensated acc;
  if constexpr (LJ >= 0) {
    batch_tiles<R, LJ>(psi, bp, eb, groups, strings, tile, acc);
  } else {
    switch (bp.L + bp.h) {
      case 8: batch_tiles<R, 0>(psi, bp, eb, groups, strings, tile, acc); break;
      case 9: batch_tiles<R, 1>(psi, bp, eb, groups, strings, tile, acc); break;
      case 10: batch_tiles<R, 2>(psi, bp, eb, groups, strings, tile, acc); break;
      case 11: batch_tiles<R, 3>(psi, bp, eb, groups, strings, tile, acc); break;
      default:
        if constexpr (kMaxTile<R> == 12) batch_tiles<R, 4>(psi, bp, eb, groups, strings, tile, acc);
        break;
    }
  }
  const double total = workgroup_total<kEnergyThreads>(acc, sums);
  if (threadIdx.x == 0) partials[eb.slot] = total;
}

// one wave per circuit
__global__ __launch_bounds__(64) void k_batch_energy_finish(const uint32_t *__restrict__ first,
                                                            const double *__restrict__ partials, double *energies) {
  double v = 0.0;
  for (uint32_t b = first[blockIdx.x] + threadIdx.x; b < first[blockIdx.x + 1]; b += 64) v += partials[b];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if (threadIdx.x == 0) energies[blockIdx.x] = v;
}

}  // namespace

template <typename R>
void batch_energy(const amp_t<R> *psi, uint32_t t, const BatchEnergyPass *passes, const BatchEnergyBlock *blocks,
                  uint32_t n_blocks, const EnergyGroup *groups, const EnergyString *strings, double *partials, hipStream_t s) {
  if (n_blocks == 0) return;
  auto go = [&](auto lj) {
    hipLaunchKernelGGL((k_batch_energy<R, decltype(lj)::value>), dim3(n_blocks), dim3(kEnergyThreads), 0, s, psi, passes,
                       blocks, groups, strings, partials);
  };
  if (t != kMixedTiles && (t < 8 || t > (uint32_t)kMaxTile<R>)) throw ValueError("batch energy: bad tile");
  switch (t) {
    case kMixedTiles: go(std::integral_constant<int, -1>{}); break;
    case 8: go(std::integral_constant<int, 0>{}); break;
    case 9: go(std::integral_constant<int, 1>{}); break;
    case 10: go(std::integral_constant<int, 2>{}); break;
    case 11: go(std::integral_constant<int, 3>{}); break;
    default:
      if constexpr (kMaxTile<R> == 12) go(std::integral_constant<int, 4>{});
      break;
  }
  QS_HIP(hipGetLastError());
}

void batch_energy_finish(const uint32_t *first, int n_circuits, const double *partials, double *energies, hipStream_t s) {
  hipLaunchKernelGGL(k_batch_energy_finish, dim3(n_circuits), dim3(64), 0, s, first, partials, energies);
  QS_HIP(hipGetLastError());
}

template void batch_energy<float>(const float2 *, uint32_t, const BatchEnergyPass *, const BatchEnergyBlock *, uint32_t,
                                  const EnergyGroup *, const EnergyString *, double *, hipStream_t);
template void batch_energy<double>(const double2 *, uint32_t, const BatchEnergyPass *, const BatchEnergyBlock *, uint32_t,
                                   const EnergyGroup *, const EnergyString *, double *, hipStream_t);

}  // namespace dev
}  // namespace qs
