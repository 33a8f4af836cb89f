// Expectation value of a sum of Pauli strings on one state, many strings from one LDS tile.
//
// A string pairs the amplitude i with i ^ x, so string by string the state is read from memory (or
// from the caches) once per string.  Here a tile is the span of a few x masks (plan_energy): every
// string whose x lies in that span finds both members of its pairs in LDS, and the state is read
// once per 7 or more strings.  The two members contribute complex-conjugate terms, so each pair is
// visited once, from the member with the highest tile-local bit of x clear, with twice the weight.
//
// A thread holds 2^(t-8) amplitudes, tile-local indices tid + 256 j, and reads their partners from
// LDS at index ^ mask: an XOR of the lane bits permutes an aligned block, so the accesses are free of
// bank conflicts.  The sign (-1)^{popcount(i & z)} splits into a uniform part (tile base and j, folded
// into the scalar weight) and the thread's own parity, applied once per string and tile.  Products
// and sums are FP64 whatever the state precision; per thread the strings' sums are Neumaier
// compensated over strings and tiles.
//
// What bounds it: FP64 issue (a conversion, two FMAs of the pair and one per string) while a few
// passes of 5 TB/s reads hide behind it.  Tile: 32 KiB, so four or five workgroups share a CU and
// one loads while the others compute; segments of 256 bytes, or 128 where that saves a read of the state.
// 28 qubits complex64, 40 random strings: 22.4 ms string by string, 3.7 ms from tiles (6 passes), 3.0 ms
// with one kernel arm per kind and the next group's record loaded ahead, 2.9 ms in 5 passes.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "energy_device.hpp"

namespace qs {
namespace dev {
namespace {

// LJ = log2 of the amplitudes per thread.  Workgroup b works on pass b / per_pass, on the tiles
// b % per_pass, + per_pass, ...; its partial sum goes to partials[b].
template <typename R, int LJ>
__global__ __launch_bounds__(kEnergyThreads) void k_energy(const amp_t<R> *__restrict__ psi, uint64_t n_amps, uint32_t L,
                                                            uint32_t h, uint64_t n_tiles, uint32_t per_pass,
                                                            const EnergyPass *__restrict__ passes,
                                                            const EnergyGroup *__restrict__ groups,
                                                            const EnergyString *__restrict__ strings,
                                                            double *__restrict__ partials) {
  __shared__ amp_t<R> tile[256 << LJ];
  __shared__ double sums[kEnergyThreads / 64];
  const EnergyPass &pass = passes[blockIdx.x / per_pass];
  uint64_t step[LJ > 0 ? LJ : 1];
  const uint64_t mine = energy_offsets<LJ>(pass, L, step);
  Compensated acc;
  for (uint64_t k = blockIdx.x % per_pass; k < n_tiles; k += per_pass)
    energy_tile<R, LJ>(psi, n_amps, energy_base(pass, L, h, k), mine, step, groups + pass.first_group, pass.n_groups, strings,
                       tile, acc);
  const double total = workgroup_total<kEnergyThreads>(acc, sums);
  if (threadIdx.x == 0) partials[blockIdx.x] = total;
}

// One workgroup: *out <- sum of the partials, in a fixed order, compensated.
__global__ __launch_bounds__(1024) void k_energy_finish(const double *__restrict__ partials, uint32_t n,
                                                        double *__restrict__ out) {
  __shared__ double sums[1024 / 64];
  Compensated acc;
  for (uint32_t i = threadIdx.x; i < n; i += 1024) acc.add(partials[i]);
  const double total = workgroup_total<1024>(acc, sums);
  if (threadIdx.x == 0) *out = total;
}

}  // namespace

template <typename R>
void energy(const amp_t<R> *psi, unsigned n, const EnergyPlan &plan, const char *d_records, const EnergyRecords &rec,
            double *partials, double *out, hipStream_t s) {
  const uint64_t tiles = n > plan.t ? uint64_t(1) << (n - plan.t) : 1;
  // a workgroup takes one pass over a share of the tiles
  const uint32_t per_pass =
      (uint32_t)std::min<uint64_t>(tiles, std::max<uint32_t>(1, kEnergyPartials / std::max(1u, plan.n_passes)));
  const uint32_t blocks = per_pass * plan.n_passes;
  auto go = [&](auto lj) {
    hipLaunchKernelGGL((k_energy<R, decltype(lj)::value>), dim3(blocks), dim3(kEnergyThreads), 0, s, psi,
                       uint64_t(1) << n, plan.L, plan.h, tiles, per_pass, (const EnergyPass *)d_records,
                       (const EnergyGroup *)(d_records + rec.groups), (const EnergyString *)(d_records + rec.strings),
                       partials);
  };
  if (blocks > 0) {
    switch (plan.t) {
      case 8: go(std::integral_constant<int, 0>{}); break;
      case 9: go(std::integral_constant<int, 1>{}); break;
      case 10: go(std::integral_constant<int, 2>{}); break;
      case 11: go(std::integral_constant<int, 3>{}); break;
      default:
        if constexpr (sizeof(R) == 4) go(std::integral_constant<int, 4>{});
        else throw ValueError("energy: bad tile");
        break;
    }
    QS_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(k_energy_finish, dim3(1), dim3(1024), 0, s, partials, blocks, out);
  QS_HIP(hipGetLastError());
}

template void energy<float>(const float2 *, unsigned, const EnergyPlan &, const char *, const EnergyRecords &, double *,
                            double *, hipStream_t);
template void energy<double>(const double2 *, unsigned, const EnergyPlan &, const char *, const EnergyRecords &, double *,
                             double *, hipStream_t);

}  // namespace dev
}  // namespace qs
