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
// one loads while the others compute; 256-byte segments, the shortest that stream at the full rate.
// 28 qubits complex64, 40 random strings: 22.4 ms string by string, 3.7 ms from tiles (6 passes), 3.0 ms
// with one kernel arm per kind and the next group's record loaded ahead.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "energy.hpp"

namespace qs {
namespace dev {
namespace {

struct Compensated {
  double s = 0.0, c = 0.0;
  __device__ __forceinline__ void add(double v) {
    const double t = s + v;
    if (fabs(s) >= fabs(v)) c += (s - t) + v;
    else c += (v - t) + s;
    s = t;
  }
};

__device__ __forceinline__ double flip(double v, uint32_t odd) {
  return __longlong_as_double(__double_as_longlong(v) ^ ((unsigned long long)odd << 63));
}

// Sum of a workgroup's compensated pairs, in a fixed order; valid in thread 0.
template <int NT>
__device__ __forceinline__ double workgroup_total(const Compensated &a, double *lds) {
  double v = a.s + a.c;
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) lds[wave] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < NT / 64; ++w) t += lds[w];
  return t;
}

// One group of kind IM: v[j] <- Re or Im of conj(a_j) b_j over the j without bit HB (HB = 0: every j), b_j
// the partner, and one weighted sum per string.
template <typename R, int NJ, int HB, bool IM>
__device__ __forceinline__ void energy_group(const amp_t<R> *__restrict__ tile, const double *__restrict__ ar,
                                             const double *__restrict__ ai, const EnergyGroup &g,
                                             const EnergyString *__restrict__ strings, uint64_t base, Compensated &acc) {
  const uint32_t tid = threadIdx.x;
  const uint32_t lo = tid ^ (g.mask & 255u), mj = g.mask & ~255u;
  double v[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    if (HB && (j & HB)) continue;
    const amp_t<R> b = tile[lo | (((uint32_t)j << 8) ^ mj)];
    const double br = b.x, bi = b.y;
    v[j] = IM ? fma(ar[j], bi, -ai[j] * br) : fma(ar[j], br, ai[j] * bi);
  }
  auto string = [&](const EnergyString &st) {
    const double w = flip(st.w, (uint32_t)__popcll(base & st.z) & 1u);
    const uint32_t zj = st.zloc >> 8;
    double sum = 0.0;
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if (HB && (j & HB)) continue;
      sum = fma(flip(w, (uint32_t)__popc((uint32_t)j & zj) & 1u), v[j], sum);
    }
    acc.add(flip(sum, (uint32_t)__popc(tid & st.zloc) & 1u));
  };
  string(g.head);
#pragma unroll 2
  for (uint32_t s = 0; s < g.more; ++s) string(strings[g.next + s]);
}

template <typename R, int LJ, bool IM>
__device__ __forceinline__ void energy_kind(const amp_t<R> *__restrict__ tile, const double *__restrict__ ar,
                                            const double *__restrict__ ai, const EnergyGroup &g,
                                            const EnergyString *__restrict__ strings, uint64_t base, Compensated &acc) {
  constexpr int NJ = 1 << LJ;
  const uint32_t mj = g.mask >> 8;
  const int hb = mj ? 31 - __clz(mj) : -1;  // uniform
  if (hb < 0) energy_group<R, NJ, 0, IM>(tile, ar, ai, g, strings, base, acc);
  if constexpr (LJ > 0) if (hb == 0) energy_group<R, NJ, 1, IM>(tile, ar, ai, g, strings, base, acc);
  if constexpr (LJ > 1) if (hb == 1) energy_group<R, NJ, 2, IM>(tile, ar, ai, g, strings, base, acc);
  if constexpr (LJ > 2) if (hb == 2) energy_group<R, NJ, 4, IM>(tile, ar, ai, g, strings, base, acc);
  if constexpr (LJ > 3) if (hb == 3) energy_group<R, NJ, 8, IM>(tile, ar, ai, g, strings, base, acc);
}

// LJ = log2 of the amplitudes per thread.  Workgroup b works on pass b / per_pass, on the tiles
// b % per_pass, + per_pass, ...; its partial sum goes to partials[b].
template <typename R, int LJ>
__global__ __launch_bounds__(kEnergyThreads) void k_energy(const amp_t<R> *__restrict__ psi, uint64_t n_amps, uint32_t L,
                                                            uint32_t h, uint64_t n_tiles, uint32_t per_pass,
                                                            const EnergyPass *__restrict__ passes,
                                                            const EnergyGroup *__restrict__ groups,
                                                            const EnergyString *__restrict__ strings,
                                                            double *__restrict__ partials) {
  constexpr int NJ = 1 << LJ;
  __shared__ amp_t<R> tile[256 << LJ];
  __shared__ double sums[kEnergyThreads / 64];
  const uint32_t tid = threadIdx.x;
  const EnergyPass &pass = passes[blockIdx.x / per_pass];
  // offset of tile-local index tid + 256 j within a tile: linear over GF(2)
  uint64_t mine = L >= 8 ? tid : tid & ((1u << L) - 1);
  for (uint32_t b = L; b < 8; ++b)
    if ((tid >> b) & 1) mine ^= pass.gen[b - L];
  uint64_t step[LJ > 0 ? LJ : 1];
#pragma unroll
  for (int b = 0; b < LJ; ++b) step[b] = (uint32_t)(8 + b) < L ? uint64_t(256) << b : pass.gen[8 + b - L];
  Compensated acc;
  for (uint64_t k = blockIdx.x % per_pass; k < n_tiles; k += per_pass) {
    uint64_t base = k << L;
    for (uint32_t b = 0; b < h; ++b) {
      const uint32_t p = pass.pivot[b];
      base = ((base >> p) << (p + 1)) | (base & ((uint64_t(1) << p) - 1));
    }
    double ar[NJ], ai[NJ];
    amp_t<R> a[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      uint64_t o = base ^ mine;
#pragma unroll
      for (int b = 0; b < LJ; ++b)
        if ((j >> b) & 1) o ^= step[b];
      if (LJ > 0 || o < n_amps) {
        a[j] = psi[o];
      } else {  // fewer than 256 amplitudes
        a[j].x = 0;
        a[j].y = 0;
      }
    }
    __syncthreads();  // the previous tile's readers are done
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      tile[tid + 256u * j] = a[j];
      ar[j] = (double)a[j].x;
      ai[j] = (double)a[j].y;
    }
    __syncthreads();
    // the next group's record loads while this one computes
    const EnergyGroup *gp = groups + pass.first_group;
    EnergyGroup cur = *gp;
    for (uint32_t g = 0; g < pass.n_groups; ++g) {
      const EnergyGroup next = *++gp;
      if (cur.kind) energy_kind<R, LJ, true>(tile, ar, ai, cur, strings, base, acc);
      else energy_kind<R, LJ, false>(tile, ar, ai, cur, strings, base, acc);
      cur = next;
    }
  }
  const double total = workgroup_total<kEnergyThreads>(acc, sums);
  if (tid == 0) partials[blockIdx.x] = total;
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
