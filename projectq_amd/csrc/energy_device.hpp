// Device code of the expectation-value kernels: one state (energy.hip) and batches of circuits
// (batch_energy.hip).
#pragma once

#include <hip/hip_runtime.h>

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


// One tile (LJ = log2 of the amplitudes per thread): its amplitudes into registers and LDS, then every
// group of the pass.  `mine` and `step` are the offsets of a thread's first amplitude and of j's bits.
template <typename R, int LJ>
__device__ __forceinline__ void energy_tile(const amp_t<R> *__restrict__ psi, uint64_t n_amps, uint64_t base, uint64_t mine,
                                            const uint64_t *step, const EnergyGroup *__restrict__ groups, uint32_t n_groups,
                                            const EnergyString *__restrict__ strings, amp_t<R> *__restrict__ tile,
                                            Compensated &acc) {
  constexpr int NJ = 1 << LJ;
  const uint32_t tid = threadIdx.x;
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
  EnergyGroup cur = *groups;
  for (uint32_t g = 0; g < n_groups; ++g) {
    const EnergyGroup next = *++groups;
    if (cur.kind) energy_kind<R, LJ, true>(tile, ar, ai, cur, strings, base, acc);
    else energy_kind<R, LJ, false>(tile, ar, ai, cur, strings, base, acc);
    cur = next;
  }
}

// offsets of tile-local index tid + 256 j within a tile of `pass`: linear over GF(2)
template <int LJ>
__device__ __forceinline__ uint64_t energy_offsets(const EnergyPass &pass, uint32_t L, uint64_t *step) {
  const uint32_t tid = threadIdx.x;
  uint64_t mine = L >= 8 ? tid : tid & ((1u << L) - 1);
  for (uint32_t b = L; b < 8; ++b)
    if ((tid >> b) & 1) mine ^= pass.gen[b - L];
#pragma unroll
  for (int b = 0; b < LJ; ++b) step[b] = (uint32_t)(8 + b) < L ? uint64_t(256) << b : pass.gen[8 + b - L];
  return mine;
}
// first index of tile k
__device__ __forceinline__ uint64_t energy_base(const EnergyPass &pass, uint32_t L, uint32_t h, uint64_t k) {
  uint64_t base = k << L;
  for (uint32_t b = 0; b < h; ++b) {
    const uint32_t p = pass.pivot[b];
    base = ((base >> p) << (p + 1)) | (base & ((uint64_t(1) << p) - 1));
  }
  return base;
}

}  // namespace
}  // namespace dev
}  // namespace qs
