// Measurement on the device: the pick of the reference's serial scan (simulator.hpp:145-186), the
// projection and the renormalisation, with one wait of the host (for the outcome) per measurement.
//
// All(Measure) measures qubit by qubit, and each measurement halves what the next one reads, so
// most of them are short and their cost was latency: three host round trips and three copies each.
// 27 qubits complex64, 8 probabilities and All(Measure): 22.3 and 5.7 ms; measuring and
// freeing 10 qubits with the rest of a variational step: 1.93 and 1.22 ms.
// Large subspaces are read once for the chunk sums (split by the measured bit, so that the norm of
// the outcome needs no second read) and written once by the collapse, which does not load what it
// clears; up to 4096 amplitudes one workgroup does everything.
// What is left between the large reads is latency, so loads go out in batches before their first use, the
// amplitudes of a subspace are found by runs of free bits (after k measured qubits: one run, not k
// fixed bits to insert), and chunks are short enough for a thousand workgroups.  One pick took 25 us, the
// chunk sums of 2^19 amplitudes 28 us and a measurement of 4096 amplitudes 112 us; now
// 13, 9 and 20 us (27 qubits complex64, 8 probabilities and All(Measure): 5.74 -> 5.32 ms).
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"
#include "measure.hpp"

namespace qs {
namespace dev {
namespace {

// index of the subspace's amplitude c
__device__ __forceinline__ uint64_t index_of(uint64_t c, const MeasureArgs &a) { return scatter_bits(c, a.free) | a.sval; }
template <typename A>
__device__ __forceinline__ double norm2(const A &a) {
  const double x = a.x, y = a.y;
  return fma(x, x, y * y);
}

// The large kernels visit spans of kBlock * kBatch compact indices, a thread those of its own number plus
// k * kBlock.  The index is linear in the counter's bits: a thread's part once, a uniform part per span and k, one
// OR per amplitude.  With a loop over the runs of free bits per amplitude the chunk sums of 28 qubits complex64 took
// 0.64 ms, now 0.56.
constexpr int kBatch = 8;
constexpr uint64_t kSpan = (uint64_t)kBlock * kBatch;
struct SpanSteps {
  uint64_t of[kBatch];
  __device__ __forceinline__ explicit SpanSteps(const BitRuns &free) {
#pragma unroll
    for (int k = 0; k < kBatch; ++k) of[k] = scatter_bits((uint64_t)k * kBlock, free);
  }
};

// Sum over a workgroup of NT threads, valid in every thread.
template <int NT>
__device__ __forceinline__ double sum_all(double v, double *lds) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, 64);
  if ((threadIdx.x & 63) == 0) lds[threadIdx.x >> 6] = v;
  __syncthreads();
  double t = 0.0;
  for (int w = 0; w < NT / 64; ++w) t += lds[w];
  __syncthreads();
  return t;
}
// Exclusive prefix sum in thread order; *total is the sum.
template <int NT>
__device__ __forceinline__ double prefix(double v, double *lds, double *total) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double incl = v;
  for (int off = 1; off < 64; off <<= 1) {
    const double o = __shfl_up(incl, off, 64);
    if (lane >= off) incl += o;
  }
  if (lane == 63) lds[wave] = incl;
  __syncthreads();
  double before = 0.0, all = 0.0;
  for (int w = 0; w < NT / 64; ++w) {
    if (w < wave) before += lds[w];
    all += lds[w];
  }
  __syncthreads();
  *total = all;
  const double excl = __shfl_up(incl, 1, 64);
  return before + (lane ? excl : 0.0);
}

// The outcome of a pick contradicts the fixed bits only in the reference's edge cases (a draw of 0 or
// beyond the total): no amplitude is left then.
__device__ __forceinline__ bool contradicts(const MeasureArgs &a, uint64_t pick) {
  return ((pick ^ a.sval) & a.mask & a.zmask) != 0;
}

// The first j in [lo, hi) at which run + value(lo) + ... + value(j) reaches the draw, hi if none; a batch of
// loads at a time.
template <class I, class F>
__device__ __forceinline__ I first_reaching(I lo, I hi, double run, double rnd, F &&value) {
  for (I j = lo; j < hi; j += kBatch) {
    double v[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) v[k] = j + k < hi ? value(j + k) : 0.0;
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      run += v[k];
      if (run >= rnd && j + k < hi) return j + k;
    }
  }
  return hi;
}
template <class I, class F>
__device__ __forceinline__ double sum_range(I lo, I hi, F &&value) {
  double sum = 0.0;
  for (I j = lo; j < hi; j += kBatch) {
    double v[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) v[k] = j + k < hi ? value(j + k) : 0.0;
#pragma unroll
    for (int k = 0; k < kBatch; ++k) sum += v[k];
  }
  return sum;
}

// The in-order scan of `len` compact indices from `start` by a workgroup of NT threads: the first index
// at which base + running norm reaches the draw, ~0 if none.  *total: base + their norm.
template <typename R, int NT>
__device__ __forceinline__ unsigned long long scan_pick(const amp_t<R> *psi, const MeasureArgs &a, uint64_t start,
                                                        uint64_t len, double base, double *lds, unsigned long long *found,
                                                        double *total) {
  const uint64_t per = (len + NT - 1) / NT;
  const uint64_t lo = min<uint64_t>(len, threadIdx.x * per), hi = min<uint64_t>(len, lo + per);
  auto value = [&](uint64_t j) { return norm2(psi[index_of(start + j, a)]); };
  const double mine = sum_range(lo, hi, value);
  if (threadIdx.x == 0) *found = ~0ull;
  double sum;
  const double run = base + prefix<NT>(mine, lds, &sum);  // its barriers order *found before the scan
  *total = base + sum;
  const uint64_t at = first_reaching(lo, hi, run, a.rnd, value);
  if (at < hi) atomicMin(found, (unsigned long long)(start + at));
  __syncthreads();
  return *found;
}

// The subspace in registers: kMeasureSmall / NT consecutive amplitudes per thread, read once.
template <typename R, int NT>
__global__ __launch_bounds__(NT) void k_measure_small(amp_t<R> *__restrict__ psi, MeasureArgs a,
                                                      unsigned long long *__restrict__ host_pick) {
  constexpr int PER = kMeasureSmall / 1024;
  __shared__ double lds[NT / 64];
  __shared__ unsigned long long found;
  uint64_t at[PER];
  amp_t<R> v[PER];
  double norm[PER], mine = 0.0;
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    const uint64_t c = (uint64_t)threadIdx.x * PER + k;
    at[k] = index_of(c, a);
    v[k].x = v[k].y = 0;
    if (c < a.n_sub) v[k] = psi[at[k]];
  }
#pragma unroll
  for (int k = 0; k < PER; ++k) mine += norm[k] = norm2(v[k]);
  uint64_t pick = ~uint64_t(0);
  if (a.rnd > 0.0) {
    if (threadIdx.x == 0) found = ~0ull;
    double total;
    double run = prefix<NT>(mine, lds, &total);  // its barriers order `found` before the scan
    unsigned long long mine_at = ~0ull;
#pragma unroll
    for (int k = PER - 1; k >= 0; --k) {  // the first that reaches the draw is kept
      double r = run;
#pragma unroll
      for (int i = 0; i <= k; ++i) r += norm[i];
      if (r >= a.rnd && (uint64_t)threadIdx.x * PER + k < a.n_sub) mine_at = (uint64_t)threadIdx.x * PER + k;
    }
    if (mine_at != ~0ull) atomicMin(&found, mine_at);
    __syncthreads();
    const unsigned long long c = found;
    if (c != ~0ull) pick = index_of(c, a);
    else pick = total >= a.rnd ? index_of(a.n_sub - 1, a) : a.n_amps - 1;
  }
  if (threadIdx.x == 0) *host_pick = pick;
  const uint64_t val = pick & a.mask;
  double kept = 0.0;
  if (!contradicts(a, pick)) {
#pragma unroll
    for (int k = 0; k < PER; ++k)
      if ((at[k] & a.mask) == val) kept += norm[k];  // 0 beyond the subspace
  }
  const double scale = 1.0 / sqrt(sum_all<NT>(kept, lds));
#pragma unroll
  for (int k = 0; k < PER; ++k) {
    if ((uint64_t)threadIdx.x * PER + k >= a.n_sub) continue;
    amp_t<R> w;
    w.x = w.y = 0;
    if ((at[k] & a.mask) == val) {
      w.x = (R)((double)v[k].x * scale);
      w.y = (R)((double)v[k].y * scale);
    }
    psi[at[k]] = w;
  }
}

// sums[2c], sums[2c + 1] <- norms of chunk c (2^lg compact indices) with the measured bit clear and set
// (of a mask of several bits: all of them set, or not)
template <typename R>
__global__ __launch_bounds__(kBlock) void k_measure_chunks(const amp_t<R> *__restrict__ psi, MeasureArgs a, int lg,
                                                           double *__restrict__ sums) {
  __shared__ double lds[kBlock / 64];
  const uint64_t base = (uint64_t)blockIdx.x << lg, len = uint64_t(1) << lg;
  double clear = 0.0, set = 0.0;
  const SpanSteps step(a.free);
  const uint64_t mine = scatter_bits(threadIdx.x, a.free);
  for (uint64_t first = 0; first < len; first += kSpan) {
    const uint64_t here = index_of(base + first, a) | mine;
    amp_t<R> v[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      v[k].x = v[k].y = 0;
      if (first + k * kBlock < len) v[k] = psi[here | step.of[k]];  // uniform: a chunk is whole rows of kBlock
    }
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      if (((here | step.of[k]) & a.mask) == a.mask) set += norm2(v[k]);
      else clear += norm2(v[k]);
    }
  }
  clear = sum_all<kBlock>(clear, lds);
  set = sum_all<kBlock>(set, lds);
  if (threadIdx.x == 0) {
    sums[2 * blockIdx.x] = clear;
    sums[2 * blockIdx.x + 1] = set;
  }
}

// One workgroup: the chunk that reaches the draw, the pick inside it, and for one measured qubit the
// norm of its outcome.
constexpr int kPickThreads = 1024;
template <typename R>
__global__ __launch_bounds__(kPickThreads) void k_measure_pick(const amp_t<R> *__restrict__ psi, MeasureArgs a, int lg,
                                                               uint32_t chunks, const double *__restrict__ sums, int single,
                                                               Measurement *__restrict__ m,
                                                               unsigned long long *__restrict__ host_pick) {
  __shared__ double lds[kPickThreads / 64];
  __shared__ unsigned long long found;
  __shared__ double before;
  uint64_t pick = ~uint64_t(0);
  if (a.rnd > 0.0) {
    const uint32_t per = (chunks + kPickThreads - 1) / kPickThreads;
    const uint32_t lo = min(chunks, threadIdx.x * per), hi = min(chunks, lo + per);
    auto value = [&](uint32_t c) { return sums[2 * c] + sums[2 * c + 1]; };
    const double mine = sum_range(lo, hi, value);
    if (threadIdx.x == 0) found = ~0ull;
    double total;
    const double start = prefix<kPickThreads>(mine, lds, &total);
    const uint32_t at = first_reaching(lo, hi, start, a.rnd, value);
    if (at < hi) atomicMin(&found, (unsigned long long)at);
    __syncthreads();
    const unsigned long long chunk = found;
    if (chunk == ~0ull) {
      pick = a.n_amps - 1;  // the draw exceeds the total norm: the scan runs off the end
    } else {
      if (chunk >= lo && chunk < hi) {
        before = start + sum_range(lo, (uint32_t)chunk, value);
      }
      __syncthreads();
      const uint64_t len = uint64_t(1) << lg;
      const unsigned long long c =
          scan_pick<R, kPickThreads>(psi, a, chunk * len, len, before, lds, &found, &total);
      pick = index_of(c != ~0ull ? (uint64_t)c : (chunk + 1) * len - 1, a);
    }
  }
  double kept = 0.0;
  if (single && !contradicts(a, pick)) {
    const uint32_t set = (pick & a.mask) ? 1 : 0;
#pragma unroll 8
    for (uint32_t c = threadIdx.x; c < chunks; c += kPickThreads) kept += sums[2 * c + set];
  }
  kept = sum_all<kPickThreads>(kept, lds);
  if (threadIdx.x == 0) {
    m->pick = pick;
    m->scale = 1.0 / sqrt(kept);
    *host_pick = pick;
  }
}

// Several measured qubits: the norm of the outcome over the amplitudes that have it, then its scale.  Over the
// whole subspace with a test of the index, 28 qubits complex64 took 0.22 ms even where one amplitude is left (8
// low qubits 1.92 ms, now 1.26).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_measure_kept(const amp_t<R> *__restrict__ psi, MeasureArgs a,
                                                         const Measurement *__restrict__ m, double *__restrict__ partials) {
  __shared__ double lds[kBlock / 64];
  const uint64_t pick = m->pick, fixed = (pick & a.mask) | (a.sval & ~a.mask);
  double kept = 0.0;
  if (!contradicts(a, pick))
    for (uint64_t c = (uint64_t)blockIdx.x * kBlock + threadIdx.x; c < a.n_kept; c += (uint64_t)gridDim.x * kBlock)
      kept += norm2(psi[scatter_bits(c, a.kept) | fixed]);
  kept = sum_all<kBlock>(kept, lds);
  if (threadIdx.x == 0) partials[blockIdx.x] = kept;
}
__global__ __launch_bounds__(kBlock) void k_measure_scale(const double *__restrict__ partials, Measurement *__restrict__ m) {
  __shared__ double lds[kBlock / 64];
  double kept = 0.0;
  for (int b = threadIdx.x; b < kReduceGrid; b += kBlock) kept += partials[b];
  kept = sum_all<kBlock>(kept, lds);
  if (threadIdx.x == 0) m->scale = 1.0 / sqrt(kept);
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_measure_collapse(amp_t<R> *__restrict__ psi, MeasureArgs a,
                                                             const Measurement *__restrict__ m) {
  const uint64_t val = m->pick & a.mask;
  const double scale = m->scale;
  const SpanSteps step(a.free);
  const uint64_t mine = scatter_bits(threadIdx.x, a.free);
  for (uint64_t first = blockIdx.x * kSpan; first < a.n_sub; first += gridDim.x * kSpan) {  // n_sub: whole spans
    const uint64_t here = index_of(first, a) | mine;
    amp_t<R> v[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      v[k].x = v[k].y = 0;
      if (((here | step.of[k]) & a.mask) == val) v[k] = psi[here | step.of[k]];
    }
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      amp_t<R> w;
      w.x = w.y = 0;
      if (((here | step.of[k]) & a.mask) == val) {
        w.x = (R)((double)v[k].x * scale);
        w.y = (R)((double)v[k].y * scale);
      }
      psi[here | step.of[k]] = w;
    }
  }
}

// SMALL: one workgroup, which writes the answer itself (up to 2^13 amplitudes).  28 qubits complex64 0.68 ms with one
// load in flight per thread, 0.50 now; 22 qubits 0.39 and 0.04 ms: most of it was 16384 atomics on one line.
template <typename R, bool SMALL>
__global__ __launch_bounds__(kBlock) void k_classical(const amp_t<R> *__restrict__ psi, uint64_t n_sub, BitRuns free,
                                                      uint64_t sval, int p, double tol, int *__restrict__ count,
                                                      int *__restrict__ flags) {
  int lo = 0, hi = 0;
  const SpanSteps step(free);
  const uint64_t mine = scatter_bits(threadIdx.x, free);
  for (uint64_t first = blockIdx.x * kSpan; first < n_sub; first += gridDim.x * kSpan) {
    const uint64_t here = scatter_bits(first, free) | sval | mine;
    amp_t<R> v[kBatch];
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      v[k].x = v[k].y = 0;
      if (first + k * kBlock + threadIdx.x < n_sub) v[k] = psi[here | step.of[k]];
    }
#pragma unroll
    for (int k = 0; k < kBatch; ++k) {
      const double x = v[k].x, y = v[k].y;
      const int big = first + k * kBlock + threadIdx.x < n_sub && (x * x + y * y) > tol;
      if (((here | step.of[k]) >> p) & 1) hi |= big;
      else lo |= big;
    }
  }
  lo = __syncthreads_or(lo);
  hi = __syncthreads_or(hi);
  if (threadIdx.x == 0) {
    if (SMALL) {
      *flags = (lo ? 1 : 0) | (hi ? 2 : 0);
    } else {
      // one side's flag is set by the first workgroups: the others only look
      if (lo && !__hip_atomic_load(&count[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicOr(&count[0], 1);
      if (hi && !__hip_atomic_load(&count[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT)) atomicOr(&count[1], 1);
    }
  }
}
__global__ void k_classical_clear(int *count) { count[threadIdx.x] = 0; }
__global__ void k_classical_flags(const int *__restrict__ count, int *__restrict__ flags) {
  *flags = (count[0] ? 1 : 0) | (count[1] ? 2 : 0);
}

unsigned grid_of(uint64_t work) { return (unsigned)std::min<uint64_t>(16384, std::max<uint64_t>(1, (work + kBlock - 1) / kBlock)); }

}  // namespace

template <typename R>
void measure(amp_t<R> *psi, const MeasureArgs &a, Measurement *m, unsigned long long *pick, double *sums, double *partials,
             hipEvent_t picked, hipStream_t s) {
  if (a.n_sub <= kMeasureSmall) {
    // as few waves as hold the subspace: their barriers are most of the time on 10 qubits and fewer
    if (a.n_sub <= 64 * 4) hipLaunchKernelGGL((k_measure_small<R, 64>), dim3(1), dim3(64), 0, s, psi, a, pick);
    else if (a.n_sub <= 256 * 4) hipLaunchKernelGGL((k_measure_small<R, 256>), dim3(1), dim3(256), 0, s, psi, a, pick);
    else hipLaunchKernelGGL((k_measure_small<R, 1024>), dim3(1), dim3(1024), 0, s, psi, a, pick);
    QS_HIP(hipGetLastError());
    QS_HIP(hipEventRecord(picked, s));
    return;
  }
  int lg = 8;  // about a thousand chunks, from 2^8 amplitudes to 2^12, then as many as fit the sums
  while (lg < 12 && (a.n_sub >> lg) > 1024) ++lg;
  while ((a.n_sub >> lg) > kMeasureChunks) ++lg;
  const uint32_t chunks = (uint32_t)(a.n_sub >> lg);
  const int single = a.mask != 0 && (a.mask & (a.mask - 1)) == 0;
  hipLaunchKernelGGL(k_measure_chunks<R>, dim3(chunks), dim3(kBlock), 0, s, psi, a, lg, sums);
  QS_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_measure_pick<R>, dim3(1), dim3(kPickThreads), 0, s, psi, a, lg, chunks, sums, single, m, pick);
  QS_HIP(hipGetLastError());
  QS_HIP(hipEventRecord(picked, s));
  if (!single) {
    hipLaunchKernelGGL(k_measure_kept<R>, dim3(kReduceGrid), dim3(kBlock), 0, s, psi, a, m, partials);
    QS_HIP(hipGetLastError());
    hipLaunchKernelGGL(k_measure_scale, dim3(1), dim3(kBlock), 0, s, partials, m);
    QS_HIP(hipGetLastError());
  }
  hipLaunchKernelGGL(k_measure_collapse<R>, dim3(grid_of(a.n_sub / kBatch)), dim3(kBlock), 0, s, psi, a, m);
  QS_HIP(hipGetLastError());
}

template <typename R>
void classical(const amp_t<R> *psi, uint64_t n_sub, const BitRuns &free, uint64_t sval, int p, double tol, int *count,
               int *flags, hipStream_t s) {
  if (n_sub <= 2 * kMeasureSmall) {
    hipLaunchKernelGGL((k_classical<R, true>), dim3(1), dim3(kBlock), 0, s, psi, n_sub, free, sval, p, tol, count, flags);
    QS_HIP(hipGetLastError());
    return;
  }
  hipLaunchKernelGGL(k_classical_clear, dim3(1), dim3(2), 0, s, count);
  QS_HIP(hipGetLastError());
  hipLaunchKernelGGL((k_classical<R, false>), dim3(grid_of(n_sub / kBatch)), dim3(kBlock), 0, s, psi, n_sub, free, sval, p, tol, count, flags);
  QS_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_classical_flags, dim3(1), dim3(1), 0, s, count, flags);
  QS_HIP(hipGetLastError());
}

#define QS_INSTANTIATE_MEASURE(R)                                                                                       \
  template void measure<R>(amp_t<R> *, const MeasureArgs &, Measurement *, unsigned long long *, double *, double *,   \
                           hipEvent_t, hipStream_t);                                                                    \
  template void classical<R>(const amp_t<R> *, uint64_t, const BitRuns &, uint64_t, int, double, int *, int *, hipStream_t);
QS_INSTANTIATE_MEASURE(double)
QS_INSTANTIATE_MEASURE(float)

}  // namespace dev
}  // namespace qs
