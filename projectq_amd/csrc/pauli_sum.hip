// A sum of Pauli strings applied to a state: qubit operators, and the Taylor terms of a time evolution
// (simulator.hpp:324-350, :386-438).
//
// Strings with the same x share the partner amplitude; their signs add up to one real (or imaginary)
// factor, of which a string costs one FP64 FMA per amplitude: the sign splits into a uniform part (tile
// base and j, folded into the scalar) and the thread's own parity.  Partners come from the tile in LDS
// where x lies in the tile's span (plan_sum), else from memory; workgroup b runs on XCD b mod 8 and takes
// its tiles from one eighth of the state, so near partners are in that XCD's L2.
//
// What bounds it: Infinity Cache traffic (state in, term out, sum in and out, partners outside the span
// that miss the L2).  Tiles of 2^10: 2^11 leave a third of the waves (147 VGPRs) for one partner more in
// LDS.  21 qubits complex128, transverse-field Ising chain (20 ZZ, 21 X), a Taylor term with its check:
// 95 us as one pass with a load and four complex operations per string, 63 us now.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "pauli_sum.hpp"

namespace qs {
namespace dev {
namespace {

__device__ __forceinline__ double flip(double v, uint32_t odd) {
  return __longlong_as_double(__double_as_longlong(v) ^ ((unsigned long long)odd << 63));
}

// u += (factor of the group's strings) b, over this thread's amplitudes; IM: times the imaginary unit
template <typename R, int NJ, bool IM>
__device__ __forceinline__ void add_group(const SumGroup &g, const EnergyString *__restrict__ strings, uint64_t base,
                                          const amp_t<R> *b, double *ur, double *ui) {
  const uint32_t tid = threadIdx.x;
  double f[NJ];
  {
    const EnergyString &st = g.head;
    const double w = flip(flip(st.w, (uint32_t)__popcll(base & st.z) & 1u), (uint32_t)__popc(tid & st.zloc) & 1u);
    const uint32_t zj = st.zloc >> 8;
#pragma unroll
    for (int j = 0; j < NJ; ++j) f[j] = flip(w, (uint32_t)__popc((uint32_t)j & zj) & 1u);
  }
#pragma unroll 4
  for (uint32_t s = 0; s < g.more; ++s) {
    const EnergyString st = strings[g.next + s];
    const uint32_t zj = st.zloc >> 8;
    const double one = flip(1.0, (uint32_t)__popc(tid & st.zloc) & 1u);
    const double w = flip(st.w, (uint32_t)__popcll(base & st.z) & 1u);
#pragma unroll
    for (int j = 0; j < NJ; ++j) f[j] = fma(flip(w, (uint32_t)__popc((uint32_t)j & zj) & 1u), one, f[j]);
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    if (IM) {
      ur[j] = fma(-f[j], (double)b[j].y, ur[j]);
      ui[j] = fma(f[j], (double)b[j].x, ui[j]);
    } else {
      ur[j] = fma(f[j], (double)b[j].x, ur[j]);
      ui[j] = fma(f[j], (double)b[j].y, ui[j]);
    }
  }
}

struct SumArgs {
  uint64_t n_amps, n_tiles, cmask;
  uint32_t L, h, n_groups;
  int first;
  double fr, fi, gr, gi;
  uint64_t gen[kEnergyMaxGens];
  uint8_t pivot[kEnergyMaxGens];
};

template <typename R, int LJ, bool EVOLVE>
__global__ __launch_bounds__(kBlock) void k_pauli_sum(const amp_t<R> *__restrict__ src, amp_t<R> *__restrict__ dst,
                                                      amp_t<R> *__restrict__ out, SumArgs a,
                                                      const SumGroup *__restrict__ groups,
                                                      const EnergyString *__restrict__ strings,
                                                      const EvolveState *__restrict__ evolve, double *__restrict__ partials) {
  constexpr int NJ = 1 << LJ;
  __shared__ amp_t<R> tile[256 << LJ];
  __shared__ double sums[kBlock / 64];
  if (EVOLVE && evolve->done) return;  // uniform over the launch
  const uint32_t tid = threadIdx.x;
  uint64_t mine = a.L >= 8 ? tid : tid & ((1u << a.L) - 1);
  for (uint32_t b = a.L; b < 8; ++b)
    if ((tid >> b) & 1) mine ^= a.gen[b - a.L];
  uint64_t step[LJ > 0 ? LJ : 1];
#pragma unroll
  for (int b = 0; b < LJ; ++b) step[b] = (uint32_t)(8 + b) < a.L ? uint64_t(256) << b : a.gen[8 + b - a.L];
  auto index = [&](uint64_t from, int j) {
    uint64_t o = from;
#pragma unroll
    for (int b = 0; b < LJ; ++b)
      if ((j >> b) & 1) o ^= step[b];
    return o;
  };
  double norm = 0.0;
  const uint64_t per = a.n_tiles >> 3;
  for (uint64_t k = blockIdx.x; k < a.n_tiles; k += gridDim.x) {
    // gridDim.x is a multiple of 8 where n_tiles is: k mod 8 stays this workgroup's XCD
    const uint64_t tix = (a.n_tiles & 7) ? k : (k & 7) * per + (k >> 3);
    uint64_t base = tix << a.L;
    for (uint32_t b = 0; b < a.h; ++b) {
      const uint32_t p = a.pivot[b];
      base = ((base >> p) << (p + 1)) | (base & ((uint64_t(1) << p) - 1));
    }
    const uint64_t here = base ^ mine;
    amp_t<R> own[NJ], b[NJ];
    double ur[NJ], ui[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const uint64_t o = index(here, j);
      own[j].x = own[j].y = 0;
      if (LJ > 0 || o < a.n_amps) own[j] = src[o];
      ur[j] = ui[j] = 0.0;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < NJ; ++j) tile[tid + 256u * j] = own[j];
    __syncthreads();
    // the next group's record loads while this one computes
    const SumGroup *gp = groups;
    SumGroup cur = a.n_groups ? *gp : SumGroup{};
    for (uint32_t g = 0; g < a.n_groups; ++g) {
      const SumGroup next = *++gp;
      if (cur.inside) {
        const uint32_t lo = tid ^ (cur.mask & 255u), mj = cur.mask & ~255u;
#pragma unroll
        for (int j = 0; j < NJ; ++j) b[j] = tile[lo | (((uint32_t)j << 8) ^ mj)];
      } else {
        const uint64_t there = here ^ cur.x;
#pragma unroll
        for (int j = 0; j < NJ; ++j) b[j] = src[index(there, j)];  // every amplitude of a state above one tile
      }
      if (cur.kind) add_group<R, NJ, true>(cur, strings, base, b, ur, ui);
      else add_group<R, NJ, false>(cur, strings, base, b, ur, ui);
      cur = next;
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      const uint64_t o = index(here, j);
      if (LJ == 0 && o >= a.n_amps) continue;
      const double vr = ur[j] * a.fr - ui[j] * a.fi, vi = ur[j] * a.fi + ui[j] * a.fr;
      amp_t<R> d;
      d.x = (R)vr;
      d.y = (R)vi;
      dst[o] = d;
      if (EVOLVE) {
        const bool on = (o & a.cmask) == a.cmask;
        if (on) {
          double xr, xi;
          if (a.first) {
            xr = (double)own[j].x * a.gr - (double)own[j].y * a.gi;
            xi = (double)own[j].x * a.gi + (double)own[j].y * a.gr;
          } else {
            const amp_t<R> x = out[o];
            xr = x.x;
            xi = x.y;
          }
          amp_t<R> y;
          y.x = (R)(xr + vr);
          y.y = (R)(xi + vi);
          out[o] = y;
          norm += vr * vr + vi * vi;
        } else if (a.first) {
          out[o] = own[j];
        }
      }
    }
  }
  if (EVOLVE) {
    for (int off = 32; off > 0; off >>= 1) norm += __shfl_down(norm, off, 64);
    if ((tid & 63) == 0) sums[tid >> 6] = norm;
    __syncthreads();
    if (tid == 0) {
      double t = 0.0;
      for (int w = 0; w < kBlock / 64; ++w) t += sums[w];
      partials[blockIdx.x] = t;
    }
  }
}

// Operators that need no tile (pauli_few): every amplitude reads its partners, from memory once where there is
// one x, from the caches on small states.  The tiles above cost them their upload, two barriers and a second read:
// 20 strings on 14 qubits 68 us through a tile, 55 here (62 with the same loop behind an upload); one string on 24 qubits
// complex64 90 and 67.  NJ amplitudes per thread: 1 on small states and for complex64 (4: 25 qubits 114 -> 132 us),
// 4 for complex128 (26 qubits 486 -> 406).
constexpr int kFewTerms = 64, kFewBits = 18;
struct FewTerms {
  uint64_t x[kFewTerms], z[kFewTerms];
  double re[kFewTerms], im[kFewTerms];
  uint32_t n;
};
template <typename R, int NJ>
__global__ __launch_bounds__(kBlock) void k_pauli_map(const amp_t<R> *__restrict__ src, amp_t<R> *__restrict__ dst,
                                                      uint64_t n_amps, FewTerms t) {
  for (uint64_t first = (uint64_t)blockIdx.x * kBlock * NJ + threadIdx.x; first < n_amps; first += (uint64_t)gridDim.x * kBlock * NJ) {
    double ur[NJ], ui[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) ur[j] = ui[j] = 0.0;
#pragma unroll 4
    for (uint32_t k = 0; k < t.n; ++k) {
      amp_t<R> b[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        b[j].x = b[j].y = 0;
        if (first + j * kBlock < n_amps) b[j] = src[(first + j * kBlock) ^ t.x[k]];
      }
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const uint32_t odd = (uint32_t)__popcll(((first + j * kBlock) ^ t.x[k]) & t.z[k]) & 1u;
        const double br = flip(b[j].x, odd), bi = flip(b[j].y, odd);
        ur[j] += br * t.re[k] - bi * t.im[k];
        ui[j] += br * t.im[k] + bi * t.re[k];
      }
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if (first + j * kBlock >= n_amps) continue;
      amp_t<R> d;
      d.x = (R)ur[j];
      d.y = (R)ui[j];
      dst[first + j * kBlock] = d;
    }
  }
}

// A launch of its own (5 us): the last workgroup of the term doing this behind an agent-scope counter
// made every workgroup write back and invalidate its L2, and the term twice as long.
__global__ __launch_bounds__(kBlock) void k_evolve_check(const double *__restrict__ partials, uint32_t n,
                                                         EvolveState *__restrict__ state, EvolveState *__restrict__ host) {
  __shared__ double sums[kBlock / 64];
  if (state->done) return;  // uniform; the host copy holds the last state
  double v = 0.0;
  for (uint32_t i = threadIdx.x; i < n; i += kBlock) v += partials[i];
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  if ((threadIdx.x & 63) == 0) sums[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kBlock / 64; ++w) t += sums[w];
    EvolveState now;
    now.done = !(sqrt(t) > 1.e-12);
    now.terms = state->terms + 1;
    *state = now;
    *host = now;
  }
}

__global__ void k_evolve_reset(EvolveState *state) {
  state->done = 0;
  state->terms = 0;
}

uint32_t workgroups(unsigned n, const SumPlan &plan) {
  const uint64_t tiles = n > plan.t ? uint64_t(1) << (n - plan.t) : 1;
  return (uint32_t)std::min<uint64_t>(tiles, kSumPartials);
}

}  // namespace

template <typename R>
void pauli_sum(const amp_t<R> *src, amp_t<R> *dst, amp_t<R> *out, unsigned n, const SumPlan &plan, const SumRecords &rec,
               std::complex<double> f, bool first, std::complex<double> g, uint64_t cmask, const EvolveState *evolve,
               double *partials, hipStream_t s) {
  SumArgs a;
  a.n_amps = uint64_t(1) << n;
  a.n_tiles = n > plan.t ? uint64_t(1) << (n - plan.t) : 1;
  a.cmask = cmask;
  a.L = plan.L;
  a.h = plan.h;
  a.n_groups = (uint32_t)plan.groups.size() - 1;
  a.first = first;
  a.fr = f.real();
  a.fi = f.imag();
  a.gr = g.real();
  a.gi = g.imag();
  for (int b = 0; b < kEnergyMaxGens; ++b) {
    a.gen[b] = plan.gen[b];
    a.pivot[b] = plan.pivot[b];
  }
  auto go = [&](auto lj) {
    constexpr int LJ = decltype(lj)::value;
    if (evolve)
      hipLaunchKernelGGL((k_pauli_sum<R, LJ, true>), dim3(workgroups(n, plan)), dim3(kBlock), 0, s, src, dst, out, a,
                         rec.groups, rec.strings, evolve, partials);
    else
      hipLaunchKernelGGL((k_pauli_sum<R, LJ, false>), dim3(workgroups(n, plan)), dim3(kBlock), 0, s, src, dst, out, a,
                         rec.groups, rec.strings, evolve, partials);
  };
  switch (plan.t) {
    case 8: go(std::integral_constant<int, 0>{}); break;
    case 9: go(std::integral_constant<int, 1>{}); break;
    case 10: go(std::integral_constant<int, 2>{}); break;
    case 11: go(std::integral_constant<int, 3>{}); break;
    default:
      if constexpr (sizeof(R) == 4) go(std::integral_constant<int, 4>{});
      else throw ValueError("pauli_sum: bad tile");
      break;
  }
  QS_HIP(hipGetLastError());
}

bool pauli_few(const std::vector<SumTerm> &terms, unsigned n) {
  if (terms.empty() || terms.size() > (size_t)kFewTerms) return false;
  if (n <= (unsigned)kFewBits) return true;
  return terms.size() == 1 || (terms.size() == 2 && (n <= kFewBits + 2 || terms[0].x == terms[1].x));
}

template <typename R>
void pauli_map(const amp_t<R> *src, amp_t<R> *dst, uint64_t n_amps, const std::vector<SumTerm> &terms, hipStream_t s) {
  FewTerms t;
  t.n = (uint32_t)terms.size();
  for (uint32_t k = 0; k < t.n; ++k) {
    t.x[k] = terms[k].x;
    t.z[k] = terms[k].z;
    t.re[k] = terms[k].c.real();
    t.im[k] = terms[k].c.imag();
  }
  auto go = [&](auto nj) {
    constexpr int NJ = decltype(nj)::value;
    const uint64_t grid = std::min<uint64_t>(16384, (n_amps + NJ * kBlock - 1) / (NJ * kBlock));
    hipLaunchKernelGGL((k_pauli_map<R, NJ>), dim3((unsigned)grid), dim3(kBlock), 0, s, src, dst, n_amps, t);
    QS_HIP(hipGetLastError());
  };
  if (sizeof(R) == 8 && n_amps > (uint64_t(1) << (kFewBits + 2))) go(std::integral_constant<int, 4>{});
  else go(std::integral_constant<int, 1>{});
}

void evolve_check(const double *partials, unsigned n, const SumPlan &plan, EvolveState *state, EvolveState *host, hipStream_t s) {
  hipLaunchKernelGGL(k_evolve_check, dim3(1), dim3(kBlock), 0, s, partials, workgroups(n, plan), state, host);
  QS_HIP(hipGetLastError());
}

void evolve_reset(EvolveState *state, hipStream_t s) {
  hipLaunchKernelGGL(k_evolve_reset, dim3(1), dim3(1), 0, s, state);
  QS_HIP(hipGetLastError());
}

template void pauli_map<float>(const float2 *, float2 *, uint64_t, const std::vector<SumTerm> &, hipStream_t);
template void pauli_map<double>(const double2 *, double2 *, uint64_t, const std::vector<SumTerm> &, hipStream_t);
template void pauli_sum<float>(const float2 *, float2 *, float2 *, unsigned, const SumPlan &, const SumRecords &,
                               std::complex<double>, bool, std::complex<double>, uint64_t, const EvolveState *, double *,
                               hipStream_t);
template void pauli_sum<double>(const double2 *, double2 *, double2 *, unsigned, const SumPlan &, const SumRecords &,
                                std::complex<double>, bool, std::complex<double>, uint64_t, const EvolveState *, double *,
                                hipStream_t);

}  // namespace dev
}  // namespace qs
