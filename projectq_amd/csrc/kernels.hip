// HIP kernels of the MI355X state-vector simulator (gfx950, wave64).
//
// Every kernel here is HBM-bound: one streaming pass over (a subspace of) the resident state.
// The dense-block kernel keeps the 2^k x 2^k matrix in scalar registers (uniform loads), holds
// the 2^k amplitudes of one group in VGPRs and streams each amplitude once in and once out.
// Reductions accumulate in FP64 whatever the state precision, with a fixed grid and a fixed
// final order so results are deterministic run to run.

#include <hip/hip_runtime.h>
#include <hipcub/hipcub.hpp>

#include <algorithm>
#include <cstdlib>
#include <type_traits>

#include "kernels.hpp"
#include "tile.hpp"

namespace qs {
namespace dev {
namespace {

template <typename A>
__device__ __forceinline__ double re(const A &a) {
  return (double)a.x;
}
template <typename A>
__device__ __forceinline__ double im(const A &a) {
  return (double)a.y;
}
template <typename R>
__device__ __forceinline__ amp_t<R> make_amp(double x, double y) {
  amp_t<R> a;
  a.x = (R)x;
  a.y = (R)y;
  return a;
}

__device__ __forceinline__ uint64_t insert_zeros(uint64_t g, const BitInsert &ins) {
  for (uint32_t i = 0; i < ins.count; ++i) {
    uint32_t p = ins.pos[i];
    g = ((g >> p) << (p + 1)) | (g & ((uint64_t(1) << p) - 1));
  }
  return g;
}

__device__ __forceinline__ uint64_t insert_one_zero(uint64_t g, int p) {
  return ((g >> p) << (p + 1)) | (g & ((uint64_t(1) << p) - 1));
}

inline int grid_for(uint64_t work, int cap = 16384) {
  uint64_t g = (work + kBlock - 1) / kBlock;
  if (g < 1) g = 1;
  if (g > (uint64_t)cap) g = cap;
  return (int)g;
}

// Sum over a workgroup of kBlock threads; result valid in thread 0.
__device__ __forceinline__ double block_sum(double v, double *lds) {
  for (int off = 32; off > 0; off >>= 1) v += __shfl_down(v, off, 64);
  int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) lds[wave] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < kBlock / 64; ++w) t += lds[w];
  __syncthreads();
  return t;
}

// Neumaier-compensated accumulator (used by the expectation value).
struct Kahan {
  double s = 0.0, c = 0.0;
  __device__ __forceinline__ void add(double v) {
    double t = s + v;
    if (fabs(s) >= fabs(v)) c += (s - t) + v;
    else c += (v - t) + s;
    s = t;
  }
  __device__ __forceinline__ double value() const { return s + c; }
};

// ------------------------------------------------------------------------------ gate blocks
template <int K>
struct Offsets {
  uint64_t o[1 << K];
};

// The matrix of a block of up to 4 qubits travels in the kernel arguments (at most 4 KiB), a 5-qubit
// one in device memory.  With an upload of its own before every gate, a 21-qubit complex128 circuit in
// 81 blocks took 1.46 ms (18 us a block, 5 of them the copy and the wait for it) and takes 1.26 ms.
template <typename R, int K>
struct BlockMatrix {
  amp_t<R> m[(1 << K) * (1 << K)];
  __device__ __forceinline__ const amp_t<R> &operator[](int i) const { return m[i]; }
};
template <typename R>
struct BlockMatrix<R, 5> {
  const amp_t<R> *__restrict__ p;
  __device__ __forceinline__ const amp_t<R> &operator[](int i) const { return p[i]; }
};

template <typename R, int K>
__global__ __launch_bounds__(kBlock) void k_apply(amp_t<R> *__restrict__ psi, uint64_t n_groups,
                                                  BitInsert ins, uint64_t cmask, Offsets<K> off,
                                                  BlockMatrix<R, K> m) {
  constexpr int D = 1 << K;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < n_groups; g += stride) {
    const uint64_t base = insert_zeros(g, ins) | cmask;
    R vr[D], vi[D];
#pragma unroll
    for (int j = 0; j < D; ++j) {
      amp_t<R> a = psi[base + off.o[j]];
      vr[j] = a.x;
      vi[j] = a.y;
    }
#pragma unroll(K <= 3 ? D : 1)
    for (int r = 0; r < D; ++r) {
      R ar = 0, ai = 0;
#pragma unroll
      for (int c = 0; c < D; ++c) {
        const amp_t<R> mc = m[r * D + c];
        ar = fma(mc.x, vr[c], ar);
        ar = fma(-mc.y, vi[c], ar);
        ai = fma(mc.x, vi[c], ai);
        ai = fma(mc.y, vr[c], ai);
      }
      amp_t<R> o;
      o.x = ar;
      o.y = ai;
      psi[base + off.o[r]] = o;
    }
  }
}

template <typename R, int K>
void launch_apply(amp_t<R> *psi, uint64_t n_groups, const BitInsert &ins, uint64_t cmask,
                  const uint32_t *tpos, const BlockMatrix<R, K> &m, hipStream_t s) {
  Offsets<K> off;
  for (int j = 0; j < (1 << K); ++j) {
    uint64_t o = 0;
    for (int l = 0; l < K; ++l)
      if ((j >> l) & 1) o |= uint64_t(1) << tpos[l];
    off.o[j] = o;
  }
  hipLaunchKernelGGL((k_apply<R, K>), dim3(grid_for(n_groups)), dim3(kBlock), 0, s, psi, n_groups,
                     ins, cmask, off, m);
  QS_HIP(hipGetLastError());
}

// ------------------------------------------------------------------------------ batched circuits
template <typename R>
__global__ __launch_bounds__(kBlock) void k_batch_zero(amp_t<R> *__restrict__ psi, uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
    psi[i] = make_amp<R>(0.0, 0.0);
}
template <typename R>
__global__ void k_batch_ones(amp_t<R> *__restrict__ psi, const uint64_t *__restrict__ off, int n) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c < n) psi[off[c]] = make_amp<R>(1.0, 0.0);
}

// ------------------------------------------------------------------------------ reductions
template <typename R>
__global__ __launch_bounds__(kBlock) void k_norm_masked(const amp_t<R> *__restrict__ psi,
                                                        uint64_t n_sub, BitInsert ins,
                                                        uint64_t val, double *partials) {
  __shared__ double lds[kBlock / 64];
  double acc = 0.0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t g = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; g < n_sub; g += stride) {
    amp_t<R> a = psi[insert_zeros(g, ins) | val];
    double x = re(a), y = im(a);
    acc = fma(x, x, fma(y, y, acc));
  }
  double t = block_sum(acc, lds);
  if (threadIdx.x == 0) partials[blockIdx.x] = t;
}

// One workgroup per output: thread t adds partials t, t + 256, ... and the workgroup's sums are added
// in a fixed order.  One thread adding the 2048 partials of a reduction took 150 us, a chain of 2048
// dependent loads and adds that every probability, norm and Taylor term waited for; this takes
// about 3 us (the launch).  `out` may be pinned host memory.
__global__ __launch_bounds__(kBlock) void k_finish_sum(const double *__restrict__ partials, int n_partials, int width,
                                                       double *__restrict__ out) {
  __shared__ double lds[kBlock / 64];
  const int j = blockIdx.x;
  double acc = 0.0;
  for (int b = threadIdx.x; b < n_partials; b += kBlock) acc += partials[(size_t)b * width + j];
  const double t = block_sum(acc, lds);
  if (threadIdx.x == 0) out[j] = t;
}

// The collapse runs over a subspace: compact index c is the amplitude
// insert_zeros(c, sub) | sval, so the bits listed in `sub` are fixed to their values in sval (the
// caller knows every amplitude outside is zero).  With sub.count = 0 it covers the whole state.
template <typename R>
__global__ __launch_bounds__(kBlock) void k_collapse(amp_t<R> *__restrict__ psi, uint64_t n_sub, BitInsert sub,
                                                     uint64_t sval, uint64_t mask, uint64_t val, double scale) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; c < n_sub; c += stride) {
    const uint64_t i = insert_zeros(c, sub) | sval;
    amp_t<R> a = psi[i];
    if ((i & mask) != val) a = make_amp<R>(0.0, 0.0);
    else a = make_amp<R>(re(a) * scale, im(a) * scale);
    psi[i] = a;
  }
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_first_pair(const amp_t<R> *__restrict__ psi,
                                                       uint64_t n_pairs, int p, double tol,
                                                       unsigned long long *key) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  unsigned long long best = ~0ull;
  for (uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n_pairs; q += stride) {
    const uint64_t i0 = insert_one_zero(q, p), i1 = i0 | (uint64_t(1) << p);
    amp_t<R> a = psi[i0], b = psi[i1];
    double n0 = re(a) * re(a) + im(a) * im(a), n1 = re(b) * re(b) + im(b) * im(b);
    if (n0 > tol) {
      best = min(best, (unsigned long long)(2 * q));
      break;  // q only grows in this thread
    }
    if (n1 > tol) {
      best = min(best, (unsigned long long)(2 * q + 1));
      break;
    }
  }
  if (best != ~0ull) atomicMin(key, best);
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_drop_bit(const amp_t<R> *__restrict__ src,
                                                     amp_t<R> *__restrict__ dst, uint64_t n_out,
                                                     int p, int value) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  const uint64_t set = uint64_t(value ? 1 : 0) << p;
  for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n_out; j += stride)
    dst[j] = src[insert_one_zero(j, p) | set];
}

// A qubit layout change, one exchange of two index bits at a time: the amplitudes whose bits a and
// b differ trade places (half the state read and written; a one-off when the layout is handed out).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_swap_bits(amp_t<R> *__restrict__ psi, uint64_t n_pairs, int lo, int hi) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t c = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; c < n_pairs; c += stride) {
    const uint64_t i = insert_one_zero(insert_one_zero(c, lo), hi) | (uint64_t(1) << lo);
    const uint64_t j = i ^ (uint64_t(1) << lo) ^ (uint64_t(1) << hi);
    const amp_t<R> x = psi[i], y = psi[j];
    psi[i] = y;
    psi[j] = x;
  }
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_scale_masked(amp_t<R> *__restrict__ psi, uint64_t n,
                                                         uint64_t cmask, double cr, double ci) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    if ((i & cmask) != cmask) continue;
    amp_t<R> a = psi[i];
    psi[i] = make_amp<R>(re(a) * cr - im(a) * ci, re(a) * ci + im(a) * cr);
  }
}

// ------------------------------------------------------------------------------ emulate_math
__device__ __forceinline__ int32_t wrap32(int64_t x) { return (int32_t)(uint32_t)(uint64_t)x; }
__device__ __forceinline__ int32_t check32(int64_t x, int &bad) {
  if (x < INT32_MIN || x > INT32_MAX) bad = 1;
  return (int32_t)x;
}
__device__ __forceinline__ int64_t floordiv(int64_t a, int64_t b) {
  int64_t q = a / b;
  if ((a % b != 0) && ((a < 0) != (b < 0))) --q;
  return q;
}
__device__ __forceinline__ int64_t py_bitlen(int64_t x) {  // len(bin(x)[2:])
  if (x == 0) return 1;
  if (x > 0) return 64 - __clzll((unsigned long long)x);
  return 64 - __clzll((unsigned long long)(-x)) + 1;
}

// new values of the registers for opcode args.opcode (include/projectq_amd.h QS_MATH_*)
__device__ void math_eval(const MathArgs &A, int32_t *v, int &bad) {
  switch (A.opcode) {
    case 0:
      for (int r = 0; r < A.n_regs; ++r) v[r] = wrap32((int64_t)v[r] + (int32_t)A.a);
      break;
    case 1:
      for (int r = 0; r < A.n_regs; ++r)
        v[r] = wrap32(wrap32((int64_t)v[r] + (int32_t)A.a) % (int32_t)A.N);
      break;
    case 2:
      for (int r = 0; r < A.n_regs; ++r)
        v[r] = wrap32(wrap32((int64_t)v[r] * (int32_t)A.a) % (int32_t)A.N);
      break;
    case 3: {
      int64_t s = (int64_t)v[0] + v[1];
      if (py_bitlen(s) > (int64_t)A.width[0]) {
        int64_t mod = int64_t(1) << A.width[0];
        s = ((s % mod) + mod) % mod;
        if (A.n_regs == 3) v[2] ^= 1;
      }
      v[1] = check32(s, bad);
      break;
    }
    case 4:
      v[1] = check32((int64_t)v[1] - v[0], bad);
      break;
    case 5:
      if (A.n_regs == 3) v[2] ^= 1;
      v[1] = check32((int64_t)v[1] - v[0], bad);
      break;
    case 6:
      if (v[1] < v[0]) v[2] = (v[2] == 0) ? 1 : 0;
      break;
    case 7:
      v[2] = check32((int64_t)v[2] + (int64_t)v[0] * v[1], bad);
      break;
    case 8:
      v[2] = check32((int64_t)v[2] - (int64_t)v[0] * v[1], bad);
      break;
    case 9: {
      int64_t dividend = v[0], rem = v[1], divisor = v[2];
      if (divisor == 0 || divisor > dividend) {
        v[0] = check32(rem, bad);
        v[1] = check32(dividend, bad);
      } else {
        int64_t q = rem + floordiv(dividend, divisor);
        v[0] = check32(dividend - q * divisor, bad);
        v[1] = check32(q, bad);
      }
      break;
    }
    case 10: {
      int64_t rem = v[0], quo = v[1], divisor = v[2];
      if (divisor == 0) {
        v[0] = check32(quo, bad);
        v[1] = check32(rem, bad);
      } else {
        v[0] = check32(rem + quo * divisor, bad);
        v[1] = 0;
      }
      break;
    }
    default:
      bad = 1;
  }
}

// destination index of basis state i (simulator.hpp:246-265)
__device__ uint64_t math_dest(uint64_t i, const MathArgs &A, const int32_t *table, int &bad) {
  if ((i & A.cmask) != A.cmask) return i;
  int32_t v[kMaxRegs];
  uint64_t packed = 0;
  int shift = 0;
  for (int r = 0; r < A.n_regs; ++r) {
    uint64_t x = 0;
    for (int b = 0; b < A.width[r]; ++b) x |= ((i >> A.pos[r][b]) & 1ull) << b;
    v[r] = (int32_t)(uint32_t)x;
    packed |= x << shift;
    shift += A.width[r];
  }
  if (table) {
    for (int r = 0; r < A.n_regs; ++r) v[r] = table[packed * A.n_regs + r];
  } else {
    math_eval(A, v, bad);
  }
  uint64_t j = i;
  for (int r = 0; r < A.n_regs; ++r)
    for (int b = 0; b < A.width[r]; ++b) {
      uint64_t want = (uint64_t)(((int64_t)v[r] >> (b < 63 ? b : 63)) & 1);
      j = (j & ~(uint64_t(1) << A.pos[r][b])) | (want << A.pos[r][b]);
    }
  return j;
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_math_permute(const amp_t<R> *__restrict__ src,
                                                         amp_t<R> *__restrict__ dst, uint64_t n,
                                                         MathArgs A, const int32_t *table,
                                                         int *err) {
  int bad = 0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint64_t j = math_dest(i, A, table, bad);
    amp_t<R> a = src[i];
    dst[j] = make_amp<R>(0.0 + re(a), 0.0 + im(a));  // newvec starts at 0 (simulator.hpp:239-240)
  }
  if (bad) atomicOr(err, 1);
}

__global__ __launch_bounds__(kBlock) void k_math_injective(uint64_t n, MathArgs A,
                                                           const int32_t *table, uint32_t *bitmap,
                                                           int *collide, int *err) {
  int bad = 0, hit = 0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    uint64_t j = math_dest(i, A, table, bad);
    uint32_t bit = 1u << (j & 31);
    uint32_t old = atomicOr(&bitmap[j >> 5], bit);
    if (old & bit) hit = 1;
  }
  if (bad) atomicOr(err, 1);
  if (hit) atomicOr(collide, 1);
}

__global__ __launch_bounds__(kBlock) void k_math_keys(uint64_t n, MathArgs A, const int32_t *table,
                                                      uint32_t *keys, uint32_t *vals, int *err) {
  int bad = 0;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    keys[i] = (uint32_t)math_dest(i, A, table, bad);
    vals[i] = (uint32_t)i;
  }
  if (bad) atomicOr(err, 1);
}

template <typename R>
__global__ __launch_bounds__(kBlock) void k_math_segments(const amp_t<R> *__restrict__ src,
                                                          amp_t<R> *__restrict__ dst, uint64_t n,
                                                          const uint32_t *keys,
                                                          const uint32_t *vals) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t j = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += stride) {
    if (j > 0 && keys[j] == keys[j - 1]) continue;
    double sr = 0.0, si = 0.0;
    uint64_t k = j;
    do {
      amp_t<R> a = src[vals[k]];
      sr += re(a);
      si += im(a);
      ++k;
    } while (k < n && keys[k] == keys[j]);
    dst[keys[j]] = make_amp<R>(sr, si);
  }
}

template <typename Ra, typename Rb>
__global__ __launch_bounds__(kBlock) void k_overlap(const amp_t<Ra> *__restrict__ a,
                                                    const amp_t<Rb> *__restrict__ b, uint64_t n,
                                                    double *partials) {
  __shared__ double lds[kBlock / 64];
  Kahan sr, si;
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    amp_t<Ra> x = a[i];
    amp_t<Rb> y = b[i];
    sr.add(re(x) * re(y) + im(x) * im(y));
    si.add(re(x) * im(y) - im(x) * re(y));
  }
  double tr = block_sum(sr.value(), lds);
  double ti = block_sum(si.value(), lds);
  if (threadIdx.x == 0) {
    partials[2 * blockIdx.x] = tr;
    partials[2 * blockIdx.x + 1] = ti;
  }
}

}  // namespace

// ------------------------------------------------------------------------------ launchers
void overlap(const void *a, bool a_c64, const void *b, bool b_c64, uint64_t n, double *partials,
             hipStream_t s) {
  dim3 g(kReduceGrid), t(kBlock);
  if (!a_c64 && !b_c64)
    hipLaunchKernelGGL((k_overlap<double, double>), g, t, 0, s, (const double2 *)a, (const double2 *)b, n, partials);
  else if (!a_c64 && b_c64)
    hipLaunchKernelGGL((k_overlap<double, float>), g, t, 0, s, (const double2 *)a, (const float2 *)b, n, partials);
  else if (a_c64 && !b_c64)
    hipLaunchKernelGGL((k_overlap<float, double>), g, t, 0, s, (const float2 *)a, (const double2 *)b, n, partials);
  else
    hipLaunchKernelGGL((k_overlap<float, float>), g, t, 0, s, (const float2 *)a, (const float2 *)b, n, partials);
  QS_HIP(hipGetLastError());
}
template <typename R>
void apply_block(amp_t<R> *psi, uint64_t n_groups, const BitInsert &ins, uint64_t cmask,
                 const uint32_t *tpos, int k, const std::complex<double> *mat, const amp_t<R> *d_mat, hipStream_t s) {
  auto go = [&](auto width) {
    constexpr int K = decltype(width)::value;
    BlockMatrix<R, K> m;
    if constexpr (K == 5) {
      m.p = d_mat;
    } else {
      for (int i = 0; i < (1 << (2 * K)); ++i) {
        m.m[i].x = (R)mat[i].real();
        m.m[i].y = (R)mat[i].imag();
      }
    }
    launch_apply<R, K>(psi, n_groups, ins, cmask, tpos, m, s);
  };
  switch (k) {
    case 1: go(std::integral_constant<int, 1>{}); break;
    case 2: go(std::integral_constant<int, 2>{}); break;
    case 3: go(std::integral_constant<int, 3>{}); break;
    case 4: go(std::integral_constant<int, 4>{}); break;
    case 5: go(std::integral_constant<int, 5>{}); break;
    default: throw ValueError("Gates with more than 5 qubits are not supported!");
  }
}

template <typename R>
void tile_pass(amp_t<R> *psi, uint64_t n_tiles, const TilePass &P, int rb, const TileStage *d_stages,
               const RegOp *d_rops, const TileOp *d_tops, const amp_t<R> *d_mats, TileForms forms, hipStream_t s) {
  if (P.h > (uint32_t)kTileMaxHigh || P.L < 1 || P.t > (uint32_t)kTileMaxBits)
    throw ValueError("tile pass: bad tile shape");
  if (rb == 5) launch_tile_pass<R, 5>(psi, n_tiles, P, d_stages, d_rops, d_tops, d_mats, forms, s);
  else if (rb == 4) launch_tile_pass<R, 4>(psi, n_tiles, P, d_stages, d_rops, d_tops, d_mats, forms, s);
  else throw ValueError("tile pass: register bits must be 4 or 5");
}

void prepare_tile_kernels() {
  static bool done = false;
  if (done) return;
  prepare_tile_kernels_of<float, 4>();
  prepare_tile_kernels_of<float, 5>();
  prepare_tile_kernels_of<double, 4>();
  prepare_tile_kernels_of<double, 5>();
  prepare_tile_kernels_pf();
  prepare_tile_kernels_phase_c64();
  prepare_tile_kernels_phase_c128();
  done = true;
}

template <typename R>
void batch_init(amp_t<R> *psi, uint64_t total, const uint64_t *state_off, int n_states, hipStream_t s) {
  hipLaunchKernelGGL(k_batch_zero<R>, dim3(grid_for(total)), dim3(kBlock), 0, s, psi, total);
  QS_HIP(hipGetLastError());
  hipLaunchKernelGGL(k_batch_ones<R>, dim3((n_states + 255) / 256), dim3(256), 0, s, psi, state_off, n_states);
  QS_HIP(hipGetLastError());
}

template <typename R>
void batch_tile_pass(amp_t<R> *psi, const BatchJob *jobs, const uint32_t *block_job, uint32_t n_blocks,
                     uint32_t max_t, int rb, const TileStage *stages, const RegOp *rops, const TileOp *tops,
                     const amp_t<R> *mats, bool two_qubit_ops, hipStream_t s) {
  if (max_t > (uint32_t)kTileMaxBits || n_blocks == 0) throw ValueError("batch pass: bad launch shape");
  if (rb == 5)
    launch_batch_tile_pass<R, 5>(psi, jobs, block_job, n_blocks, max_t, stages, rops, tops, mats, two_qubit_ops, s);
  else if (rb == 4)
    launch_batch_tile_pass<R, 4>(psi, jobs, block_job, n_blocks, max_t, stages, rops, tops, mats, two_qubit_ops, s);
  else throw ValueError("batch pass: register bits must be 4 or 5");
}

template <typename R>
void norm_masked(const amp_t<R> *psi, uint64_t n_sub, const BitInsert &ins, uint64_t val,
                 double *partials, hipStream_t s) {
  hipLaunchKernelGGL(k_norm_masked<R>, dim3(kReduceGrid), dim3(kBlock), 0, s, psi, n_sub, ins, val,
                     partials);
  QS_HIP(hipGetLastError());
}

void finish_sum(const double *partials, int n_partials, int width, double *out, hipStream_t s) {
  hipLaunchKernelGGL(k_finish_sum, dim3(width), dim3(kBlock), 0, s, partials, n_partials, width, out);
  QS_HIP(hipGetLastError());
}

template <typename R>
void collapse(amp_t<R> *psi, uint64_t n_sub, const BitInsert &sub, uint64_t sval, uint64_t mask, uint64_t val,
              double scale, hipStream_t s) {
  hipLaunchKernelGGL(k_collapse<R>, dim3(grid_for(n_sub)), dim3(kBlock), 0, s, psi, n_sub, sub, sval, mask, val,
                     scale);
  QS_HIP(hipGetLastError());
}

template <typename R>
void first_pair(const amp_t<R> *psi, uint64_t n_pairs, int p, double tol, unsigned long long *key,
                hipStream_t s) {
  hipLaunchKernelGGL(k_first_pair<R>, dim3(grid_for(n_pairs)), dim3(kBlock), 0, s, psi, n_pairs, p,
                     tol, key);
  QS_HIP(hipGetLastError());
}

template <typename R>
void drop_bit(const amp_t<R> *src, amp_t<R> *dst, uint64_t n_out, int p, int value, hipStream_t s) {
  hipLaunchKernelGGL(k_drop_bit<R>, dim3(grid_for(n_out)), dim3(kBlock), 0, s, src, dst, n_out, p,
                     value);
  QS_HIP(hipGetLastError());
}

template <typename R>
void swap_bits(amp_t<R> *psi, uint64_t n_amps, int a, int b, hipStream_t s) {
  if (a == b || n_amps < 4) return;
  const int lo = a < b ? a : b, hi = a < b ? b : a;
  hipLaunchKernelGGL(k_swap_bits<R>, dim3(grid_for(n_amps / 4)), dim3(kBlock), 0, s, psi, n_amps / 4, lo, hi);
  QS_HIP(hipGetLastError());
}

template <typename R>
void scale_masked(amp_t<R> *psi, uint64_t n, uint64_t cmask, double cr, double ci, hipStream_t s) {
  hipLaunchKernelGGL(k_scale_masked<R>, dim3(grid_for(n)), dim3(kBlock), 0, s, psi, n, cmask, cr, ci);
  QS_HIP(hipGetLastError());
}

template <typename R>
void math_permute(const amp_t<R> *src, amp_t<R> *dst, uint64_t n, const MathArgs &args,
                  const int32_t *table, int *err, hipStream_t s) {
  hipLaunchKernelGGL(k_math_permute<R>, dim3(grid_for(n)), dim3(kBlock), 0, s, src, dst, n, args,
                     table, err);
  QS_HIP(hipGetLastError());
}

void math_injective(uint64_t n, const MathArgs &args, const int32_t *table, uint32_t *bitmap,
                    int *collide, int *err, hipStream_t s) {
  hipLaunchKernelGGL(k_math_injective, dim3(grid_for(n)), dim3(kBlock), 0, s, n, args, table, bitmap,
                     collide, err);
  QS_HIP(hipGetLastError());
}

template <typename R>
void math_accumulate(const amp_t<R> *src, amp_t<R> *dst, uint64_t n, const MathArgs &args,
                     const int32_t *table, int *err, hipStream_t s) {
  if (n > (uint64_t(1) << 30))
    throw ValueError("emulate_math: a non-injective function on more than 30 qubits is not supported");
  uint32_t *buf = nullptr;
  QS_HIP(hipMalloc(&buf, 4 * n * sizeof(uint32_t)));
  uint32_t *k_in = buf, *v_in = buf + n, *k_out = buf + 2 * n, *v_out = buf + 3 * n;
  void *tmp = nullptr;
  size_t tmp_bytes = 0;
  int bits = 1;
  while ((uint64_t(1) << bits) < n) ++bits;
  try {
    hipLaunchKernelGGL(k_math_keys, dim3(grid_for(n)), dim3(kBlock), 0, s, n, args, table, k_in,
                       v_in, err);
    QS_HIP(hipGetLastError());
    QS_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, k_in, k_out, v_in, v_out, (int)n, 0,
                                              bits, s));
    QS_HIP(hipMalloc(&tmp, tmp_bytes));
    QS_HIP(hipcub::DeviceRadixSort::SortPairs(tmp, tmp_bytes, k_in, k_out, v_in, v_out, (int)n, 0,
                                              bits, s));
    hipLaunchKernelGGL(k_math_segments<R>, dim3(grid_for(n)), dim3(kBlock), 0, s, src, dst, n, k_out,
                       v_out);
    QS_HIP(hipGetLastError());
    QS_HIP(hipStreamSynchronize(s));
  } catch (...) {
    (void)hipStreamSynchronize(s);
    (void)hipFree(tmp);
    (void)hipFree(buf);
    throw;
  }
  QS_HIP(hipFree(tmp));
  QS_HIP(hipFree(buf));
}

// ------------------------------------------------------------------------------ instantiations
template <typename S, typename D>
__global__ __launch_bounds__(kBlock) void k_convert_amps(const amp_t<S> *__restrict__ src, amp_t<D> *__restrict__ dst,
                                                         uint64_t n) {
  const uint64_t stride = (uint64_t)gridDim.x * blockDim.x;
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride) {
    const amp_t<S> a = src[i];
    amp_t<D> b;
    b.x = (D)a.x;
    b.y = (D)a.y;
    dst[i] = b;
  }
}

template <typename S, typename D>
void convert_amps(const amp_t<S> *src, amp_t<D> *dst, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL((k_convert_amps<S, D>), dim3(grid_for(n)), dim3(kBlock), 0, s, src, dst, n);
  QS_HIP(hipGetLastError());
}
template void convert_amps<double, float>(const amp_t<double> *, amp_t<float> *, uint64_t, hipStream_t);
template void convert_amps<float, double>(const amp_t<float> *, amp_t<double> *, uint64_t, hipStream_t);

#define QS_INSTANTIATE(R)                                                                          \
  template void batch_init<R>(amp_t<R> *, uint64_t, const uint64_t *, int, hipStream_t);          \
  template void batch_tile_pass<R>(amp_t<R> *, const BatchJob *, const uint32_t *, uint32_t,       \
                                   uint32_t, int, const TileStage *, const RegOp *, const TileOp *,\
                                   const amp_t<R> *, bool, hipStream_t);                                \
  template void tile_pass<R>(amp_t<R> *, uint64_t, const TilePass &, int, const TileStage *,      \
                             const RegOp *, const TileOp *, const amp_t<R> *, TileForms, hipStream_t); \
  template void apply_block<R>(amp_t<R> *, uint64_t, const BitInsert &, uint64_t,                 \
                               const uint32_t *, int, const std::complex<double> *, const amp_t<R> *, hipStream_t); \
  template void norm_masked<R>(const amp_t<R> *, uint64_t, const BitInsert &, uint64_t, double *, \
                               hipStream_t);                                                      \
  template void collapse<R>(amp_t<R> *, uint64_t, const BitInsert &, uint64_t, uint64_t, uint64_t, double,    \
                            hipStream_t);                                                         \
  template void first_pair<R>(const amp_t<R> *, uint64_t, int, double, unsigned long long *,      \
                              hipStream_t);                                                       \
  template void drop_bit<R>(const amp_t<R> *, amp_t<R> *, uint64_t, int, int, hipStream_t);       \
  template void swap_bits<R>(amp_t<R> *, uint64_t, int, int, hipStream_t);                          \
  template void scale_masked<R>(amp_t<R> *, uint64_t, uint64_t, double, double, hipStream_t);     \
  template void math_permute<R>(const amp_t<R> *, amp_t<R> *, uint64_t, const MathArgs &,         \
                                const int32_t *, int *, hipStream_t);                             \
  template void math_accumulate<R>(const amp_t<R> *, amp_t<R> *, uint64_t, const MathArgs &,      \
                                   const int32_t *, int *, hipStream_t);

QS_INSTANTIATE(double)
QS_INSTANTIATE(float)

}  // namespace dev
}  // namespace qs
