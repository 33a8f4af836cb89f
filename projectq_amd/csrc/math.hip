// emulate_math as a gather: every destination amplitude reads its source (math_map.hpp), so the
// writes run in memory order and no pass over the state is needed to find out that the map is one to
// one.
//
// What bounds it: HBM, one read and one write of the state, once the reads are arranged.  An
// addition b <- a + b sends the amplitudes of one cache line to as many different rows, so in memory
// order every 8- or 16-byte access is a line of its own.  The traversal therefore puts 256
// contiguous bytes and the lowest bits of the changing registers into one workgroup (MathGather::
// order): its reads are a parallelogram of whole lines but for the edges, and neighbouring workgroups,
// which share the edges, run on one XCD and meet in its L2.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "kernels.hpp"
#include "math_map.hpp"

namespace qs {
namespace dev {
namespace {

constexpr int kMathBits = 8 + kMathThreadBits;  // amplitudes per workgroup: 2^12, 16 per thread

// workgroup -> tile: workgroup b runs on XCD b mod 8, which gets a contiguous eighth of the tiles
__device__ __forceinline__ uint64_t tile_of(uint64_t b, uint64_t n_tiles) {
  return (n_tiles & 7) ? b : (b & 7) * (n_tiles >> 3) + (b >> 3);
}

template <typename R, int S>
__global__ __launch_bounds__(kBlock) void k_math_gather(const amp_t<R> *__restrict__ src, amp_t<R> *__restrict__ dst,
                                                        uint64_t n_amps, uint64_t n_tiles, MathGather G) {
  constexpr int NJ = 1 << (kMathBits - 8);
  constexpr bool MOD = S == kSrcAddMod || S == kSrcMulMod;
  const uint64_t first = tile_of(blockIdx.x, n_tiles) << kMathBits;
  // index and register values are linear in the counter bits: a thread's part, and a uniform one
  const uint64_t it = scatter_bits(threadIdx.x, G.order) | scatter_bits(first, G.order);
  uint64_t rt[3];
#pragma unroll
  for (int r = 0; r < 3; ++r) rt[r] = r < G.n_regs ? gather_bits(it, G.reg[r]) : 0;
  auto part = [](int j, auto &&of_bit) {  // of counter bits 8..11 = j, uniform
    decltype(of_bit(0)) v = 0;
#pragma unroll
    for (int b = 0; b < kMathThreadBits; ++b)
      if ((j >> b) & 1) v |= of_bit(b);
    return v;
  };
  auto step = [&](int b) { return G.step[b]; };
  amp_t<R> out[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const uint64_t i = it | part(j, step);
    out[j].x = 0;
    out[j].y = 0;
    if ((first | threadIdx.x | ((uint64_t)j << 8)) >= n_amps) continue;
    uint64_t s = i;
    if ((i & G.cmask) == G.cmask) {
      uint64_t u = rt[0] | part(j, [&](int b) { return G.reg_step[b][0]; });
      uint64_t v = rt[1] | part(j, [&](int b) { return G.reg_step[b][1]; });
      uint64_t w = rt[2] | part(j, [&](int b) { return G.reg_step[b][2]; });
      const bool any = math_source<S>(G, u, v, w);
      s = i & ~G.changed;
      if constexpr (MOD) {
        if (any) {
          double x = 0.0, y = 0.0;  // newvec starts at 0 and adds in index order (simulator.hpp:239-266)
          do {
            const amp_t<R> a = src[s | scatter_bits(u, G.reg[0])];
            x += (double)a.x;
            y += (double)a.y;
            u += G.N;
          } while (u >> G.width[0] == 0);
          out[j].x = (R)x;
          out[j].y = (R)y;
        }
        continue;
      }
      (void)any;  // one to one
      const uint64_t values[3] = {u, v, w};
#pragma unroll
      for (int r = 0; r < 3; ++r)
        if (G.moves[r]) s |= scatter_bits(values[r], G.reg[r]);
    }
    out[j] = src[s];
  }
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    if ((first | threadIdx.x | ((uint64_t)j << 8)) >= n_amps) continue;
    amp_t<R> a;
    a.x = (R)0 + out[j].x;  // newvec starts at 0 (simulator.hpp:239-240): -0 becomes +0
    a.y = (R)0 + out[j].y;
    dst[it | part(j, step)] = a;
  }
}

// Additions of a constant (MathAdd): a source costs a few operations however its bits lie, so the destinations
// go in memory order with eight loads in flight per thread.  Bound by HBM on large states: 27 qubits complex64, all in
// one register, 0.42 ms (5.1 TB/s; 0.58 by k_math_gather); by the launch on small ones: 16 qubits in descending
// order 24 us (55 by the gather's loop over 16 runs of bits).
template <typename R>
__global__ __launch_bounds__(kBlock) void k_math_add(const amp_t<R> *__restrict__ src, amp_t<R> *__restrict__ dst,
                                                     uint64_t n_amps, MathAdd A) {
  constexpr int NJ = 8;
  for (uint64_t first = (uint64_t)blockIdx.x * kBlock * NJ + threadIdx.x; first < n_amps; first += (uint64_t)gridDim.x * kBlock * NJ) {
    amp_t<R> v[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      v[j].x = v[j].y = 0;
      if (first + j * kBlock < n_amps) v[j] = src[add_source(A, first + j * kBlock)];
    }
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      if (first + j * kBlock >= n_amps) continue;
      amp_t<R> a;
      a.x = (R)0 + v[j].x;  // newvec starts at 0 (simulator.hpp:239-240): -0 becomes +0
      a.y = (R)0 + v[j].y;
      dst[first + j * kBlock] = a;
    }
  }
}

// In place through LDS tiles (MathTile): a tile is read whole, then its amplitudes take their sources from
// LDS.  Indices whose controls are not set are neither read nor written (but for controls inside the lowest
// 256 bytes), where the gather copies them to the other buffer, and no second buffer is needed.
// 14 controlled multiplications modulo an 8-bit N at 22 qubits complex128: 29 us each as a gather (134 MB),
// 24 us here (67 MB; fixing one index bit leaves half of the memory channels idle, so half the traffic
// is not half the time).  Tiles of 2^8 to 2^11 amplitudes measured the same.
template <typename R, int S>
__global__ __launch_bounds__(kBlock) void k_math_tile(amp_t<R> *__restrict__ psi, MathGather G, MathTile T) {
  constexpr int JB = (sizeof(R) == 4 ? kMathTileBits64 : kMathTileBits128) - 8, NJ = 1 << JB;
  constexpr bool MOD = S == kSrcAddMod || S == kSrcMulMod;
  __shared__ amp_t<R> tile[NJ * kBlock];
  const uint64_t base = scatter_bits(blockIdx.x, T.tile_id) | T.fixed;
  // index and register values are linear in the tile-local bits: a thread's part, and a uniform one
  const uint32_t size = 1u << T.m;
  const uint64_t it = base | scatter_bits(threadIdx.x, T.tile);
  uint64_t rt[3];
#pragma unroll
  for (int r = 0; r < (MOD ? 1 : 3); ++r) rt[r] = r < G.n_regs ? gather_bits(it, G.reg[r]) : 0;
  auto part = [](int j, auto &&of_bit) {  // of the bits above a thread's, uniform
    decltype(of_bit(0)) v = 0;
#pragma unroll
    for (int b = 0; b < JB; ++b)
      if ((j >> b) & 1) v |= of_bit(b);
    return v;
  };
  auto index = [&](int j) { return it | part(j, [&](int b) { return T.step[b]; }); };
  amp_t<R> a[NJ];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    if ((uint32_t)j * kBlock + threadIdx.x < size) a[j] = psi[index(j)];
#pragma unroll
  for (int j = 0; j < NJ; ++j)
    if ((uint32_t)j * kBlock + threadIdx.x < size) tile[j * kBlock + threadIdx.x] = a[j];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < NJ; ++j) {
    const uint32_t l = (uint32_t)j * kBlock + threadIdx.x;
    if (l >= size) continue;
    const uint64_t i = index(j);
    uint32_t s = l;
    amp_t<R> out;
    out.x = 0;
    out.y = 0;
    bool sum = false;
    if ((i & G.cmask) == G.cmask) {
      uint64_t u = rt[0] | part(j, [&](int b) { return T.reg_step[b][0]; });
      s = l & ~T.changed;
      if constexpr (MOD) {
        sum = true;
        const uint32_t N = (uint32_t)G.N;
        if ((uint32_t)u < N) {  // no source from N on
          uint32_t from = residue_source32<S>((uint32_t)u, (uint32_t)G.a, N, (uint32_t)(G.magic >> 32));
          double x = 0.0, y = 0.0;  // newvec starts at 0 and adds in index order (simulator.hpp:239-266)
          do {
            const amp_t<R> b = tile[s | scatter_bits32(from, T.local[0])];
            x += (double)b.x;
            y += (double)b.y;
            from += N;
          } while (from >> G.width[0] == 0);
          out.x = (R)x;
          out.y = (R)y;
        }
      } else {
        uint64_t v = rt[1] | part(j, [&](int b) { return T.reg_step[b][1]; });
        uint64_t w = rt[2] | part(j, [&](int b) { return T.reg_step[b][2]; });
        (void)math_source<S>(G, u, v, w);  // one to one
        const uint64_t values[3] = {u, v, w};
#pragma unroll
        for (int r = 0; r < 3; ++r)
          if (G.moves[r]) s |= scatter_bits32((uint32_t)values[r], T.local[r]);
      }
    }
    if (!sum) {
      const amp_t<R> b = tile[s];
      out.x = (R)0 + b.x;  // newvec starts at 0 (simulator.hpp:239-240): -0 becomes +0
      out.y = (R)0 + b.y;
    }
    psi[i] = out;
  }
}

template <class F>
void with_source(const MathGather &G, F &&go) {
  switch (G.source) {
    case kSrcAddConstant: go(std::integral_constant<int, kSrcAddConstant>{}); break;
    case kSrcSubtract: go(std::integral_constant<int, kSrcSubtract>{}); break;
    case kSrcAdd: go(std::integral_constant<int, kSrcAdd>{}); break;
    case kSrcCompare: go(std::integral_constant<int, kSrcCompare>{}); break;
    case kSrcMulSubtract: go(std::integral_constant<int, kSrcMulSubtract>{}); break;
    case kSrcMulAdd: go(std::integral_constant<int, kSrcMulAdd>{}); break;
    case kSrcAddMod: go(std::integral_constant<int, kSrcAddMod>{}); break;
    default: go(std::integral_constant<int, kSrcMulMod>{}); break;
  }
}

}  // namespace

template <typename R>
void math_gather(const amp_t<R> *src, amp_t<R> *dst, uint64_t n_amps, const MathGather &G, hipStream_t s) {
  const uint64_t n_tiles = (n_amps + (uint64_t(1) << kMathBits) - 1) >> kMathBits;
  with_source(G, [&](auto source) {
    hipLaunchKernelGGL((k_math_gather<R, decltype(source)::value>), dim3((unsigned)n_tiles), dim3(kBlock), 0, s, src,
                       dst, n_amps, n_tiles, G);
  });
  QS_HIP(hipGetLastError());
}

template <typename R>
void math_add(const amp_t<R> *src, amp_t<R> *dst, uint64_t n_amps, const MathAdd &A, hipStream_t s) {
  const uint64_t grid = std::min<uint64_t>(16384, (n_amps + 8 * kBlock - 1) / (8 * kBlock));
  hipLaunchKernelGGL(k_math_add<R>, dim3((unsigned)grid), dim3(kBlock), 0, s, src, dst, n_amps, A);
  QS_HIP(hipGetLastError());
}

template <typename R>
void math_tile(amp_t<R> *psi, uint64_t n_amps, const MathGather &G, const MathTile &T, hipStream_t s) {
  const uint64_t n_tiles = uint64_t(1) << T.outside;
  if (T.m > (sizeof(R) == 4 ? kMathTileBits64 : kMathTileBits128) || (n_tiles << T.m) > n_amps)
    throw ValueError("math_tile: bad tile");
  with_source(G, [&](auto source) {
    hipLaunchKernelGGL((k_math_tile<R, decltype(source)::value>), dim3((unsigned)n_tiles), dim3(kBlock), 0, s, psi, G, T);
  });
  QS_HIP(hipGetLastError());
}

template void math_gather<float>(const float2 *, float2 *, uint64_t, const MathGather &, hipStream_t);
template void math_gather<double>(const double2 *, double2 *, uint64_t, const MathGather &, hipStream_t);
template void math_add<float>(const float2 *, float2 *, uint64_t, const MathAdd &, hipStream_t);
template void math_add<double>(const double2 *, double2 *, uint64_t, const MathAdd &, hipStream_t);
template void math_tile<float>(float2 *, uint64_t, const MathGather &, const MathTile &, hipStream_t);
template void math_tile<double>(double2 *, uint64_t, const MathGather &, const MathTile &, hipStream_t);

}  // namespace dev
}  // namespace qs
