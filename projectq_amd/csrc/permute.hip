// Qubit layout change: dst <- src with its index bits permuted, one pass through LDS tiles (PermTile).
//
// Bound by HBM: one read and one write of the state.  What it takes to get there: segments of at least
// 512 bytes on both sides, 16-byte accesses, eight loads in flight per thread, and an LDS layout under which
// neither the writes in source order nor the reads in destination order meet bank conflicts (a
// permutation reads with strides of powers of two).  With 8-byte accesses, bank conflicts and the smallest tile
// that held both ends' segments, against this: 30 qubits complex64 8.96 -> 4.54 ms (3.8 TB/s), 27 qubits
// complex128 2.5 -> 1.1 ms, 23 qubits complex64 139 -> 26 us.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "kernels.hpp"

namespace qs {
namespace dev {
namespace {

// amplitudes per 16-byte access
template <typename R>
constexpr int kPair = sizeof(R) == 4 ? 2 : 1;
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));

// SCALE: the amplitudes are multiplied by `scale` as well (in FP64, as k_scale_masked does)
template <typename R, bool SCALE>
__global__ __launch_bounds__(kBlock) void k_permute_tiles(const amp_t<R> *__restrict__ src, amp_t<R> *__restrict__ dst,
                                                          uint64_t n_tiles, PermTile P, double scale) {
  constexpr int VN = kPair<R>, V0 = VN == 2 ? 1 : 0, JB = 3, NJ = 1 << JB;  // tile bits V0.. thread, V0 + 8.. turn
  extern __shared__ __align__(16) unsigned char smem[];
  amp_t<R> *tile = reinterpret_cast<amp_t<R> *>(smem);
  const uint32_t units = (1u << P.m) / VN;
  // everything is linear over GF(2): a thread's own part once, and a uniform part per turn
  uint64_t src_t = 0, dst_t = 0;
  uint32_t in_t = 0, out_t = 0;
  for (uint32_t b = 0; b < 8 && V0 + b < P.m; ++b)
    if ((threadIdx.x >> b) & 1) {
      src_t |= uint64_t(1) << P.src_pos[V0 + b];
      dst_t |= uint64_t(1) << P.dst_pos[V0 + b];
      in_t ^= P.slot_src[V0 + b];
      out_t ^= P.slot_dst[V0 + b];
    }
  uint64_t src_j[JB], dst_j[JB];
  uint32_t in_j[JB], out_j[JB];
#pragma unroll
  for (uint32_t b = 0; b < JB; ++b) {
    const bool have = V0 + 8 + b < P.m;
    src_j[b] = have ? uint64_t(1) << P.src_pos[V0 + 8 + b] : 0;
    dst_j[b] = have ? uint64_t(1) << P.dst_pos[V0 + 8 + b] : 0;
    in_j[b] = have ? P.slot_src[V0 + 8 + b] : 0;
    out_j[b] = have ? P.slot_dst[V0 + 8 + b] : 0;
  }
  auto of = [](int j, const auto *bits) {
    auto v = bits[0] & 0;
#pragma unroll
    for (int b = 0; b < JB; ++b)
      if ((j >> b) & 1) v ^= bits[b];
    return v;
  };
  auto scaled = [&](R v) { return SCALE ? (R)((double)v * scale) : v; };
  for (uint64_t id = blockIdx.x; id < n_tiles; id += gridDim.x) {
    uint64_t sb = src_t, db = dst_t;
    for (uint32_t i = 0; i < P.n_outer; ++i) {
      const uint64_t bit = (id >> i) & 1u;
      sb |= bit << P.outer_src[i];
      db |= bit << P.outer_dst[i];
    }
    if constexpr (VN == 2) {
      const uint32_t pair = P.slot_dst[0];
      f32x4 v[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if ((uint32_t)j * kBlock + threadIdx.x < units)
          v[j] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(src + (sb ^ of(j, src_j))));
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if ((uint32_t)j * kBlock + threadIdx.x < units) {
          const uint32_t s = in_t ^ of(j, in_j);
          tile[s] = amp_t<R>{v[j].x, v[j].y};
          tile[s ^ 1u] = amp_t<R>{v[j].z, v[j].w};
        }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if ((uint32_t)j * kBlock + threadIdx.x < units) {
          const uint32_t s = out_t ^ of(j, out_j);
          const amp_t<R> a = tile[s], b = tile[s ^ pair];
          f32x4 o = {scaled(a.x), scaled(a.y), scaled(b.x), scaled(b.y)};
          __builtin_nontemporal_store(o, reinterpret_cast<f32x4 *>(dst + (db ^ of(j, dst_j))));
        }
    } else {
      f64x2 v[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if ((uint32_t)j * kBlock + threadIdx.x < units)
          v[j] = __builtin_nontemporal_load(reinterpret_cast<const f64x2 *>(src + (sb ^ of(j, src_j))));
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if ((uint32_t)j * kBlock + threadIdx.x < units)
          reinterpret_cast<f64x2 *>(tile)[in_t ^ of(j, in_j)] = v[j];
      __syncthreads();
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        if ((uint32_t)j * kBlock + threadIdx.x < units) {
          const f64x2 a = reinterpret_cast<const f64x2 *>(tile)[out_t ^ of(j, out_j)];
          f64x2 o = {scaled(a.x), scaled(a.y)};
          __builtin_nontemporal_store(o, reinterpret_cast<f64x2 *>(dst + (db ^ of(j, dst_j))));
        }
    }
    __syncthreads();  // the tile is free for the next turn
  }
}

}  // namespace

template <typename R>
void permute_tiles(const amp_t<R> *src, amp_t<R> *dst, uint64_t n_amps, const PermTile &P, double scale, hipStream_t s) {
  // a turn of 256 threads takes 2^8 units of 16 bytes, 8 turns at most; a pair needs one tile bit
  const uint32_t most = sizeof(R) == 4 ? 12 : 11;
  if (P.m > most || P.m < (sizeof(R) == 4 ? 1u : 0u) || (uint64_t(1) << P.m) > n_amps || P.m + P.n_outer > 64 ||
      (P.m > 0 && (P.src_pos[0] != 0 || P.dst_pos[0] != 0)))
    throw ValueError("permute_tiles: bad tile");
  const uint64_t n_tiles = n_amps >> P.m;
  const uint64_t grid = std::min<uint64_t>(n_tiles, 16384);
  auto go = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3((unsigned)grid), dim3(kBlock), sizeof(amp_t<R>) << P.m, s, src, dst, n_tiles, P, scale);
  };
  if (scale == 1.0) go(k_permute_tiles<R, false>);
  else go(k_permute_tiles<R, true>);
  QS_HIP(hipGetLastError());
}

template void permute_tiles<float>(const float2 *, float2 *, uint64_t, const PermTile &, double, hipStream_t);
template void permute_tiles<double>(const double2 *, double2 *, uint64_t, const PermTile &, double, hipStream_t);

}  // namespace dev
}  // namespace qs
