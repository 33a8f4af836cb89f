// Device code and launchers of the tile passes (k_tile_pass, k_tile_pass_pf, k_batch_tile_pass).
// The templates compile for minutes, so each instantiation has a source file of its own
// (tile_*.hip) and they build in parallel.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdlib>
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "layout.hpp"

namespace qs {
namespace dev {

// set the dynamic-LDS limit of every tile-pass kernel (call before any graph capture)
void prepare_tile_kernels();

// Launchers of one (state precision, register bits) combination, explicitly instantiated by
// tile_c64_rb4.hip, tile_c64_rb5.hip, tile_c128_rb4.hip and tile_c128_rb5.hip; the pipelined kernel
// (complex64, RB = 4) is in tile_pf.hip.
template <typename R, int RB>
void launch_tile_pass(amp_t<R> *psi, uint64_t n_tiles, const TilePass &P, const TileStage *d_stages,
                      const RegOp *d_rops, const TileOp *d_tops, const amp_t<R> *d_mats, TileForms forms,
                      hipStream_t s);
// passes with phase ops: tiles of a multiple of kStreamChunk * kBlock 16-byte vectors, RB = 4
// (tile_c64_phase.hip, tile_c128_phase.hip)
void launch_tile_pass_phase(float2 *psi, uint64_t n_tiles, const TilePass &P, const TileStage *d_stages,
                            const RegOp *d_rops, const TileOp *d_tops, const float2 *d_mats, unsigned grid, size_t lds,
                            hipStream_t s);
void launch_tile_pass_phase(double2 *psi, uint64_t n_tiles, const TilePass &P, const TileStage *d_stages,
                            const RegOp *d_rops, const TileOp *d_tops, const double2 *d_mats, unsigned grid, size_t lds,
                            hipStream_t s);
void prepare_tile_kernels_phase_c64();
void prepare_tile_kernels_phase_c128();
template <typename R, int RB>
void launch_batch_tile_pass(amp_t<R> *psi, const BatchJob *jobs, const uint32_t *block_job, uint32_t n_blocks,
                            uint32_t max_t, const TileStage *stages, const RegOp *rops, const TileOp *tops,
                            const amp_t<R> *mats, bool two_qubit_ops, hipStream_t s);
template <typename R, int RB>
void prepare_tile_kernels_of();
// false where the pipelined kernel does not apply
bool launch_tile_pass_pf(float2 *psi, uint64_t n_tiles, const TilePass &P, const TileStage *d_stages,
                         const RegOp *d_rops, const TileOp *d_tops, const float2 *d_mats, bool two_qubit_ops,
                         unsigned grid, size_t lds, hipStream_t s);
void prepare_tile_kernels_pf();

#ifdef QS_TILE_KERNELS
namespace {

__device__ __forceinline__ uint64_t insert_one_zero(uint64_t g, int p) {
  return ((g >> p) << (p + 1)) | (g & ((uint64_t(1) << p) - 1));
}

// largest dynamic LDS of a tile kernel: the biggest tile plus the biggest segment table
template <typename R>
constexpr int kTileLdsMax = int(sizeof(amp_t<R>) << kTileMaxBits) + int(sizeof(uint64_t) << kTileMaxHigh);

template <class K>
void allow_lds(K kernel, int bytes) {
  QS_HIP(hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes));
}

template <typename R>
__device__ __forceinline__ uint32_t slot(uint32_t x);
template <>
__device__ __forceinline__ uint32_t slot<float>(uint32_t x) {
  return lds_slot_c64(x);
}
template <>
__device__ __forceinline__ uint32_t slot<double>(uint32_t x) {
  return lds_slot_c128(x);
}
// Both swizzles are linear over GF(2): for indices a, b without common bits,
// slot(a | b) = slot(a) ^ slot(b).  The kernels use this to address a group of amplitudes with
// one XOR per access: the per-thread part slot(lb) is computed once and the per-amplitude parts
// slot(offset) are uniform over the workgroup.  slot_bytes gives the byte offset in the tile.
template <typename R>
__device__ __forceinline__ uint32_t slot_bytes(uint32_t x) {
  return slot<R>(x) * (uint32_t)sizeof(amp_t<R>);
}
// Tiles are addressed by raw LDS byte address.  The tile kernels declare no static LDS, so the
// dynamic buffer (and the tile) starts at LDS address 0 and base ^ offset == base + offset; the
// XOR-composed offsets then need no add before the ds instruction.
template <typename T>
using lds_ptr = __attribute__((address_space(3))) T *;
__device__ __forceinline__ uint32_t lds_address(const void *p) {
  return (uint32_t)(uintptr_t)(lds_ptr<const char>)(p);
}
// T is a builtin vector type (16-byte tile streaming); amplitudes go through lds_*_amp.
template <typename T>
__device__ __forceinline__ T lds_load(uint32_t lds_byte_addr) {
  return *(lds_ptr<const T>)(lds_byte_addr);
}
template <typename T>
__device__ __forceinline__ void lds_store(uint32_t lds_byte_addr, const T &v) {
  *(lds_ptr<T>)(lds_byte_addr) = v;
}
template <typename R>
using re2_t = R __attribute__((ext_vector_type(2)));
template <typename R>
__device__ __forceinline__ amp_t<R> lds_load_amp(uint32_t lds_byte_addr) {
  const re2_t<R> v = lds_load<re2_t<R>>(lds_byte_addr);
  amp_t<R> a;
  a.x = v.x;
  a.y = v.y;
  return a;
}
template <typename R>
__device__ __forceinline__ void lds_store_amp(uint32_t lds_byte_addr, const amp_t<R> &a) {
  re2_t<R> v;
  v.x = a.x;
  v.y = a.y;
  lds_store<re2_t<R>>(lds_byte_addr, v);
}

// One TileOp of any width straight on the LDS tile (NT threads per workgroup).
template <typename R, int K, int NT = kBlock>
__device__ __forceinline__ void tile_apply(amp_t<R> *__restrict__ tile, uint32_t t,
                                           const TileOp *__restrict__ op,
                                           const amp_t<R> *__restrict__ m) {
  constexpr int D = 1 << K;
  const uint32_t nfixed = op->nfixed, lcmask = op->lcmask;
  const uint32_t ngroups = 1u << (t - nfixed);
  for (uint32_t g = threadIdx.x; g < ngroups; g += NT) {
    uint32_t lb = g;
    for (uint32_t i = 0; i < nfixed; ++i) {
      const uint32_t p = op->fixed[i];
      lb = ((lb >> p) << (p + 1)) | (lb & ((1u << p) - 1));
    }
    lb |= lcmask;
    uint32_t sb = lds_address(tile) + slot_bytes<R>(lb);
    asm volatile("" : "+v"(sb));
    R vr[D], vi[D];
#pragma unroll
    for (int j = 0; j < D; ++j) {
      const amp_t<R> a = lds_load_amp<R>(sb ^ slot_bytes<R>(op->off[j]));
      vr[j] = a.x;
      vi[j] = a.y;
    }
    asm volatile("" : "+v"(sb));
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
      lds_store_amp<R>(sb ^ slot_bytes<R>(op->off[r]), o);
    }
  }
}

// ---- register-stage ops: NR = 2^RB amplitudes of one thread, register index bit i <-> stage
// bit i.  C is the op's control among the register bits (-1: none); it is a compile-time
// constant, so a controlled op touches only the indices with bit C set and a controlled X is a
// renaming of registers.
//
// Controls on tile bits outside the register bits hold for some threads and not others.  They do
// not branch: ops with such controls run the PRED form, in which every lane runs the op and lanes
// whose controls fail (`act` false) apply the identity -- the matrix is blended with the
// identity, or the results are selected.  With no divergent branch in the op loop the
// op dispatch stays uniform control flow, which the compiler lays out without copying the
// amplitude registers at every merge (with -structurizecfg-skip-uniform-regions).
__host__ __device__ constexpr bool reg_ctrl_ok(int i, int C) { return C < 0 || ((i >> (C < 0 ? 0 : C)) & 1); }

template <typename R>
__device__ __forceinline__ R blend(bool act, R v, R id) { return act ? v : id; }

template <typename R, int RB, bool PRED, int C, int B>
__device__ __forceinline__ void rop_general(R *vr, R *vi, const amp_t<R> *__restrict__ m, bool act) {
  R ar = m[0].x, ai = m[0].y, br = m[1].x, bi = m[1].y;
  R cr = m[2].x, ci = m[2].y, dr = m[3].x, di = m[3].y;
  if constexpr (PRED) {
    ar = blend<R>(act, ar, 1), ai = blend<R>(act, ai, 0), br = blend<R>(act, br, 0), bi = blend<R>(act, bi, 0);
    cr = blend<R>(act, cr, 0), ci = blend<R>(act, ci, 0), dr = blend<R>(act, dr, 1), di = blend<R>(act, di, 0);
  }
#pragma unroll
  for (int i = 0; i < (1 << RB); ++i) {
    if ((i & (1 << B)) || !reg_ctrl_ok(i, C)) continue;
    const int j = i | (1 << B);
    const R xr = vr[i], xi = vi[i], yr = vr[j], yi = vi[j];
    vr[i] = fma(ar, xr, fma(-ai, xi, fma(br, yr, -bi * yi)));
    vi[i] = fma(ar, xi, fma(ai, xr, fma(br, yi, bi * yr)));
    vr[j] = fma(cr, xr, fma(-ci, xi, fma(dr, yr, -di * yi)));
    vi[j] = fma(cr, xi, fma(ci, xr, fma(dr, yi, di * yr)));
  }
}
template <typename R, int RB, bool PRED, int C, int B>
__device__ __forceinline__ void rop_real(R *vr, R *vi, const amp_t<R> *__restrict__ m, bool act) {
  R a = m[0].x, b = m[1].x, c = m[2].x, d = m[3].x;
  if constexpr (PRED) a = blend<R>(act, a, 1), b = blend<R>(act, b, 0), c = blend<R>(act, c, 0), d = blend<R>(act, d, 1);
#pragma unroll
  for (int i = 0; i < (1 << RB); ++i) {
    if ((i & (1 << B)) || !reg_ctrl_ok(i, C)) continue;
    const int j = i | (1 << B);
    const R xr = vr[i], xi = vi[i], yr = vr[j], yi = vi[j];
    vr[i] = fma(a, xr, b * yr);
    vi[i] = fma(a, xi, b * yi);
    vr[j] = fma(c, xr, d * yr);
    vi[j] = fma(c, xi, d * yi);
  }
}
template <typename R, int RB, bool PRED, int C, int B>
__device__ __forceinline__ void rop_diag(R *vr, R *vi, const amp_t<R> *__restrict__ m, bool act) {
  R ar = m[0].x, ai = m[0].y, dr = m[3].x, di = m[3].y;
  if constexpr (PRED) ar = blend<R>(act, ar, 1), ai = blend<R>(act, ai, 0), dr = blend<R>(act, dr, 1), di = blend<R>(act, di, 0);
#pragma unroll
  for (int i = 0; i < (1 << RB); ++i) {
    if (!reg_ctrl_ok(i, C)) continue;
    const R fr = (i & (1 << B)) ? dr : ar, fi = (i & (1 << B)) ? di : ai;
    const R xr = vr[i], xi = vi[i];
    vr[i] = fma(fr, xr, -fi * xi);
    vi[i] = fma(fr, xi, fi * xr);
  }
}
template <typename R, int RB, bool PRED, int C, int B>
__device__ __forceinline__ void rop_anti(R *vr, R *vi, const amp_t<R> *__restrict__ m, bool act) {
  const R br = m[1].x, bi = m[1].y, cr = m[2].x, ci = m[2].y;
#pragma unroll
  for (int i = 0; i < (1 << RB); ++i) {
    if ((i & (1 << B)) || !reg_ctrl_ok(i, C)) continue;
    const int j = i | (1 << B);
    const R xr = vr[i], xi = vi[i], yr = vr[j], yi = vi[j];
    const R nr_i = fma(br, yr, -bi * yi), ni_i = fma(br, yi, bi * yr);
    const R nr_j = fma(cr, xr, -ci * xi), ni_j = fma(cr, xi, ci * xr);
    vr[i] = PRED ? blend<R>(act, nr_i, xr) : nr_i;
    vi[i] = PRED ? blend<R>(act, ni_i, xi) : ni_i;
    vr[j] = PRED ? blend<R>(act, nr_j, yr) : nr_j;
    vi[j] = PRED ? blend<R>(act, ni_j, yi) : ni_j;
  }
}
template <typename R, int RB, bool PRED, int C, int B>
__device__ __forceinline__ void rop_x(R *vr, R *vi, const amp_t<R> *__restrict__, bool act) {
  if constexpr (PRED) {
#pragma unroll
    for (int i = 0; i < (1 << RB); ++i) {
      if ((i & (1 << B)) || !reg_ctrl_ok(i, C)) continue;
      const int j = i | (1 << B);
      const R xr = vr[i], xi = vi[i], yr = vr[j], yi = vi[j];
      vr[i] = blend<R>(act, yr, xr);
      vi[i] = blend<R>(act, yi, xi);
      vr[j] = blend<R>(act, xr, yr);
      vi[j] = blend<R>(act, xi, yi);
    }
    return;
  }
#pragma unroll
  for (int i = 0; i < (1 << RB); ++i) {
    if ((i & (1 << B)) || !reg_ctrl_ok(i, C)) continue;
    const int j = i | (1 << B);
    const R xr = vr[i], xi = vi[i];
    vr[i] = vr[j];
    vi[i] = vi[j];
    vr[j] = xr;
    vi[j] = xi;
  }
}
// Z (diag(1, -1)): the amplitudes with bit B set change sign, in place (an XOR of the sign bit;
// predicated lanes XOR with zero).  A CNOT between 1-qubit gates on its target reaches the tile
// kernels as H, controlled Z, H with the H's merged into those gates (cnot_to_cz in planner.cpp).
template <typename R>
__device__ __forceinline__ R flip_sign(R x, bool act) {
  if constexpr (sizeof(R) == 4) return __uint_as_float(__float_as_uint(x) ^ (act ? 0x80000000u : 0u));
  else return __longlong_as_double(__double_as_longlong(x) ^ (act ? (1ll << 63) : 0ll));
}
template <typename R, int RB, bool PRED, int C, int B>
__device__ __forceinline__ void rop_z(R *vr, R *vi, const amp_t<R> *__restrict__, bool act) {
#pragma unroll
  for (int i = 0; i < (1 << RB); ++i) {
    if (!(i & (1 << B)) || !reg_ctrl_ok(i, C)) continue;
    vr[i] = flip_sign<R>(vr[i], PRED ? act : true);
    vi[i] = flip_sign<R>(vi[i], PRED ? act : true);
  }
}
template <typename R, int RB, bool PRED, int C, int B0, int B1>
__device__ __forceinline__ void rop_general2(R *vr, R *vi, const amp_t<R> *__restrict__ m, bool act) {
  R mr[16], mi[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) {
    mr[k] = m[k].x;
    mi[k] = m[k].y;
    if constexpr (PRED) mr[k] = blend<R>(act, mr[k], (k % 5) == 0 ? R(1) : R(0)), mi[k] = blend<R>(act, mi[k], 0);
  }
#pragma unroll
  for (int i = 0; i < (1 << RB); ++i) {
    if ((i & ((1 << B0) | (1 << B1))) || !reg_ctrl_ok(i, C)) continue;
    const int idx[4] = {i, i | (1 << B0), i | (1 << B1), i | (1 << B0) | (1 << B1)};
    R xr[4], xi[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      xr[c] = vr[idx[c]];
      xi[c] = vi[idx[c]];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      R sr = 0, si = 0;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        sr = fma(mr[r * 4 + c], xr[c], fma(-mi[r * 4 + c], xi[c], sr));
        si = fma(mr[r * 4 + c], xi[c], fma(mi[r * 4 + c], xr[c], si));
      }
      vr[idx[r]] = sr;
      vi[idx[r]] = si;
    }
  }
}
template <typename R, int RB, bool PRED, int C, int B0, int B1>
__device__ __forceinline__ void rop_diag2(R *vr, R *vi, const amp_t<R> *__restrict__ m, bool act) {
  R fr[4], fi[4];
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    fr[s] = m[s * 5].x;  // diagonal element s of the 4x4 matrix
    fi[s] = m[s * 5].y;
    if constexpr (PRED) fr[s] = blend<R>(act, fr[s], 1), fi[s] = blend<R>(act, fi[s], 0);
  }
#pragma unroll
  for (int i = 0; i < (1 << RB); ++i) {
    if (!reg_ctrl_ok(i, C)) continue;
    const int s = ((i >> B0) & 1) | (((i >> B1) & 1) << 1);
    const R xr = vr[i], xi = vi[i];
    vr[i] = fma(fr[s], xr, -fi[s] * xi);
    vi[i] = fma(fr[s], xi, fi[s] * xr);
  }
}

// Dispatch on the kind, register bits and register control of an op (cb = 1 + control bit, 0 =
// none), in one function so that the amplitude registers stay in registers.  Combinations the
// planner never emits (a control on a target, bits >= RB) do nothing.
#define QS_R1(FN, C, B)                                          \
  if constexpr ((B) < RB && (C) < RB && (C) != (B)) FN<R, RB, PRED, C, B>(vr, vi, m, act);
#define QS_R1C(FN, B)                                            \
  switch (cb) {                                                  \
    case 0: QS_R1(FN, -1, B) break;                              \
    case 1: QS_R1(FN, 0, B) break;                               \
    case 2: QS_R1(FN, 1, B) break;                               \
    case 3: QS_R1(FN, 2, B) break;                               \
    case 4: QS_R1(FN, 3, B) break;                               \
    default: QS_R1(FN, 4, B) break;                              \
  }
#define QS_R1B(FN)                                               \
  switch (b0) {                                                  \
    case 0: QS_R1C(FN, 0) break;                                 \
    case 1: QS_R1C(FN, 1) break;                                 \
    case 2: QS_R1C(FN, 2) break;                                 \
    case 3: QS_R1C(FN, 3) break;                                 \
    default: QS_R1C(FN, 4) break;                                \
  }
#define QS_R2(FN, C, B0, B1)                                                            \
  if constexpr ((B1) < RB && (C) < RB && (C) != (B0) && (C) != (B1)) FN<R, RB, PRED, C, B0, B1>(vr, vi, m, act);
#define QS_R2C(FN, B0, B1)                                       \
  switch (cb) {                                                  \
    case 0: QS_R2(FN, -1, B0, B1) break;                         \
    case 1: QS_R2(FN, 0, B0, B1) break;                          \
    case 2: QS_R2(FN, 1, B0, B1) break;                          \
    case 3: QS_R2(FN, 2, B0, B1) break;                          \
    case 4: QS_R2(FN, 3, B0, B1) break;                          \
    default: QS_R2(FN, 4, B0, B1) break;                         \
  }
#define QS_R2B(FN)                                               \
  switch (b0 * 8 + b1) {                                         \
    case 0 * 8 + 1: QS_R2C(FN, 0, 1) break;                      \
    case 0 * 8 + 2: QS_R2C(FN, 0, 2) break;                      \
    case 0 * 8 + 3: QS_R2C(FN, 0, 3) break;                      \
    case 1 * 8 + 2: QS_R2C(FN, 1, 2) break;                      \
    case 1 * 8 + 3: QS_R2C(FN, 1, 3) break;                      \
    case 2 * 8 + 3: QS_R2C(FN, 2, 3) break;                      \
    case 0 * 8 + 4: QS_R2C(FN, 0, 4) break;                      \
    case 1 * 8 + 4: QS_R2C(FN, 1, 4) break;                      \
    case 2 * 8 + 4: QS_R2C(FN, 2, 4) break;                      \
    default: QS_R2C(FN, 3, 4) break;                             \
  }

// TWO = false: a kernel for passes with no 2-qubit register op (the host picks it per pass); the
// dispatch then holds only the 1-qubit forms, and the register allocator works on far fewer arms.
template <typename R, int RB, bool PRED, bool TWO = true>
__device__ __forceinline__ void reg_op(uint32_t code, R *vr, R *vi, const amp_t<R> *__restrict__ m, bool act) {
  uint32_t kind = (code >> 8) & 15u;
  const uint32_t b0 = code & 15u, b1 = (code >> 4) & 15u, cb = code >> 12;
  (void)b1;
  // the full kernel runs a Z op as the diagonal op it is (its matrix is diag(1, -1)): a set of Z
  // arms beside the 2-qubit ones measured 4% slower on every pass
  if constexpr (TWO) kind = kind == kOp1Z ? kOp1Diag : kind;
  switch (kind) {
    case kOp1General: QS_R1B(rop_general) break;
    case kOp1Real: QS_R1B(rop_real) break;
    case kOp1Diag: QS_R1B(rop_diag) break;
    case kOp1Anti: QS_R1B(rop_anti) break;
    case kOp1X: QS_R1B(rop_x) break;
    case kOp1Z:
      if constexpr (!TWO) { QS_R1B(rop_z) }
      break;
    default:
      if constexpr (TWO) {
        if (kind == kOp2General) QS_R2B(rop_general2)
        else QS_R2B(rop_diag2)
      }
      break;
  }
}
#undef QS_R1
#undef QS_R1C
#undef QS_R1B
#undef QS_R2
#undef QS_R2C
#undef QS_R2B

// Expanded by index: as a loop over i with a test of the mask it was simplified before it was unrolled, and
// some amplitudes ended up in scratch memory.
template <typename R, int I, int S>
__device__ __forceinline__ void phase_one(R *vr, R *vi, R fr, R fi) {
  if constexpr ((I & S) == S) {
    const R xr = vr[I], xi = vi[I];
    vr[I] = fma(fr, xr, -fi * xi);
    vi[I] = fma(fr, xi, fi * xr);
  }
}
template <typename R, int S, int... I>
__device__ __forceinline__ void rop_phase(R *vr, R *vi, R fr, R fi, std::integer_sequence<int, I...>) {
  (phase_one<R, I, S>(vr, vi, fr, fi), ...);
}
// A group of phases.  A phase gate (a factor where some bits are all set) costs a predicated complex
// product on one number per thread, and the amplitudes are touched once per group: as a diagonal op each
// of them costs 64 FMAs and, like every op, moves all amplitude registers at the end of its arm.  27 qubits
// complex128, a QFT and 5 layers of rotations: the first pass (189 of 201 ops are controlled phases)
// 6.6 -> 3.2 ms, the circuit 8 passes of 2.8 ms -> 7 of 2.3 ms.  The factors of consecutive records load
// together (unrolled); one record at a time the first pass took 5.4 ms.
template <typename R, int RB>
__device__ __forceinline__ void phase_group(const RegOp *__restrict__ op, uint64_t base, uint32_t lb, R *vr, R *vi,
                                            const amp_t<R> *__restrict__ mats) {
  static_assert(RB == 4, "the masks below");
  using Amps = std::make_integer_sequence<int, 1 << RB>;
  const RegOp *__restrict__ terms = op + 1;
  const amp_t<R> *__restrict__ f = mats + op->mat;
  const uint32_t n = op->rcmask;
  R x = 1, y = 0;
#pragma unroll 4
  for (uint32_t i = 0; i < n; ++i) {
    const uint64_t gc = terms[i].gcmask;
    const uint32_t lc = terms[i].lcmask;
    const bool act = (base & gc) == gc && (lb & lc) == lc;
    const R fr = blend<R>(act, f[i].x, 1), fi = blend<R>(act, f[i].y, 0), old = x;
    x = fma(fr, old, -fi * y);
    y = fma(fr, y, fi * old);
  }
  switch (op->code & 15u) {
    case 0: rop_phase<R, 0>(vr, vi, x, y, Amps{}); break;
    case 1: rop_phase<R, 1>(vr, vi, x, y, Amps{}); break;
    case 2: rop_phase<R, 2>(vr, vi, x, y, Amps{}); break;
    case 3: rop_phase<R, 3>(vr, vi, x, y, Amps{}); break;
    case 4: rop_phase<R, 4>(vr, vi, x, y, Amps{}); break;
    case 5: rop_phase<R, 5>(vr, vi, x, y, Amps{}); break;
    case 6: rop_phase<R, 6>(vr, vi, x, y, Amps{}); break;
    case 7: rop_phase<R, 7>(vr, vi, x, y, Amps{}); break;
    case 8: rop_phase<R, 8>(vr, vi, x, y, Amps{}); break;
    case 9: rop_phase<R, 9>(vr, vi, x, y, Amps{}); break;
    case 10: rop_phase<R, 10>(vr, vi, x, y, Amps{}); break;
    case 11: rop_phase<R, 11>(vr, vi, x, y, Amps{}); break;
    case 12: rop_phase<R, 12>(vr, vi, x, y, Amps{}); break;
    case 13: rop_phase<R, 13>(vr, vi, x, y, Amps{}); break;
    case 14: rop_phase<R, 14>(vr, vi, x, y, Amps{}); break;
    default: rop_phase<R, 15>(vr, vi, x, y, Amps{}); break;
  }
}

// One register op: global controls are uniform over the block (a branch); tile-bit controls are
// per lane (the predicated form).
template <typename R, int RB, bool TWO = true>
__device__ __forceinline__ void reg_apply(const RegOp *__restrict__ op, uint64_t base, uint32_t lb, R *vr, R *vi,
                                          const amp_t<R> *__restrict__ mats) {
  const uint64_t gc = op->gcmask;
  const uint32_t lc = op->lcmask;
  if ((base & gc) == gc) {
    if (lc == 0) reg_op<R, RB, false, TWO>(op->code, vr, vi, mats + op->mat, true);
    else reg_op<R, RB, true, TWO>(op->code, vr, vi, mats + op->mat, (lb & lc) == lc);
  }
}

// TURN ops per turn of the op loop (with phases always 1).  With 2 the register allocator moves the amplitudes between
// register sets once per turn rather than once per op (worth about 2% on the pass kernel), at
// the price of a second copy of the op dispatch; kernels off the hot path use 1.
template <typename R, int RB, int TURN, int NT = kBlock, bool TWO = true, bool PH = false>
__device__ __forceinline__ void reg_stage(amp_t<R> *__restrict__ tile, uint32_t t, uint64_t base,
                                          const TileStage *__restrict__ st,
                                          const RegOp *__restrict__ rops,
                                          const amp_t<R> *__restrict__ mats) {
  constexpr int NR = 1 << RB;
  uint32_t soff[NR];  // byte offset (swizzled) of register i relative to the group's base
#pragma unroll
  for (int i = 0; i < NR; ++i) soff[i] = st->soff[i];
  const uint32_t ngroups = 1u << (t - RB);
  const uint32_t ob = st->begin, oe = st->end;
  for (uint32_t g = threadIdx.x; g < ngroups; g += NT) {
    uint32_t lb = g;
#pragma unroll
    for (int b = 0; b < RB; ++b) {
      const uint32_t p = st->fixed[b];
      lb = ((lb >> p) << (p + 1)) | (lb & ((1u << p) - 1));
    }
    uint32_t sb = lds_address(tile) + slot_bytes<R>(lb);
    asm volatile("" : "+v"(sb));  // keeps the address math at one XOR per access
    R vr[NR], vi[NR];
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      const amp_t<R> a = lds_load_amp<R>(sb ^ soff[i]);
      vr[i] = a.x;
      vi[i] = a.y;
    }
    if constexpr (PH) {
      for (uint32_t o = ob; o < oe; ++o) {
        const RegOp *op = rops + o;
        if ((op->code >> 8 & 15u) == kOpPhases) {
          phase_group<R, RB>(op, base, lb, vr, vi, mats);
          o += op->rcmask;
        } else {
          reg_apply<R, RB, TWO>(op, base, lb, vr, vi, mats);
        }
      }
    } else {
      for (uint32_t o = ob; o < oe; o += TURN) {
        reg_apply<R, RB, TWO>(rops + o, base, lb, vr, vi, mats);
        if constexpr (TURN == 2) {
          if (o + 1 < oe) reg_apply<R, RB, TWO>(rops + o + 1, base, lb, vr, vi, mats);
        }
      }
    }
    // Recompute the LDS addresses for the write-back instead of keeping 2^RB of them live across
    // the ops (the empty asm makes sb opaque to common-subexpression elimination).
    asm volatile("" : "+v"(sb));
#pragma unroll
    for (int i = 0; i < NR; ++i) {
      amp_t<R> a;
      a.x = vr[i];
      a.y = vi[i];
      lds_store_amp<R>(sb ^ soff[i], a);
    }
  }
}

// 16-byte vectors of amplitudes used to stream tiles (2 x complex64 or 1 x complex128)
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef double f64x2 __attribute__((ext_vector_type(2)));
template <typename R>
struct Vec16 {
  using type = f32x4;
  static constexpr int n = 2;
};
template <>
struct Vec16<double> {
  using type = f64x2;
  static constexpr int n = 1;
};

// The LDS side of tile streaming: one 16-byte global vector holds one complex128 amplitude or
// the complex64 pair (l, l + 1).  The swizzle keeps such a pair adjacent but may swap it
// (slot(l + 1) = slot(l) ^ 1), so complex64 pairs move as two 8-byte accesses.
template <typename R>
__device__ __forceinline__ void tile_put16(uint32_t addr, const typename Vec16<R>::type &v) {
  if constexpr (sizeof(R) == 4) {
    re2_t<float> a, b;
    a.x = v.x;
    a.y = v.y;
    b.x = v.z;
    b.y = v.w;
    lds_store<re2_t<float>>(addr, a);
    lds_store<re2_t<float>>(addr ^ 8u, b);
  } else {
    lds_store<typename Vec16<R>::type>(addr, v);
  }
}
// The read of a 16-byte vector for the store, which may relabel qubits: the pair (l, l + 1) of the stored tile comes
// from computed-tile slots addr and addr ^ pair (pair = the slot bytes of the partner's bit).
template <typename R>
__device__ __forceinline__ typename Vec16<R>::type tile_get16p(uint32_t addr, uint32_t pair) {
  if constexpr (sizeof(R) == 4) {
    const re2_t<float> a = lds_load<re2_t<float>>(addr), b = lds_load<re2_t<float>>(addr ^ pair);
    typename Vec16<R>::type v;
    v.x = a.x;
    v.y = a.y;
    v.z = b.x;
    v.w = b.y;
    return v;
  } else {
    return lds_load<typename Vec16<R>::type>(addr);
  }
}

// Streaming accesses of the tile passes: every amplitude is read and written exactly once per
// pass, so the accesses carry the non-temporal hint unless QS_TILE_TEMPORAL is defined.
template <typename V>
__device__ __forceinline__ V stream_load(const V *p) {
#ifdef QS_TILE_TEMPORAL
  return *p;
#else
  return __builtin_nontemporal_load(p);
#endif
}
template <typename V>
__device__ __forceinline__ void stream_store(V *p, const V &v) {
#ifdef QS_TILE_TEMPORAL
  *p = v;
#else
  __builtin_nontemporal_store(v, p);
#endif
}

// Global index of the first amplitude of tile `tix`: the low L bits and the high tile positions
// (ascending, all >= L) are zero and the remaining bits hold tix.  The loop has a fixed trip count
// so the positions are read at static offsets of the kernel argument (scalar loads).
__device__ __forceinline__ uint64_t tile_base(uint64_t tix, const TilePass &P) {
  uint64_t g = tix << P.L;
#pragma unroll
  for (int b = 0; b < kTileMaxHigh; ++b)
    if (b < (int)P.h) g = insert_one_zero(g, (int)P.hpos[b]);
  return g;
}

// 16-byte accesses each thread keeps in flight while streaming a tile.
constexpr int kStreamChunk = 8;

// Tile-local index of the computed tile that index x of the stored tile takes (the relabelling of
// P.sperm; x itself when there is none).  GF(2)-linear in x.
__device__ __forceinline__ uint32_t store_source(uint32_t x, const TilePass &P) {
  uint32_t y = 0;
#pragma unroll
  for (int b = 0; b < kTileMaxBits; ++b)
    if (b < (int)P.t) y |= ((x >> b) & 1u) << P.sperm[b];
  return y;
}

// The stages of a pass on one tile resident in LDS, a workgroup barrier after each.
template <typename R, int RB, int TURN, int NT = kBlock, bool TWO = true, bool PH = false>
__device__ __forceinline__ void run_stages(amp_t<R> *__restrict__ tile, uint32_t t, uint64_t base, uint32_t n_stages,
                                           const TileStage *__restrict__ stages, const RegOp *__restrict__ rops,
                                           const TileOp *__restrict__ tops, const amp_t<R> *__restrict__ mats) {
  for (uint32_t s = 0; s < n_stages; ++s) {
    const TileStage *st = stages + s;
    if (st->kind == kStageRegisters) {
      reg_stage<R, RB, TURN, NT, TWO, PH>(tile, t, base, st, rops, mats);
    } else {
      const TileOp *op = tops + st->begin;
      const uint64_t gc = op->gcmask;
      if ((base & gc) == gc) {
        const amp_t<R> *m = mats + op->mat;
        switch (op->k) {
          case 1: tile_apply<R, 1, NT>(tile, t, op, m); break;
          case 2: tile_apply<R, 2, NT>(tile, t, op, m); break;
          case 3: tile_apply<R, 3, NT>(tile, t, op, m); break;
          case 4: tile_apply<R, 4, NT>(tile, t, op, m); break;
          default: tile_apply<R, 5, NT>(tile, t, op, m); break;
        }
      }
    }
    __syncthreads();
  }
}

// One tile of one pass: load the 2^t amplitudes into LDS, run the stages, store them back.
// `seg` holds the 2^h segment offsets of the pass (shared memory, filled by the caller).
// FULL: 2^t is a multiple of kStreamChunk * kBlock * VN, so every streamed vector exists and the
// accesses need no guard (straight-line code lets the memory counters be waited on exactly).
template <typename R, int RB, bool FULL, bool TWO = true, bool PH = false>
__device__ __forceinline__ void tile_body(amp_t<R> *__restrict__ psi, uint64_t tix, const TilePass &P,
                                          const uint64_t *seg, amp_t<R> *__restrict__ tile,
                                          const TileStage *__restrict__ stages,
                                          const RegOp *__restrict__ rops, const TileOp *__restrict__ tops,
                                          const amp_t<R> *__restrict__ mats) {
  using V = typename Vec16<R>::type;
  constexpr int VN = Vec16<R>::n;
  constexpr uint32_t kStep = kBlock * VN;
  const uint32_t t = P.t, L = P.L;
  const uint32_t tsize = 1u << t, segmask = (1u << L) - 1;
  const uint64_t base = tile_base(tix, P);
  for (uint32_t l0 = threadIdx.x * VN; l0 < tsize; l0 += kStreamChunk * kStep) {
    const uint32_t s0 = lds_address(tile) + slot_bytes<R>(l0);  // l0 shares no bit with j * kStep
    V v[kStreamChunk];
#pragma unroll
    for (int j = 0; j < kStreamChunk; ++j) {
      const uint32_t l = l0 + j * kStep;
      if (FULL || l < tsize) v[j] = stream_load(reinterpret_cast<const V *>(psi + (base | seg[l >> L] | (l & segmask))));
    }
#pragma unroll
    for (int j = 0; j < kStreamChunk; ++j) {
      const uint32_t l = l0 + j * kStep;
      if (FULL || l < tsize) tile_put16<R>(s0 ^ slot_bytes<R>(j * kStep), v[j]);
    }
  }
  __syncthreads();
  run_stages<R, RB, 1, kBlock, TWO, PH>(tile, t, base, P.n_stages, stages, rops, tops, mats);
  // the store reads the computed tile through the relabelling (linear: sources of disjoint bit
  // sets combine by XOR)
  const uint32_t src_thread = store_source(threadIdx.x * VN, P), pair = slot_bytes<R>(store_source(1, P));
  for (uint32_t l0 = threadIdx.x * VN; l0 < tsize; l0 += kStreamChunk * kStep) {
    const uint32_t s0 = lds_address(tile) + slot_bytes<R>(src_thread ^ store_source(l0 - threadIdx.x * VN, P));
    V v[kStreamChunk];
#pragma unroll
    for (int j = 0; j < kStreamChunk; ++j) {
      const uint32_t l = l0 + j * kStep;
      if (FULL || l < tsize) v[j] = tile_get16p<R>(s0 ^ slot_bytes<R>(store_source(j * kStep, P)), pair);
    }
#pragma unroll
    for (int j = 0; j < kStreamChunk; ++j) {
      const uint32_t l = l0 + j * kStep;
      if (FULL || l < tsize) stream_store(reinterpret_cast<V *>(psi + (base | seg[l >> L] | (l & segmask))), v[j]);
    }
  }
  __syncthreads();
}

template <int NT = kBlock>
__device__ __forceinline__ void fill_segments(const TilePass &P, uint64_t *seg) {
  for (uint32_t sgi = threadIdx.x; sgi < (1u << P.h); sgi += NT) {
    uint64_t o = 0;
    for (uint32_t b = 0; b < P.h; ++b)
      if ((sgi >> b) & 1) o |= uint64_t(1) << P.hpos[b];
    seg[sgi] = o;
  }
  __syncthreads();
}

}  // namespace
#endif  // QS_TILE_KERNELS

}  // namespace dev
}  // namespace qs
