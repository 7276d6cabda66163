// rms_norm's reduction (kappa/qwen3/norms.py:10-16), shared by the stand-alone
// norm kernel and the split router that normalises its own input.
#pragma once

#include "common.h"

namespace kmoe {

// A row of D elements staged in LDS for its reduction: slices of 64 elements, 16 bytes
// apart more than their size, so that the lanes' slices start in distinct banks
// and stay 16-byte aligned.
template <typename A>
struct NormRow {
  static constexpr int kPiece = 16 / sizeof(A);             // elements of a 16-byte piece
  static constexpr int kSlice = kRouterSlice + kPiece;      // elements per staged slice
  // f32 elements per lane in flight where a row or a scale moves element by element (the
  // compiler keeps enough bf16 ones in flight by itself)
  static constexpr int kBatch = 32;
  static constexpr int kPieces = 64 * kRouterSlice / kPiece / 64;  // pieces per lane of the widest row (D = 4096)
  __host__ __device__ static size_t bytes(int D) {
    return (size_t)((D + kRouterSlice - 1) / kRouterSlice) * kSlice * sizeof(A);
  }
  __device__ __forceinline__ static int at(int d) { return (d >> 6) * kSlice + (d & 63); }
  // rows that move in 16-byte pieces
  __device__ __forceinline__ static bool pieces(const A* src, int D) {
    return D % kRouterSlice == 0 && (reinterpret_cast<uintptr_t>(src) & 15) == 0;
  }
  __device__ __forceinline__ static void unpack(const uint4& v, float* f) {
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (sizeof(A) == 2) {
        f[2 * i] = __uint_as_float(w[i] << 16);
        f[2 * i + 1] = __uint_as_float(w[i] & 0xffff0000u);
      } else {
        f[i] = __uint_as_float(w[i]);
      }
    }
  }
};

// One wave: stage the row src[0..D) in LDS (NormRow) and return
//   r = 1 / sqrt(S / D + eps),  S = sum_d src[d]^2
// in the canonical order: each square rounded to float, lane s adds the
// squares of slice s (64 indices) in a sequential chain from +0.0f, and the
// slice sums are combined by the zero-padded pairwise tree p[l] += p[l + st]
// (the router's order); IEEE division and square root. The row stays in LDS
// for the caller and, where it moves in pieces (NormRow::pieces), piece lane + 64 i
// in v[i]; every lane of the wave must call it, and gets r.
template <typename A>
__device__ __forceinline__ float wave_rms_factor(const A* __restrict__ src, int D, float eps, A* row,
                                                 uint4 (&v)[NormRow<A>::kPieces]) {
#pragma clang fp contract(off)
  using R = NormRow<A>;
  const int lane = threadIdx.x & 63;
  const int NS = (D + kRouterSlice - 1) / kRouterSlice;
  int P = 1;
  while (P < NS) P <<= 1;
  const bool pieces = R::pieces(src, D);
  if (pieces) {
    const int n = D / R::kPiece;
#pragma unroll
    for (int i = 0; i < R::kPieces; ++i) {
      v[i] = uint4{0u, 0u, 0u, 0u};
      if (lane + 64 * i < n) v[i] = reinterpret_cast<const uint4*>(src)[lane + 64 * i];
    }
#pragma unroll
    for (int i = 0; i < R::kPieces; ++i)
      if (lane + 64 * i < n) *reinterpret_cast<uint4*>(row + R::at((lane + 64 * i) * R::kPiece)) = v[i];
  } else {
    // floats in batches, all issued before their LDS writes (addresses clamped into the
    // row, so no load sits behind a branch): 4096 misaligned rows of 2048 floats take
    // 17.2 us; one element at a time, with the chains read from LDS likewise, 36.3
    if constexpr (sizeof(A) == 4) {
      for (int base = 0; base < D; base += 64 * R::kBatch) {
        A e[R::kBatch];
#pragma unroll
        for (int j = 0; j < R::kBatch; ++j) e[j] = src[min(base + 64 * j + lane, D - 1)];
#pragma unroll
        for (int j = 0; j < R::kBatch; ++j) {
          const int d = base + 64 * j + lane;
          if (d < D) row[R::at(d)] = e[j];
        }
      }
    } else {
      for (int d = lane; d < D; d += 64) row[R::at(d)] = src[d];
    }
    // the last slice is filled up with zeros, whose squares leave its chain as it is
    const int tail = (NS - 1) * kRouterSlice + lane;
    if (tail >= D) row[R::at(tail)] = 0;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  float acc = 0.0f;
  if (lane < NS) {
    const A* sl = row + lane * R::kSlice;
    // the slice's reads are all in flight before the chain starts
    uint4 p[kRouterSlice / R::kPiece];
#pragma unroll
    for (int i = 0; i < kRouterSlice / R::kPiece; ++i) p[i] = reinterpret_cast<const uint4*>(sl)[i];
#pragma unroll
    for (int i = 0; i < kRouterSlice / R::kPiece; ++i) {
      float f[R::kPiece];
      R::unpack(p[i], f);
#pragma unroll
      for (int j = 0; j < R::kPiece; ++j) {
        const float sq = f[j] * f[j];
        acc = acc + sq;
      }
    }
  }
  for (int st = 1; st < P; st <<= 1) {
    const float o = __shfl_down(acc, st, 64);
    if ((lane & (2 * st - 1)) == 0) acc = acc + o;
  }
  const float total = __shfl(acc, 0, 64);
  const float var = total / (float)D;
  return 1.0f / sqrtf(var + eps);
}

// One normalised element: round_act((x * r) * scale), each product rounded.
template <typename A>
__device__ __forceinline__ float rms_apply(float x, float r, float s) {
#pragma clang fp contract(off)
  const float n = x * r;
  return Act<A>::round(n * s);
}

}  // namespace kmoe
