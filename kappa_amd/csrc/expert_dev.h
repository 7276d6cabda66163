// Device helpers shared by the expert kernels: bf16 packing, the MFMA step,
// streaming loads, the tile lookup of the grouped GEMMs and their LDS rings.
#pragma once

#include <hip/hip_runtime.h>

#include "common.h"

namespace kmoe {

// two floats -> one dword of bf16 (RNE), a in the low half: one v_cvt_pk_bf16_f32
__device__ __forceinline__ uint32_t pack_bf16x2(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){a, b}, bf16x2));
}

__device__ __forceinline__ bf16x8 as_bf16x8(const uint4 v) { return __builtin_bit_cast(bf16x8, v); }

// rows a (even k) and b (odd k) of two columns -> one dword of one column each
__device__ __forceinline__ uint32_t pair_lo(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x05040100u); }
__device__ __forceinline__ uint32_t pair_hi(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

// eight rows of two columns (one dword per row) -> the operands of the two columns
__device__ __forceinline__ void transpose2(const uint32_t* r, bf16x8& c0, bf16x8& c1) {
  c0 = as_bf16x8(uint4{pair_lo(r[0], r[1]), pair_lo(r[2], r[3]), pair_lo(r[4], r[5]), pair_lo(r[6], r[7])});
  c1 = as_bf16x8(uint4{pair_hi(r[0], r[1]), pair_hi(r[2], r[3]), pair_hi(r[4], r[5]), pair_hi(r[6], r[7])});
}

// 16 bytes with a nontemporal load: for data a kernel reads exactly once, such
// as the decode weights (streaming reads this way sustain ~7.1 TB/s on MI355X
// against ~6.3 TB/s for ordinary loads, which also allocate in the caches)
__device__ __forceinline__ uint4 load_stream16(const int8_t* p) {
  typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
  const u32x4 v = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(p));
  return uint4{v.x, v.y, v.z, v.w};
}

__device__ __forceinline__ floatx4 mfma16(const bf16x8 a, const bf16x8 b, const floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}

// Block-wide tile prefix over experts: mtp[e] = sum_{e' < e} ceil(min(group_size[e'], cap) / BM), mtp[E] = total.
// The first 256 threads compute it (E <= 1024); blockDim.x must be a multiple of 64, at least 256.
// wsum: 4 ints of LDS scratch. offs (optional, E + 1 ints of LDS): a copy of offsets, so
// the caller's later lookups of its expert's row range are LDS reads, not another global
// round trip.
template <int BM>
__device__ void tile_prefix(const int32_t* __restrict__ offsets, int E, int cap, int* mtp, int* wsum,
                            int* offs = nullptr) {
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  int c[4];
  int local = 0, incl = 0;
  if (tid < 256) {
    // offsets[4 tid .. 4 tid + 4], clamped to the array: five loads in flight
    // together (guarded loads would each wait a round trip of their own)
    int o[5];
#pragma unroll
    for (int i = 0; i < 5; ++i) o[i] = offsets[min(tid * 4 + i, E)];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = tid * 4 + i;
      c[i] = e < E ? (min(o[i + 1] - o[i], cap) + BM - 1) / BM : 0;
      if (offs != nullptr && e <= E) offs[e] = o[i];
      local += c[i];
    }
    if (offs != nullptr && tid * 4 + 4 == E) offs[E] = o[4];
    incl = local;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int v = __shfl_up(incl, off, 64);
      if (lane >= off) incl += v;
    }
    if (lane == 63) wsum[wv] = incl;
  }
  __syncthreads();
  if (tid < 256) {
    int base = 0;
    for (int w = 0; w < wv; ++w) base += wsum[w];
    int run = base + incl - local;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = tid * 4 + i;
      if (e < E) mtp[e] = run;
      run += c[i];
    }
    if (tid == 255) mtp[E] = base + incl;
  }
  __syncthreads();
}

// largest e in [0, E) with mtp[e] <= v (mtp non-decreasing, mtp[0] = 0)
__device__ __forceinline__ int tile_expert(const int* mtp, int E, int v) {
  int lo = 0, hi = E - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (mtp[mid] <= v)
      lo = mid;
    else
      hi = mid - 1;
  }
  return lo;
}

typedef __attribute__((address_space(3))) void lds_void;

__device__ __forceinline__ uint32_t lds_addr(const void* p) { return (uint32_t)(uintptr_t)(const lds_void*)p; }

// 16 bytes per lane from global memory (sbase + voff) into LDS at lds + 16 * lane.
// sbase and lds must be wave-uniform. The LDS address goes through M0: the
// asm keeps the caller's M0 (saved and restored, so no clobber of a register
// the compiler reserves) and puts one wait state between the SALU write of M0
// and the LDS-DMA load that reads it (a gfx9 hazard the compiler does not see
// inside inline asm).
__device__ __forceinline__ void dma16(uint32_t voff, const void* sbase, uint32_t lds) {
  uint32_t m0save;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2\n\ts_mov_b32 m0, %0"
      : "=&s"(m0save)
      : "v"(voff), "s"(sbase), "s"(lds)
      : "memory");
}
// The same with the nontemporal hint, for weights no other tile re-reads.
__device__ __forceinline__ void dma16_stream(uint32_t voff, const void* sbase, uint32_t lds) {
  uint32_t m0save;
  asm volatile(
      "s_mov_b32 %0, m0\n\ts_mov_b32 m0, %3\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2 nt\n\ts_mov_b32 m0, %0"
      : "=&s"(m0save)
      : "v"(voff), "s"(sbase), "s"(lds)
      : "memory");
}

// Wait until at most N of this wave's vector-memory loads are outstanding and
// its LDS reads are done, then a workgroup barrier. The "memory" clobber keeps
// every LDS access on its side.
template <int N>
__device__ __forceinline__ void vm_barrier() {
  static_assert(N >= 0 && N < 64, "vmcnt range");
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(N) : "memory");
}

// An A stage is [row][8 x 16 B]: slot x of row r holds piece x ^ (r & 7) of the row's
// chunk (int8 planes, kOrder = 0) or, for bf16 chunks (kOrder = 1), piece
// order(x ^ (r & 7)) with order(y) = 2 (y & 3) + (y >> 2). A fragment read takes
// the four pieces q, q + 4, .. of the lane groups q: 0..3 or 4..7 of an int8
// chunk, but every second piece (2 q + st) of a bf16 one, whose order makes them
// four adjacent slots too. With the even slots as they came the reads counted 3
// bank-conflict cycles each.
template <int kOrder>
__device__ __forceinline__ int a_piece_at(int r, int slot) {
  const int y = slot ^ (r & 7);
  return kOrder ? ((y & 3) << 1) | (y >> 2) : y;
}
// element offset of piece p of row r
template <int kOrder>
__device__ __forceinline__ int a_at(int r, int p) {
  const int y = kOrder ? (p >> 1) | ((p & 1) << 2) : p;
  return r * 64 + ((y ^ (r & 7)) << 3);
}

}  // namespace kmoe
