// Router logits, top-k with renormalised weights, and the stable dispatch sort.
//
// Reference: _route (kappa/qwen3/ffn_moe.py:38-56) and the ordering part of
// _moe_ragged (kappa/qwen3/ffn_moe.py:189-200, 212).
#include <float.h>

#include <algorithm>
#include <cmath>

#include "common.h"
#include "expert_dev.h"
#include "launch.h"
#include "norm.h"
#include "route_dev.h"

namespace kmoe {

// ---------------------------------------------------------------------------
// Router weight rows. A lane owns EPL consecutive experts of one hidden row
// and loads them with 16-byte loads, or one 8- or 4-byte load when the EPL
// experts take 8 or 4 bytes; LPR = E / EPL lanes cover a row contiguously.
// ---------------------------------------------------------------------------
template <int RT, int EPL>
struct RouterRow {
  static constexpr int kBytes = EPL * (RT == 0 ? 4 : (RT == 1 ? 2 : 1));
  static constexpr int kWords = kBytes / 4;
  struct Raw {
    uint32_t w[kWords];
  };
  __device__ __forceinline__ static void load(const void* rw, int64_t elem, Raw& r) {
    load_at(reinterpret_cast<const char*>(rw) + elem * (kBytes / EPL), 0, r);
  }
  // row pointer (uniform across the wave) plus a per-lane byte offset
  __device__ __forceinline__ static void load_at(const char* row, int off, Raw& r) {
    const char* p = row + off;
    if constexpr (kWords % 4 == 0) {
#pragma unroll
      for (int q = 0; q < kWords / 4; ++q) {
        const uint4 v = reinterpret_cast<const uint4*>(p)[q];
        r.w[4 * q] = v.x, r.w[4 * q + 1] = v.y, r.w[4 * q + 2] = v.z, r.w[4 * q + 3] = v.w;
      }
    } else if constexpr (kWords == 2) {
      const uint2 v = *reinterpret_cast<const uint2*>(p);
      r.w[0] = v.x, r.w[1] = v.y;
    } else {
      static_assert(kWords == 1, "router rows of 4, 8 or 16k bytes per lane");
      r.w[0] = *reinterpret_cast<const uint32_t*>(p);
    }
  }
  // to_compute_dtype(router_w, f32) (kappa/qwen3/quant.py:34-38): int8 is f32(q) * f32(scale)
  __device__ __forceinline__ static void convert(const Raw& r, const float* sc, float* out) {
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      if constexpr (RT == 0) {
        out[i] = __uint_as_float(r.w[i]);
      } else if constexpr (RT == 1) {
        const uint32_t v = r.w[i >> 1];
        out[i] = __uint_as_float((i & 1) ? (v & 0xffff0000u) : (v << 16));
      } else {
        const int8_t q = (int8_t)((r.w[i >> 2] >> (8 * (i & 3))) & 0xffu);
        out[i] = (float)q * sc[i];
      }
    }
  }
  __device__ __forceinline__ static float load1(const void* rw, int64_t elem, float sc) {
    if constexpr (RT == 0) return reinterpret_cast<const float*>(rw)[elem];
    if constexpr (RT == 1) return bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(rw)[elem]);
    return (float)reinterpret_cast<const int8_t*>(rw)[elem] * sc;
  }
};

__device__ __forceinline__ float load_scale(const void* scale, int scale_bf16, int64_t i) {
  return scale_bf16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(scale)[i])
                    : reinterpret_cast<const float*>(scale)[i];
}

// ---------------------------------------------------------------------------
// Fused router: logits in the canonical order, top-k, softmax.
//
// logits[t,e] = tree_s( fmaf-chain_{d in slice s}( x[t,d] * r[d,e] ) ) with
// slices of 64 hidden indices and the pairwise tree p[i] += p[i+st],
// st = 1, 2, 4, ... over the slices zero-padded to P = next power of two.
//
// Slice s is owned by lane group lg = s % SPW of wave-group s / SPW (a lane
// group is LPR lanes covering all experts; SPW groups per wave). A wave runs
// G wave-groups one after the other; the tree levels st < SPW are shuffles
// between lane groups, the levels SPW <= st < SPW*G combine the G wave-groups
// in registers, and the remaining levels combine the waves' partials through
// LDS, one element's partials per thread. x for the TB tokens of the block
// is staged in LDS as f32 [slice][64][TB] (slice pitch padded by 4 floats:
// the lane groups of a wave read different slices in distinct banks); the
// same LDS then holds the wave partials [wave][TB][E].
//
// Then one wave per token selects the top K (value descending, ties to the
// lower expert index; NaN ranks as -inf) with K wave-wide arg-max rounds, and
// lane j < K writes selection j and its softmax weight
//   w_j = expf(l_j - l_0) / sum_{i<K} expf(l_i - l_0)   (sum in i order),
// rounded to the activation dtype when out_bf16.
// ---------------------------------------------------------------------------
template <int TB, int EPL>
struct Acc {
  float v[TB][EPL];
};

template <typename A, int RT, int EPL, int TB, int G>
__global__ __launch_bounds__(1024) void k_route(int T, int D, int E, int K, int LPR, int SPW, int P,
                                                 const A* __restrict__ x, const void* __restrict__ rw,
                                                 const void* __restrict__ rscale, int scale_bf16, int scale_pc,
                                                 float* __restrict__ logits, int32_t* __restrict__ topk_idx,
                                                 float* __restrict__ topk_w, int out_bf16) {
  using Row = RouterRow<RT, EPL>;
  // rows per prefetch stage: a stage of raw rows is 32 registers for one
  // token per block (latency-bound: a 64-row slice of a bf16 router takes 8
  // dependent memory round trips), 16 registers otherwise (two stages and the
  // accumulators fit the 128 registers of a 1024-thread block)
  constexpr int RW = TB == 1 && G == 1 ? 32 : 16;
  constexpr int U0 = RW / Row::kWords < 1 ? 1 : RW / Row::kWords;
  constexpr int U = U0 < 16 / TB ? U0 : 16 / TB;
  extern __shared__ float lds[];
  const int NWB = blockDim.x >> 6;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int S = (D + kRouterSlice - 1) / kRouterSlice;
  const int XP = kRouterSlice * TB + 4;
  const int t0 = blockIdx.x * TB;
#pragma unroll
  for (int tt = 0; tt < TB; ++tt)
    for (int d = threadIdx.x; d < D; d += blockDim.x)
      lds[(d >> 6) * XP + (d & 63) * TB + tt] = (t0 + tt < T) ? Act<A>::load(x, (int64_t)(t0 + tt) * D + d) : 0.0f;
  __syncthreads();

  const int lg = lane / LPR, le = lane - lg * LPR;
  const int e0 = le * EPL;
  const bool lane_on = lg < SPW && e0 < E;
  const bool vec = (E % 8) == 0 && e0 + EPL <= E;
  float sc[EPL];
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    sc[i] = 0.0f;
    if (RT == 2 && e0 + i < E) sc[i] = load_scale(rscale, scale_bf16, scale_pc ? e0 + i : 0);
  }

  Acc<TB, EPL> p0, p1;
#pragma unroll
  for (int gi = 0; gi < G; ++gi) {
    Acc<TB, EPL> c;
#pragma unroll
    for (int tt = 0; tt < TB; ++tt)
#pragma unroll
      for (int i = 0; i < EPL; ++i) c.v[tt][i] = 0.0f;
    const int s = (w * G + gi) * SPW + lg;
    if (lane_on && s < S) {
      const int d0 = s * kRouterSlice;
      const int d1 = min(D, d0 + kRouterSlice);
      const float* xs = lds + s * XP - d0 * TB;
      if (vec && d1 - d0 == kRouterSlice) {
        // two register stages used in turn (the loop body covers 2U rows, and
        // 2U divides the 64 rows of a slice), so no stage is copied
        static_assert(kRouterSlice % (2 * U) == 0, "two stages per step");
        typename Row::Raw b0[U], b1[U];
        auto rows = [&](const typename Row::Raw* raw, int db) {
#pragma unroll
          for (int u = 0; u < U; ++u) {
            float r[EPL], xv[TB];
            Row::convert(raw[u], sc, r);
            // the x stage is 16-byte aligned for TB >= 4 (slice stride
            // 64*TB + 4 floats, row stride TB floats)
            if constexpr (TB % 4 == 0) {
#pragma unroll
              for (int q = 0; q < TB / 4; ++q) {
                const float4 v4 = *reinterpret_cast<const float4*>(xs + (db + u) * TB + 4 * q);
                xv[4 * q] = v4.x, xv[4 * q + 1] = v4.y, xv[4 * q + 2] = v4.z, xv[4 * q + 3] = v4.w;
              }
            } else {
#pragma unroll
              for (int tt = 0; tt < TB; ++tt) xv[tt] = xs[(db + u) * TB + tt];
            }
#pragma unroll
            for (int tt = 0; tt < TB; ++tt)
#pragma unroll
              for (int i = 0; i < EPL; ++i) c.v[tt][i] = __builtin_fmaf(xv[tt], r[i], c.v[tt][i]);
          }
        };
#pragma unroll
        for (int u = 0; u < U; ++u) Row::load(rw, (int64_t)(d0 + u) * E + e0, b0[u]);
        for (int db = d0; db < d1; db += 2 * U) {
#pragma unroll
          for (int u = 0; u < U; ++u) Row::load(rw, (int64_t)(db + U + u) * E + e0, b1[u]);
          rows(b0, db);
          if (db + 2 * U < d1) {
#pragma unroll
            for (int u = 0; u < U; ++u) Row::load(rw, (int64_t)(db + 2 * U + u) * E + e0, b0[u]);
          }
          rows(b1, db + U);
        }
      } else {
        for (int d = d0; d < d1; ++d) {
          float r[EPL];
#pragma unroll
          for (int i = 0; i < EPL; ++i) r[i] = (e0 + i < E) ? Row::load1(rw, (int64_t)d * E + e0 + i, sc[i]) : 0.0f;
#pragma unroll
          for (int tt = 0; tt < TB; ++tt) {
            const float xv = xs[d * TB + tt];
#pragma unroll
            for (int i = 0; i < EPL; ++i) c.v[tt][i] = __builtin_fmaf(xv, r[i], c.v[tt][i]);
          }
        }
      }
    }
    // tree levels st < SPW: lane group lg += lane group lg + st
    for (int st = 1; st < SPW && st < P; st <<= 1) {
#pragma unroll
      for (int tt = 0; tt < TB; ++tt)
#pragma unroll
        for (int i = 0; i < EPL; ++i) c.v[tt][i] = c.v[tt][i] + __shfl_down(c.v[tt][i], st * LPR, 64);
    }
    // tree levels over the wave's G wave-groups (G <= 4)
#pragma unroll
    for (int tt = 0; tt < TB; ++tt)
#pragma unroll
      for (int i = 0; i < EPL; ++i) {
        if (G == 1 || gi == 0) {
          p0.v[tt][i] = c.v[tt][i];
        } else if (gi == 1) {
          p0.v[tt][i] = p0.v[tt][i] + c.v[tt][i];
        } else if (gi == 2) {
          p1.v[tt][i] = c.v[tt][i];
        } else {
          p1.v[tt][i] = p1.v[tt][i] + c.v[tt][i];
          p0.v[tt][i] = p0.v[tt][i] + p1.v[tt][i];
        }
      }
  }
  __syncthreads();  // x no longer needed: the LDS now holds the wave partials
  float* part = lds;
  const int TE = TB * E;
  if (lg == 0) {
#pragma unroll
    for (int tt = 0; tt < TB; ++tt)
#pragma unroll
      for (int i = 0; i < EPL; ++i)
        if (e0 + i < E) part[(size_t)w * TE + tt * E + e0 + i] = p0.v[tt][i];
  }
  __syncthreads();
  // the tree levels across the NWB waves (a power of two, at most 16): a
  // thread takes an element's NWB partials and applies the levels
  // p[g] += p[g + st], st = 1, 2, 4, 8, in registers
  for (int rem = threadIdx.x; rem < TE; rem += blockDim.x) {
    float v[16];
#pragma unroll
    for (int g = 0; g < 16; ++g) v[g] = g < NWB ? part[(size_t)g * TE + rem] : 0.0f;
#pragma unroll
    for (int st = 1; st < 16; st <<= 1)
#pragma unroll
      for (int g = 0; g + st < 16; g += 2 * st)
        if (g + st < NWB) v[g] = v[g] + v[g + st];
    part[rem] = v[0];
  }
  __syncthreads();

  // top-k: lane owns experts lane + 64*i, i < EPL (E <= 64 * EPL); the
  // per-wave selection scratch sits after the partials
  TopkLds* tk = reinterpret_cast<TopkLds*>(lds + (size_t)NWB * TE);
  for (int tt = w; tt < TB; tt += NWB) {
    const int t = t0 + tt;
    if (t >= T) break;
    float v[EPL];
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      const int e = lane + 64 * i;
      const float q = e < E ? part[tt * E + e] : 0.0f;
      v[i] = (e < E && q == q) ? q : -INFINITY;
      if (logits && e < E) logits[(int64_t)t * E + e] = q;
    }
    if (E <= 128 || EPL < 4)
      wave_topk<(EPL < 2 ? EPL : 2)>(t, E, K, v, topk_idx, topk_w, out_bf16, nullptr, tk[w]);
    else if (E <= 256 || EPL < 8)
      wave_topk<(EPL < 4 ? EPL : 4)>(t, E, K, v, topk_idx, topk_w, out_bf16, nullptr, tk[w]);
    else if (E <= 512 || EPL < 16)
      wave_topk<(EPL < 8 ? EPL : 8)>(t, E, K, v, topk_idx, topk_w, out_bf16, nullptr, tk[w]);
    else
      wave_topk<EPL>(t, E, K, v, topk_idx, topk_w, out_bf16, nullptr, tk[w]);
  }
}

// ---------------------------------------------------------------------------
// Split router for small token counts (decode): the same canonical logits as
// k_route, computed by many blocks per token instead of one.
//
// k_route_slices, block (g, tb): wave w runs the fmaf chain of slice
// s = 4g + w for the TB tokens tb*TB .. tb*TB+TB-1 (with a SliceNorm, x is
// the residual stream and the block first normalises its tokens' rows -
// rms_norm of kappa/qwen3/norms.py:10-16 - writing its four slices of the
// normalised rows for the expert kernels), a lane owning EPL
// consecutive experts (all 64 rows of the slice in flight at once when they
// fit in 64 registers). The block then applies tree levels st = 1 and 2 to its
// four slices (the zero-padded tree's aligned group of four) and writes the
// group partial part[t][g][e], g < Q = max(1, P / 4).
// k_route_finish, one wave per token: tree levels st = 4, 8, ... over the Q
// group partials (the levels st >= 4 of the same tree), then the top-k and
// softmax of k_route.
// ---------------------------------------------------------------------------
template <typename A, int RT, int EPL, int TB>
__global__ __launch_bounds__(256) void k_route_slices(int T, int D, int E, int P, int Q, const A* __restrict__ x,
                                                       const void* __restrict__ rw, const void* __restrict__ rscale,
                                                       int scale_bf16, int scale_pc, float* __restrict__ part,
                                                       const kmoe_host::SliceNorm nm) {
  using Row = RouterRow<RT, EPL>;
  constexpr int U = Row::kWords <= 1 ? 64 : 64 / Row::kWords;  // rows per load stage
  __shared__ float xs[4][kRouterSlice][TB];
  __shared__ float red[2][TB * EPL][64];
  __shared__ float rfac[TB];
  extern __shared__ __attribute__((aligned(16))) uint8_t nrow[];  // with nm.scale: TB staged rows (NormRow)
  const int g = blockIdx.x, t0 = blockIdx.y * TB;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int s = 4 * g + w;
  const int d0 = s * kRouterSlice;
  const size_t NRB = NormRow<A>::bytes(D);
  if (nm.scale) {
    // x is the residual stream h: wave tt reduces row t0 + tt (the canonical
    // rms_norm order); the slices are normalised below
    if (w < TB && t0 + w < T) {
      uint4 held[NormRow<A>::kPieces];
      const float r =
          wave_rms_factor(x + (int64_t)(t0 + w) * D, D, nm.eps, reinterpret_cast<A*>(nrow + w * NRB), held);
      if (lane == 0) rfac[w] = r;
    }
    __syncthreads();
  }
  for (int i = threadIdx.x; i < 4 * kRouterSlice * TB; i += blockDim.x) {
    const int tt = i % TB, r = (i / TB) % kRouterSlice, ws = i / (TB * kRouterSlice);
    const int d = (4 * g + ws) * kRouterSlice + r;
    float v = 0.0f;
    if (t0 + tt < T && d < D) {
      if (nm.scale) {
        // the block's input h2 = round_act((h * r) * scale): staged here and
        // written out for the expert kernels (each block writes its slices)
        const float sc = load_scale(nm.scale, nm.scale_bf16, d);
        v = rms_apply<A>(Act<A>::load(reinterpret_cast<const A*>(nrow + tt * NRB), NormRow<A>::at(d)), rfac[tt], sc);
        Act<A>::store(reinterpret_cast<A*>(nm.h2), (int64_t)(t0 + tt) * D + d, v);
      } else {
        v = Act<A>::load(x, (int64_t)(t0 + tt) * D + d);
      }
    }
    xs[ws][r][tt] = v;
  }
  const int LPR = (E + EPL - 1) / EPL;
  const int e0 = lane * EPL;
  float sc[EPL];
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    sc[i] = 0.0f;
    if (RT == 2 && e0 + i < E) sc[i] = load_scale(rscale, scale_bf16, scale_pc ? e0 + i : 0);
  }
  float acc[TB][EPL];
#pragma unroll
  for (int tt = 0; tt < TB; ++tt)
#pragma unroll
    for (int i = 0; i < EPL; ++i) acc[tt][i] = 0.0f;
  __syncthreads();
  if (lane < LPR && d0 < D) {
    const int n = min(kRouterSlice, D - d0);
    if (E % EPL == 0 && n == kRouterSlice) {
      // row pointers are uniform (scalar registers), the lane offset is e0
      constexpr int kBpe = Row::kBytes / EPL;
      const char* row0 = reinterpret_cast<const char*>(rw) + (int64_t)d0 * E * kBpe;
      const int64_t pitch = (int64_t)E * kBpe;
      const int loff = e0 * kBpe;
      for (int db = 0; db < kRouterSlice; db += U) {
        typename Row::Raw raw[U];
#pragma unroll
        for (int u = 0; u < U; ++u) Row::load_at(row0 + (db + u) * pitch, loff, raw[u]);
#pragma unroll
        for (int u = 0; u < U; ++u) {
          float r[EPL];
          Row::convert(raw[u], sc, r);
#pragma unroll
          for (int tt = 0; tt < TB; ++tt) {
            const float xv = xs[w][db + u][tt];
#pragma unroll
            for (int i = 0; i < EPL; ++i) acc[tt][i] = __builtin_fmaf(xv, r[i], acc[tt][i]);
          }
        }
      }
    } else {
      for (int r0 = 0; r0 < n; ++r0) {
        float r[EPL];
#pragma unroll
        for (int i = 0; i < EPL; ++i)
          r[i] = (e0 + i < E) ? Row::load1(rw, (int64_t)(d0 + r0) * E + e0 + i, sc[i]) : 0.0f;
#pragma unroll
        for (int tt = 0; tt < TB; ++tt) {
          const float xv = xs[w][r0][tt];
#pragma unroll
          for (int i = 0; i < EPL; ++i) acc[tt][i] = __builtin_fmaf(xv, r[i], acc[tt][i]);
        }
      }
    }
  }
  // tree levels st = 1 (slices 0+1, 2+3) and st = 2 (0+2) of the group
  if (w & 1) {
#pragma unroll
    for (int tt = 0; tt < TB; ++tt)
#pragma unroll
      for (int i = 0; i < EPL; ++i) red[w >> 1][tt * EPL + i][lane] = acc[tt][i];
  }
  __syncthreads();
  if (!(w & 1) && 1 < P) {
#pragma unroll
    for (int tt = 0; tt < TB; ++tt)
#pragma unroll
      for (int i = 0; i < EPL; ++i) acc[tt][i] = acc[tt][i] + red[w >> 1][tt * EPL + i][lane];
  }
  __syncthreads();
  if (w == 2) {
#pragma unroll
    for (int tt = 0; tt < TB; ++tt)
#pragma unroll
      for (int i = 0; i < EPL; ++i) red[0][tt * EPL + i][lane] = acc[tt][i];
  }
  __syncthreads();
  if (w != 0 || lane >= LPR) return;
#pragma unroll
  for (int tt = 0; tt < TB; ++tt) {
    if (t0 + tt >= T) break;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      const float v = 2 < P ? acc[tt][i] + red[0][tt * EPL + i][lane] : acc[tt][i];
      if (e0 + i < E) part[((int64_t)(t0 + tt) * Q + g) * E + e0 + i] = v;
    }
  }
}

template <int EPL>
__global__ __launch_bounds__(256) void k_route_finish(int T, int E, int K, int Q, const float* __restrict__ part,
                                                       float* __restrict__ logits, int32_t* __restrict__ topk_idx,
                                                       float* __restrict__ topk_w, int out_bf16) {
  __shared__ TopkLds tk[4];
  const int w = threadIdx.x >> 6;
  const int t = blockIdx.x * 4 + w;
  if (t >= T) return;  // per wave: this kernel has no block-wide barrier
  finish_token<EPL>(t, E, K, Q, part, logits, topk_idx, topk_w, out_bf16, nullptr, tk[w]);
}

__global__ __launch_bounds__(256) void k_dispatch_count(int T, int E, int K, const int32_t* __restrict__ topk_idx,
                                                         int32_t* __restrict__ hist) {
  __shared__ unsigned long long mask[kMaxExperts];
  chunk_masks(T, E, K, blockIdx.x, topk_idx, mask);
  for (int e = threadIdx.x; e < E; e += blockDim.x) hist[(int64_t)blockIdx.x * E + e] = __popcll(mask[e]);
}

// T <= NW <= 16: the finish is one block of NW waves, one token each, so it
// also runs the dispatch sort of the tokens (the selections pass through LDS;
// no second kernel). At larger T a single block's serial top-ks and sort
// cost more than the separate dispatch kernel.
template <int EPL, int NW>
__global__ __launch_bounds__(64 * NW) void k_route_finish_dispatch(
    int T, int E, int K, int Q, const float* __restrict__ part, float* __restrict__ logits,
    int32_t* __restrict__ topk_idx, float* __restrict__ topk_w, int out_bf16, int32_t* __restrict__ group_sizes,
    int32_t* __restrict__ offsets, int32_t* __restrict__ active, int32_t* __restrict__ sorted_token,
    int32_t* __restrict__ sorted_expert, int32_t* __restrict__ inv, int cap) {
  static_assert(NW >= 4 && NW <= 16, "dispatch_chunk needs 256 threads; one wave per token");
  __shared__ TopkLds tk[NW];
  __shared__ DispatchLds L;
  __shared__ int32_t idx_lds[NW * kMaxTopK];
  const int w = threadIdx.x >> 6;
  if (w < T) finish_token<EPL>(w, E, K, Q, part, logits, topk_idx, topk_w, out_bf16, idx_lds, tk[w]);
  __syncthreads();
  if (dispatch_fits_wave(T * K, E))
    dispatch_wave(T, E, K, idx_lds, group_sizes, offsets, active, sorted_token, sorted_expert, inv, cap);
  else
    dispatch_chunk(T, E, K, 0, 1, idx_lds, nullptr, group_sizes, offsets, active, sorted_token, sorted_expert, inv,
                   cap, L);
}

__global__ __launch_bounds__(256) void k_dispatch_scatter(int T, int E, int K, int nblk,
                                                           const int32_t* __restrict__ topk_idx,
                                                           const int32_t* __restrict__ hist,
                                                           int32_t* __restrict__ group_sizes,
                                                           int32_t* __restrict__ offsets, int32_t* __restrict__ active,
                                                           int32_t* __restrict__ sorted_token,
                                                           int32_t* __restrict__ sorted_expert,
                                                           int32_t* __restrict__ inv, int cap) {
  __shared__ DispatchLds L;
  dispatch_chunk(T, E, K, blockIdx.x, nblk, topk_idx, hist, group_sizes, offsets, active, sorted_token, sorted_expert,
                 inv, cap, L);
}


// ---------------------------------------------------------------------------
// Two-phase router: bf16 activations and router, D a multiple of 256, E % 16 == 0,
// E <= 256.
//
// Bit-exact top-k needs the canonical logits (k_route's order) only where the
// ranking is in doubt. k_route_logits computes every logit on the matrix cores
// (v_mfma_f32_16x16x32_bf16: exact products, f32 sums in the hardware's order, the
// reduction split over blocks): L~[t,e]. The exact sum, the canonical L and L~
// differ by at most c * sum_d |x_d r_de| <= c * ||x_t|| * ||r_e|| (Cauchy-Schwarz),
// where c covers the MFMA's accumulation and the sums of the splits (taken as up to
// 2D roundings of up to 2u each, u = 2^-24), the canonical chains and tree (64 +
// log2 P roundings), the rounding of the norms and of L~ -/+ delta (the host passes
// c). So L lies in [lo, hi] = [L~ - delta, L~ + delta], delta = c * ||x_t|| * ||r_e|| +
// 1e-30. The norms are f32 sums of squares, each at least kNormFloor: below it squares
// underflow and the computed sum says nothing, above it what underflow takes from
// it (at most 4096 * 2^-126) is less than c's room. Let tau be the K-th largest lo (the search stops at 16 key bits, which can
// only lower it). An expert whose hi is below tau has K experts strictly above
// it and cannot be selected, ties included; the top K are among the
// candidates {e : hi_e >= tau}. k_route_select recomputes the candidates' logits in
// the canonical order, ranks them (value descending, ties to the lower index)
// and takes the softmax of the first K, as wave_topk does. A token with a
// non-finite L~ or bound takes every expert as a candidate.
//
// k_route_logits also writes the router transposed to rTq [E][8][S][8] bf16: element
// (e, d = 64 s + 8 i + j) at ((e * 8 + i) * S + s) * 8 + j. Eight consecutive
// hidden indices of one expert (its MFMA operand, and eight steps of a slice
// chain) are one 16-byte piece, and the pieces i of the S slices of one expert are
// contiguous, so the slice lanes of a chain read 16 S consecutive bytes per step.
//
// Both kernels are chains of L2 round trips, not bandwidth: 30B-A3B T = 333 / 1500 /
// 4096 9 + 15, 11 + 18 and 14 + 21 us, 235B-A22B T = 2048 16 + 33 us. As one kernel (16
// tokens per block, every block streaming the whole transposed router that a third
// kernel had prepared) it took 5 + 36 us at 30B-A3B T = 4096 and 5 + 58 us at 235B-A22B
// T = 2048, and below 2048 tokens the all-VALU router ran (32 / 35 us at T = 333 / 1500,
// and 5 us for the histograms).
// ---------------------------------------------------------------------------

// Block (tile, ks, h): the partial logits of 64 tokens x 128 experts (128 h ..) over
// reduction steps [ks, ks + 1) * D / 32 / KS (a step is 32 hidden indices):
// part[ks][t][e]. The block's four waves take its steps in turn, so no wave loads what
// another does: lane (c, q) reads experts 8 c .. 8 c + 7 of rows 8 q .. 8 q + 7 (16
// lanes cover 256 consecutive bytes of a row) and pairs rows in registers
// (transpose2), and 16 bytes of the rows of the four 16-token tiles; U steps are in
// flight at once, which is a wave's whole share up to 16 steps per block. The router
// is the first MFMA operand, so a lane ends with 32 consecutive experts of a token
// of each tile; the waves' sums meet in LDS, wave w finishing tile w. A step's
// transposed operands are written to rTq by one of the tiles; tile 0 also sums the
// squares of its router columns: npart[ks][e]. The blocks zero the histograms
// together. The same work with 32 experts per wave and all steps in each took
// 17 / 19 us (30B-A3B T = 4096, 235B-A22B T = 2048), 19 / 21 with the token rows staged
// in LDS, of which the router's 4-byte loads were 9.
constexpr int kLogitWaves = 4;
__global__ __launch_bounds__(64 * kLogitWaves, 1) void k_route_logits(
    int T, int D, int E, int KS, const uint16_t* __restrict__ x, const uint16_t* __restrict__ r,
    uint16_t* __restrict__ rtq, float* __restrict__ npart, float* __restrict__ part, int32_t* __restrict__ hist,
    int nhist) {
  constexpr int U = 4;
  __shared__ floatx4 red[kLogitWaves][kLogitWaves - 1][8][64];  // [tile][other wave][4-expert run][lane]
  __shared__ float nred[kLogitWaves][128];
  const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, q = lane >> 4;
  const int tile = blockIdx.x, tiles = gridDim.x, ks = blockIdx.y;
  const int t0 = tile * 64, e0 = blockIdx.z * 128;
  for (int i = ((blockIdx.z * KS + ks) * tiles + tile) * 256 + threadIdx.x; i < nhist;
       i += gridDim.z * KS * tiles * 256)
    hist[i] = 0;
  const int S = D >> 6, steps = (D >> 5) / KS, st0 = ks * steps;
  const int e = e0 + 8 * c;
  const bool on = e < E;
  const uint16_t* xr[4];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi) xr[mi] = x + (int64_t)min(t0 + 16 * mi + c, T - 1) * D + 8 * q;
  floatx4 acc[8][4];
  float nn[8];
#pragma unroll
  for (int j = 0; j < 8; ++j) {
    nn[j] = 0.0f;
#pragma unroll
    for (int mi = 0; mi < 4; ++mi) acc[j][mi] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  for (int sb = w; sb < steps; sb += kLogitWaves * U) {
    uint4 a[U][4], b[U][8];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      if (sb + kLogitWaves * u < steps) {
        const int k0 = (st0 + sb + kLogitWaves * u) * 32;
        const uint16_t* rp = r + (int64_t)(k0 + 8 * q) * E + e;
#pragma unroll
        for (int i = 0; i < 8; ++i)
          b[u][i] = on ? *reinterpret_cast<const uint4*>(rp + (int64_t)i * E) : uint4{0u, 0u, 0u, 0u};
#pragma unroll
        for (int mi = 0; mi < 4; ++mi) a[u][mi] = *reinterpret_cast<const uint4*>(xr[mi] + k0);
      }
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int sl = sb + kLogitWaves * u;
      if (sl < steps) {
        uint32_t rows[4][8];  // [expert pair][row]
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          rows[0][i] = b[u][i].x;
          rows[1][i] = b[u][i].y;
          rows[2][i] = b[u][i].z;
          rows[3][i] = b[u][i].w;
        }
        const int d = (st0 + sl) * 32 + 8 * q;
#pragma unroll
        for (int p = 0; p < 4; ++p) {
          bf16x8 f[2];
          transpose2(rows[p], f[0], f[1]);
          if (sl % tiles == tile && on) {
#pragma unroll
            for (int j = 0; j < 2; ++j)
              *reinterpret_cast<uint4*>(rtq + ((int64_t)((e + 2 * p + j) * 8 + ((d & 63) >> 3)) * S + (d >> 6)) * 8) =
                  __builtin_bit_cast(uint4, f[j]);
          }
          if (tile == 0) {
#pragma unroll
            for (int i = 0; i < 8; ++i) {
              const float lo = __uint_as_float(rows[p][i] << 16), hi = __uint_as_float(rows[p][i] & 0xffff0000u);
              nn[2 * p] = __builtin_fmaf(lo, lo, nn[2 * p]);
              nn[2 * p + 1] = __builtin_fmaf(hi, hi, nn[2 * p + 1]);
            }
          }
#pragma unroll
          for (int j = 0; j < 2; ++j)
#pragma unroll
            for (int mi = 0; mi < 4; ++mi)
              acc[2 * p + j][mi] = mfma16(f[j], as_bf16x8(a[u][mi]), acc[2 * p + j][mi]);
        }
      }
    }
  }
  // lane (c, q), register (j, mi, i): token 16 mi + c, expert e0 + 32 q + 8 i + j. Runs of four
  // experts: run n holds 32 q + 4 n ..
#pragma unroll
  for (int mi = 0; mi < 4; ++mi) {
    if (mi == w) continue;
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      const int i = n >> 1, j = 4 * (n & 1);
      red[mi][w < mi ? w : w - 1][n][lane] = floatx4{acc[j][mi][i], acc[j + 1][mi][i], acc[j + 2][mi][i], acc[j + 3][mi][i]};
    }
  }
  if (tile == 0) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      nn[j] += __shfl_xor(nn[j], 16, 64);
      nn[j] += __shfl_xor(nn[j], 32, 64);
      if (q == 0) nred[w][8 * c + j] = nn[j];
    }
  }
  __syncthreads();
  if (tile == 0 && threadIdx.x < 128 && e0 + (int)threadIdx.x < E)
    npart[ks * E + e0 + threadIdx.x] =
        ((nred[0][threadIdx.x] + nred[1][threadIdx.x]) + nred[2][threadIdx.x]) + nred[3][threadIdx.x];
#pragma unroll
  for (int mi = 0; mi < 4; ++mi) {
    if (mi != w) continue;
    const int t = t0 + 16 * mi + c;
    float* o = part + ((int64_t)ks * T + t) * E + e0 + 32 * q;
#pragma unroll
    for (int n = 0; n < 8; ++n) {
      const int i = n >> 1, j = 4 * (n & 1);
      floatx4 v = floatx4{acc[j][mi][i], acc[j + 1][mi][i], acc[j + 2][mi][i], acc[j + 3][mi][i]};
#pragma unroll
      for (int k = 0; k < kLogitWaves - 1; ++k) v += red[mi][k][n][lane];
      if (t < T && e0 + 32 * q + 4 * n < E) *reinterpret_cast<floatx4*>(o + 4 * n) = v;
    }
  }
}

// Order-preserving key of a float (-0.0 keyed as +0.0), as wave_topk.
__device__ __forceinline__ uint32_t float_key(float v) {
  const uint32_t u = __float_as_uint(v == 0.0f ? 0.0f : v);
  return (u >> 31) ? ~u : (u | 0x80000000u);
}

constexpr float kNormFloor = 0x1p-100f;  // of a squared norm
constexpr int kSelectWaves = 4;        // tokens per block of k_route_select, one wave each
constexpr int kRouteSliceBytes = 144;  // a 64-element bf16 slice of x in LDS, padded by 16 bytes

// One wave per token (no block barrier): the bound and the candidates from the
// partial logits, their canonical logits (P lanes per chain, the slice count rounded
// up to a power of two; 64 / P chains side by side, two rounds of them in flight),
// rank, softmax, and the per-64-token expert counts.
template <int EPL, int P>
__global__ __launch_bounds__(64 * kSelectWaves, EPL <= 2 ? 4 : 2) void k_route_select(
    int T, int D, int E, int K, int KS, const uint16_t* __restrict__ x, const uint16_t* __restrict__ rtq,
    const float* __restrict__ npart, const float* __restrict__ part, float cbound, int32_t* __restrict__ topk_idx,
    float* __restrict__ topk_w, int32_t* __restrict__ hist, int out_bf16) {
  static_assert(EPL <= 4, "experts per lane");
  constexpr int CP = 64 / P;  // chains side by side in a wave
  __shared__ TopkLds tk[kSelectWaves];
  __shared__ __attribute__((aligned(16))) uint8_t xlds[kSelectWaves][P * kRouteSliceBytes];
  __shared__ int32_t cand_lds[kSelectWaves][64 * EPL];
  __shared__ float cval_lds[kSelectWaves][64 * EPL];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int t = blockIdx.x * kSelectWaves + w;
  if (t >= T) return;
  int32_t* cand = cand_lds[w];
  float* cval = cval_lds[w];
  const int S = D >> 6;
  const int s = lane % P, g = lane / P;
  // everything the bound needs, requested together: the lane's slice of x, the
  // partial logits and the column norms of its experts
  // (through LDS: read a slice per lane, a row's 16-byte pieces are 128 bytes apart
  // and every load of the eight touches every cache line of the row)
  uint8_t* xl = xlds[w];
  const int pieces = D >> 3;
  uint4 xv[8];
#pragma unroll
  for (int i = 0; i < P / 8; ++i)
    if (lane + 64 * i < pieces) xv[i] = reinterpret_cast<const uint4*>(x + (int64_t)t * D)[lane + 64 * i];
  float pl[EPL][kRouteMaxSplits], pn[EPL][kRouteMaxSplits];
#pragma unroll
  for (int i = 0; i < EPL; ++i)
#pragma unroll
    for (int k = 0; k < kRouteMaxSplits; ++k) {
      const bool on = k < KS && lane + 64 * i < E;
      pl[i][k] = on ? part[((int64_t)k * T + t) * E + lane + 64 * i] : 0.0f;
      pn[i][k] = on ? npart[k * E + lane + 64 * i] : 0.0f;
    }
#pragma unroll
  for (int i = 0; i < P / 8; ++i) {
    const int pc = lane + 64 * i;
    if (pc < pieces) *reinterpret_cast<uint4*>(xl + (pc >> 3) * kRouteSliceBytes + (pc & 7) * 16) = xv[i];
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int i = 0; i < 8; ++i)
    xv[i] = s < S ? *reinterpret_cast<const uint4*>(xl + s * kRouteSliceBytes + 16 * i) : uint4{0u, 0u, 0u, 0u};
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const uint32_t wd[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float lo = __uint_as_float(wd[j] << 16), hi = __uint_as_float(wd[j] & 0xffff0000u);
      ss = __builtin_fmaf(lo, lo, ss);
      ss = __builtin_fmaf(hi, hi, ss);
    }
  }
#pragma unroll
  for (int o = 1; o < P; o <<= 1) ss += __shfl_xor(ss, o, 64);
  const float nxv = sqrtf(ss < kNormFloor ? kNormFloor : ss);
  float lo[EPL], hi[EPL];
  bool bad = !(nxv <= 3.0e38f);
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    lo[i] = -INFINITY;
    hi[i] = -INFINITY;
    if (lane + 64 * i < E) {
      float v = pl[i][0], n2 = pn[i][0];
#pragma unroll
      for (int k = 1; k < kRouteMaxSplits; ++k) {
        v += pl[i][k];
        n2 += pn[i][k];
      }
      const float dl = __builtin_fmaf(cbound * nxv, sqrtf(n2 < kNormFloor ? kNormFloor : n2), 1e-30f);
      lo[i] = v - dl;
      hi[i] = v + dl;
      bad = bad || !(lo[i] >= -3.0e38f && hi[i] <= 3.0e38f);
    }
  }
  const bool all = __ballot(bad) != 0ull;
  // tau: a lower bound of the K-th largest lo, to 16 key bits
  uint32_t lk[EPL];
#pragma unroll
  for (int i = 0; i < EPL; ++i) lk[i] = lane + 64 * i < E ? float_key(lo[i]) : 0u;
  uint32_t thr = 0;
  if (!all) {
    for (int b = 31; b >= 16; --b) {
      const uint32_t c = thr | (1u << b);
      int cnt = 0;
#pragma unroll
      for (int i = 0; i < EPL; ++i) cnt += __popcll(__ballot(lk[i] >= c));
      if (cnt >= K) thr = c;
    }
  }
  // the candidates, in expert order
  const unsigned long long below = (1ull << lane) - 1ull;
  int nc = 0;
#pragma unroll
  for (int i = 0; i < EPL; ++i) {
    const int e = lane + 64 * i;
    const bool c = e < E && (all || float_key(hi[i]) >= thr);
    const unsigned long long mk = __ballot(c);
    if (c) cand[nc + __popcll(mk & below)] = e;
    nc += __popcll(mk);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  // canonical logits of the candidates: lane s of a group of P runs slice s of
  // candidates g, g + CP, ... (x[64 s ..] times r[64 s ..][e], one fmaf chain
  // from +0), then the pairwise tree over the P slices
  auto piece = [&](int c, int i) {
    // chains past the candidates do no loads and are not stored
    return s < S && c < nc ? reinterpret_cast<const uint4*>(rtq + ((int64_t)cand[c] * 8 * S + s) * 8)[(int64_t)i * S]
                           : uint4{0u, 0u, 0u, 0u};
  };
  for (int cb = 0; cb < nc; cb += 2 * CP) {
    const int c0 = cb + g, c1 = cb + CP + g;
    uint4 r0[8], r1[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      r0[i] = piece(c0, i);
      r1[i] = piece(c1, i);
    }
    float a0 = 0.0f, a1 = 0.0f;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      // (x stays packed across the rounds: its 64 floats would cost half the waves)
      asm volatile("" : "+v"(xv[i].x), "+v"(xv[i].y), "+v"(xv[i].z), "+v"(xv[i].w));
      const uint32_t xw[4] = {xv[i].x, xv[i].y, xv[i].z, xv[i].w};
      const uint32_t w0[4] = {r0[i].x, r0[i].y, r0[i].z, r0[i].w};
      const uint32_t w1[4] = {r1[i].x, r1[i].y, r1[i].z, r1[i].w};
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float xl = __uint_as_float(xw[j] << 16), xh = __uint_as_float(xw[j] & 0xffff0000u);
        a0 = __builtin_fmaf(xl, __uint_as_float(w0[j] << 16), a0);
        a1 = __builtin_fmaf(xl, __uint_as_float(w1[j] << 16), a1);
        a0 = __builtin_fmaf(xh, __uint_as_float(w0[j] & 0xffff0000u), a0);
        a1 = __builtin_fmaf(xh, __uint_as_float(w1[j] & 0xffff0000u), a1);
      }
    }
#pragma unroll
    for (int st = 1; st < P; st <<= 1) {
      a0 = a0 + __shfl_down(a0, st, P);
      a1 = a1 + __shfl_down(a1, st, P);
    }
    if (s == 0 && c0 < nc) cval[c0] = a0;
    if (s == 0 && c1 < nc) cval[c1] = a1;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  if (nc <= 64) {
    // rank the candidates (value descending, ties to the lower expert; NaN as
    // -inf), then the softmax of the first K in rank order (the sum in rank
    // order, as wave_topk)
    float mv = -INFINITY;
    int me = 0x7fffffff, rank = 0;
    if (lane < nc) {
      const float q = cval[lane];
      mv = q == q ? q : -INFINITY;
      me = cand[lane];
      for (int c = 0; c < nc; ++c) {
        const float qc0 = cval[c];
        const float qc = qc0 == qc0 ? qc0 : -INFINITY;
        rank += (qc > mv) || (qc == mv && cand[c] < me);
      }
    }
    if (lane < nc && rank < K) {
      tk[w].sidx[rank] = me;
      tk[w].key[rank] = __float_as_uint(mv);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const float l0 = __uint_as_float(tk[w].key[0]);
    const float ej = lane < K ? expf(__uint_as_float(tk[w].key[lane]) - l0) : 0.0f;
    float ssum = 0.0f;
    for (int j = 0; j < K; ++j) ssum = ssum + __shfl(ej, j, 64);
    if (lane < K) {
      const int e = tk[w].sidx[lane];
      const float p = ej / ssum;
      topk_w[(int64_t)t * K + lane] = out_bf16 ? round_bf16(p) : p;
      topk_idx[(int64_t)t * K + lane] = e;
      atomicAdd(&hist[(int64_t)(t / kDispatchBlock) * E + e], 1);
    }
  } else {
    // more than 64 candidates (a token taking every expert): wave_topk over the
    // canonical logits by expert; the candidate list is increasing in expert
    float v[EPL];
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
      const int e = lane + 64 * i;
      v[i] = -INFINITY;
      if (e < E) {
        int a = 0, z = nc - 1;
        while (a < z) {
          const int mid = (a + z) >> 1;
          if (cand[mid] < e)
            a = mid + 1;
          else
            z = mid;
        }
        if (cand[a] == e) {
          const float q = cval[a];
          v[i] = q == q ? q : -INFINITY;
        }
      }
    }
    wave_topk<EPL>(t, E, K, v, topk_idx, topk_w, out_bf16, nullptr, tk[w]);
    if (lane < K) atomicAdd(&hist[(int64_t)(t / kDispatchBlock) * E + topk_idx[(int64_t)t * K + lane]], 1);
  }
}

}  // namespace kmoe

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
namespace kmoe_host {

using namespace kmoe;

struct RouteShape {
  int S, P, EPL, LPR, SPW, G, NWB, TB;
  size_t lds;
};

static RouteShape route_shape(const kmoe_desc& d) {
  RouteShape r;
  const int D = (int)d.hidden, E = (int)d.num_experts;
  const int T = (int)d.tokens;
  r.S = (D + kRouterSlice - 1) / kRouterSlice;
  r.P = 1;
  while (r.P < r.S) r.P <<= 1;
  r.EPL = E <= 512 ? 8 : 16;
  r.LPR = (E + r.EPL - 1) / r.EPL;
  r.SPW = 1;
  while (2 * r.SPW * r.LPR <= 64) r.SPW <<= 1;
  const int NG = r.P > r.SPW ? r.P / r.SPW : 1;
  r.G = NG > 16 ? NG / 16 : 1;
  r.NWB = NG / r.G;
  // tokens per block: accumulators within the register budget, x stage <= 80 KB
  // (two blocks per CU), partials <= 64 KB, and enough blocks to cover the chip
  int tb = 8;
  const int acc_cap = r.G > 1 ? 2 * r.EPL : 64;
  auto x_bytes = [&](int t) { return (size_t)4 * r.S * (kRouterSlice * t + 4); };
  auto part_bytes = [&](int t) { return (size_t)4 * r.NWB * t * E + r.NWB * sizeof(TopkLds); };
  while (tb > 1 && (tb * r.EPL > acc_cap || x_bytes(tb) > 81920 || part_bytes(tb) > 65536)) tb >>= 1;
  // two blocks per CU where four tokens per block still give them (T = 2048:
  // 35.9 -> 32.3 us); fewer tokens per block re-read the router too often
  while (tb > 4 && (T + tb - 1) / tb < 512) tb >>= 1;
  while (tb > 1 && (T + tb - 1) / tb < 256) tb >>= 1;
  r.TB = tb;
  r.lds = std::max(x_bytes(tb), part_bytes(tb));
  return r;
}

template <typename A, int RT, int EPL, int TB, int G>
static void launch_route_k(const kmoe_desc& d, const RouteShape& rs, const void* x, const kmoe_weight& r,
                           float* logits, int32_t* topk_idx, float* topk_w, hipStream_t st) {
  const int T = (int)d.tokens, D = (int)d.hidden, E = (int)d.num_experts, K = (int)d.top_k;
  const int scale_bf16 = (r.dtype == KMOE_DTYPE_I8 && r.scale_dtype == KMOE_DTYPE_BF16) ? 1 : 0;
  const int scale_pc = (r.dtype == KMOE_DTYPE_I8 && r.scale_kind == KMOE_SCALE_CHANNEL) ? 1 : 0;
  const int out_bf16 = d.act_dtype == KMOE_DTYPE_BF16 ? 1 : 0;
  hipLaunchKernelGGL((k_route<A, RT, EPL, TB, G>), dim3((T + TB - 1) / TB), dim3(64 * rs.NWB), rs.lds, st, T, D, E,
                     K, rs.LPR, rs.SPW, rs.P, reinterpret_cast<const A*>(x), r.values, r.scale, scale_bf16,
                     scale_pc, logits, topk_idx, topk_w, out_bf16);
}

template <typename A, int RT, int EPL>
static void route_tb(const kmoe_desc& d, const RouteShape& rs, const void* x, const kmoe_weight& r, float* logits,
                     int32_t* idx, float* w, hipStream_t st) {
  if (rs.G == 4) {
    if (rs.TB == 2) return launch_route_k<A, RT, EPL, 2, 4>(d, rs, x, r, logits, idx, w, st);
    return launch_route_k<A, RT, EPL, 1, 4>(d, rs, x, r, logits, idx, w, st);
  }
  if (rs.G == 2) {
    if (rs.TB == 2) return launch_route_k<A, RT, EPL, 2, 2>(d, rs, x, r, logits, idx, w, st);
    return launch_route_k<A, RT, EPL, 1, 2>(d, rs, x, r, logits, idx, w, st);
  }
  switch (rs.TB) {
    case 8:
      if constexpr (EPL == 8) return launch_route_k<A, RT, EPL, 8, 1>(d, rs, x, r, logits, idx, w, st);
      [[fallthrough]];
    case 4:
      if constexpr (EPL == 8) return launch_route_k<A, RT, EPL, 4, 1>(d, rs, x, r, logits, idx, w, st);
      [[fallthrough]];
    case 2:
      return launch_route_k<A, RT, EPL, 2, 1>(d, rs, x, r, logits, idx, w, st);
    default:
      return launch_route_k<A, RT, EPL, 1, 1>(d, rs, x, r, logits, idx, w, st);
  }
}

template <typename A, int RT>
static void route_epl(const kmoe_desc& d, const RouteShape& rs, const void* x, const kmoe_weight& r, float* logits,
                      int32_t* idx, float* w, hipStream_t st) {
  if (rs.EPL == 8) return route_tb<A, RT, 8>(d, rs, x, r, logits, idx, w, st);
  return route_tb<A, RT, 16>(d, rs, x, r, logits, idx, w, st);
}

template <typename A>
static void route_rt(const kmoe_desc& d, const RouteShape& rs, const void* x, const kmoe_weight& r, float* logits,
                     int32_t* idx, float* w, hipStream_t st) {
  if (r.dtype == KMOE_DTYPE_F32) return route_epl<A, 0>(d, rs, x, r, logits, idx, w, st);
  if (r.dtype == KMOE_DTYPE_BF16) return route_epl<A, 1>(d, rs, x, r, logits, idx, w, st);
  return route_epl<A, 2>(d, rs, x, r, logits, idx, w, st);
}

hipError_t launch_route(const kmoe_desc& d, const void* x, const kmoe_weight& r, float* logits, int32_t* topk_idx,
                        float* topk_w, int32_t* hist, hipStream_t st) {
  const RouteShape rs = route_shape(d);
  if (d.act_dtype == KMOE_DTYPE_BF16)
    route_rt<uint16_t>(d, rs, x, r, logits, topk_idx, topk_w, st);
  else
    route_rt<float>(d, rs, x, r, logits, topk_idx, topk_w, st);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess || !hist) return err;
  return launch_dispatch_count(d, topk_idx, hist, st);
}

hipError_t launch_dispatch_count(const kmoe_desc& d, const int32_t* topk_idx, int32_t* hist, hipStream_t st) {
  const int T = (int)d.tokens, E = (int)d.num_experts, K = (int)d.top_k;
  const int nblk = (T + kDispatchBlock - 1) / kDispatchBlock;
  hipLaunchKernelGGL(k_dispatch_count, dim3(nblk), dim3(256), 0, st, T, E, K, topk_idx, hist);
  return hipGetLastError();
}

// Split router: experts per lane for the slice kernel (>= 4 bytes of weights
// per row and lane, at most 64 lanes per row), tokens per block, group count.
struct SplitShape {
  int EPL, TB, P, Q;
};

static SplitShape split_shape(const kmoe_desc& d, const kmoe_weight& r) {
  SplitShape sh;
  const int E = (int)d.num_experts, T = (int)d.tokens;
  const int S = (int)((d.hidden + kRouterSlice - 1) / kRouterSlice);
  const int min_epl = r.dtype == KMOE_DTYPE_F32 ? 1 : (r.dtype == KMOE_DTYPE_BF16 ? 2 : 4);
  sh.EPL = min_epl;
  while (sh.EPL * 64 < E) sh.EPL <<= 1;
  sh.TB = T <= 16 ? 1 : (T <= 64 ? 2 : 4);
  sh.P = 1;
  while (sh.P < S) sh.P <<= 1;
  sh.Q = route_split_groups(d);
  return sh;
}

template <typename A, int RT, int EPL, int TB>
static void launch_slices(const kmoe_desc& d, const SplitShape& sh, const void* x, const kmoe_weight& r, float* part,
                          const SliceNorm& nm, hipStream_t st) {
  const int T = (int)d.tokens, D = (int)d.hidden, E = (int)d.num_experts;
  const int scale_bf16 = (r.dtype == KMOE_DTYPE_I8 && r.scale_dtype == KMOE_DTYPE_BF16) ? 1 : 0;
  const int scale_pc = (r.dtype == KMOE_DTYPE_I8 && r.scale_kind == KMOE_SCALE_CHANNEL) ? 1 : 0;
  const size_t lds = nm.scale ? (size_t)TB * NormRow<A>::bytes(D) : 0;
  hipLaunchKernelGGL((k_route_slices<A, RT, EPL, TB>), dim3(sh.Q, (T + TB - 1) / TB), dim3(256), lds, st, T, D, E,
                     sh.P, sh.Q, reinterpret_cast<const A*>(x), r.values, r.scale, scale_bf16, scale_pc, part, nm);
}

template <typename A, int RT, int EPL>
static void slices_tb(const kmoe_desc& d, const SplitShape& sh, const void* x, const kmoe_weight& r, float* part,
                      const SliceNorm& nm, hipStream_t st) {
  if (sh.TB == 1) return launch_slices<A, RT, EPL, 1>(d, sh, x, r, part, nm, st);
  if (sh.TB == 2) return launch_slices<A, RT, EPL, 2>(d, sh, x, r, part, nm, st);
  return launch_slices<A, RT, EPL, 4>(d, sh, x, r, part, nm, st);
}

template <typename A, int RT>
static void slices_epl(const kmoe_desc& d, const SplitShape& sh, const void* x, const kmoe_weight& r, float* part,
                       const SliceNorm& nm, hipStream_t st) {
  switch (sh.EPL) {
    case 1:
      if constexpr (RT == 0) return slices_tb<A, RT, 1>(d, sh, x, r, part, nm, st);
      [[fallthrough]];
    case 2:
      if constexpr (RT != 2) return slices_tb<A, RT, 2>(d, sh, x, r, part, nm, st);
      [[fallthrough]];
    case 4:
      return slices_tb<A, RT, 4>(d, sh, x, r, part, nm, st);
    case 8:
      return slices_tb<A, RT, 8>(d, sh, x, r, part, nm, st);
    default:
      return slices_tb<A, RT, 16>(d, sh, x, r, part, nm, st);
  }
}

template <typename A>
static void slices_rt(const kmoe_desc& d, const SplitShape& sh, const void* x, const kmoe_weight& r, float* part,
                      const SliceNorm& nm, hipStream_t st) {
  if (r.dtype == KMOE_DTYPE_F32) return slices_epl<A, 0>(d, sh, x, r, part, nm, st);
  if (r.dtype == KMOE_DTYPE_BF16) return slices_epl<A, 1>(d, sh, x, r, part, nm, st);
  return slices_epl<A, 2>(d, sh, x, r, part, nm, st);
}

template <int EPL>
static void launch_finish(const kmoe_desc& d, const SplitShape& sh, const float* part, float* logits,
                          int32_t* topk_idx, float* topk_w, const DispatchOut* ds, hipStream_t st) {
  const int T = (int)d.tokens, E = (int)d.num_experts, K = (int)d.top_k;
  const int out_bf16 = d.act_dtype == KMOE_DTYPE_BF16 ? 1 : 0;
  if (ds && T <= 4)
    hipLaunchKernelGGL((k_route_finish_dispatch<EPL, 4>), dim3(1), dim3(256), 0, st, T, E, K, sh.Q, part, logits,
                       topk_idx, topk_w, out_bf16, ds->group_sizes, ds->offsets, ds->active, ds->sorted_token,
                       ds->sorted_expert, ds->inv, capacity_of(d));
  else if (ds)
    hipLaunchKernelGGL((k_route_finish_dispatch<EPL, 16>), dim3(1), dim3(1024), 0, st, T, E, K, sh.Q, part, logits,
                       topk_idx, topk_w, out_bf16, ds->group_sizes, ds->offsets, ds->active, ds->sorted_token,
                       ds->sorted_expert, ds->inv, capacity_of(d));
  else
    hipLaunchKernelGGL((k_route_finish<EPL>), dim3((T + 3) / 4), dim3(256), 0, st, T, E, K, sh.Q, part, logits,
                       topk_idx, topk_w, out_bf16);
}

hipError_t launch_route_slices(const kmoe_desc& d, const void* x, const kmoe_weight& r, float* part, hipStream_t st,
                               const SliceNorm* norm) {
  const SplitShape sh = split_shape(d, r);
  const SliceNorm nm = norm ? *norm : SliceNorm{nullptr, 0, 0.0f, nullptr};
  if (d.act_dtype == KMOE_DTYPE_BF16)
    slices_rt<uint16_t>(d, sh, x, r, part, nm, st);
  else
    slices_rt<float>(d, sh, x, r, part, nm, st);
  return hipGetLastError();
}

hipError_t launch_route_split(const kmoe_desc& d, const void* x, const kmoe_weight& r, float* part, float* logits,
                              int32_t* topk_idx, float* topk_w, hipStream_t st, const SliceNorm* norm,
                              const DispatchOut* dispatch) {
  // the dispatch rides along when the finish is a single block
  const DispatchOut* ds = dispatch && split_router_dispatches(d) ? dispatch : nullptr;
  const SplitShape sh = split_shape(d, r);
  const SliceNorm nm = norm ? *norm : SliceNorm{nullptr, 0, 0.0f, nullptr};
  if (d.act_dtype == KMOE_DTYPE_BF16)
    slices_rt<uint16_t>(d, sh, x, r, part, nm, st);
  else
    slices_rt<float>(d, sh, x, r, part, nm, st);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  const int E = (int)d.num_experts;
  if (E <= 64)
    launch_finish<1>(d, sh, part, logits, topk_idx, topk_w, ds, st);
  else if (E <= 128)
    launch_finish<2>(d, sh, part, logits, topk_idx, topk_w, ds, st);
  else if (E <= 256)
    launch_finish<4>(d, sh, part, logits, topk_idx, topk_w, ds, st);
  else if (E <= 512)
    launch_finish<8>(d, sh, part, logits, topk_idx, topk_w, ds, st);
  else
    launch_finish<16>(d, sh, part, logits, topk_idx, topk_w, ds, st);
  return hipGetLastError();
}

hipError_t launch_dispatch(const kmoe_desc& d, const int32_t* topk_idx, const int32_t* hist, int32_t* group_sizes,
                           int32_t* offsets, int32_t* active, int32_t* sorted_token, int32_t* sorted_expert,
                           int32_t* inv, hipStream_t st) {
  const int T = (int)d.tokens, E = (int)d.num_experts, K = (int)d.top_k;
  const int nblk = (T + kDispatchBlock - 1) / kDispatchBlock;
  if (!hist && nblk > 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_dispatch_scatter, dim3(nblk), dim3(256), 0, st, T, E, K, nblk, topk_idx, hist, group_sizes,
                     offsets, active, sorted_token, sorted_expert, inv, capacity_of(d));
  return hipGetLastError();
}

// Two-phase router: the partial logits (with the transposed router, its column
// norms and the histograms zeroed), then the bound, the candidates' canonical
// logits, top-k, softmax and the per-64-token expert counts (launch_dispatch
// reads them as it reads k_dispatch_count's).
template <int EPL>
static void route_select_p(const kmoe_desc& d, int KS, const uint16_t* x, const uint16_t* rtq, const float* npart,
                           const float* part, float cb, int32_t* topk_idx, float* topk_w, int32_t* hist,
                           hipStream_t st) {
  const int T = (int)d.tokens, D = (int)d.hidden, E = (int)d.num_experts, K = (int)d.top_k;
  const dim3 grid((T + kSelectWaves - 1) / kSelectWaves), block(64 * kSelectWaves);
  const int out_bf16 = d.act_dtype == KMOE_DTYPE_BF16 ? 1 : 0;
  const int S = D / 64;
  // P lanes per candidate chain: the slice count rounded up to a power of two
  if (S <= 8)
    hipLaunchKernelGGL((k_route_select<EPL, 8>), grid, block, 0, st, T, D, E, K, KS, x, rtq, npart, part, cb, topk_idx,
                       topk_w, hist, out_bf16);
  else if (S <= 16)
    hipLaunchKernelGGL((k_route_select<EPL, 16>), grid, block, 0, st, T, D, E, K, KS, x, rtq, npart, part, cb, topk_idx,
                       topk_w, hist, out_bf16);
  else if (S <= 32)
    hipLaunchKernelGGL((k_route_select<EPL, 32>), grid, block, 0, st, T, D, E, K, KS, x, rtq, npart, part, cb, topk_idx,
                       topk_w, hist, out_bf16);
  else
    hipLaunchKernelGGL((k_route_select<EPL, 64>), grid, block, 0, st, T, D, E, K, KS, x, rtq, npart, part, cb, topk_idx,
                       topk_w, hist, out_bf16);
}

hipError_t launch_route_mfma(const kmoe_desc& d, const void* x, const kmoe_weight& r, void* scratch,
                             int32_t* topk_idx, float* topk_w, int32_t* hist, hipStream_t st) {
  const int T = (int)d.tokens, D = (int)d.hidden, E = (int)d.num_experts;
  const int KS = route_mfma_splits(d);
  char* base = reinterpret_cast<char*>(scratch);
  uint16_t* rtq = reinterpret_cast<uint16_t*>(base);
  float* npart = reinterpret_cast<float*>(base + route_mfma_scratch_offsets(d, 1));
  float* part = reinterpret_cast<float*>(base + route_mfma_scratch_offsets(d, 2));
  const int nhist = ((T + kDispatchBlock - 1) / kDispatchBlock) * E;
  const uint16_t* xb = reinterpret_cast<const uint16_t*>(x);
  const uint16_t* rb = reinterpret_cast<const uint16_t*>(r.values);
  hipLaunchKernelGGL(k_route_logits, dim3((T + 63) / 64, KS, (E + 127) / 128), dim3(64 * kLogitWaves), 0, st, T, D, E,
                     KS, xb, rb, rtq, npart, part, hist, nhist);
  hipError_t err = hipGetLastError();
  if (err != hipSuccess) return err;
  // the error bound's constant, relative to ||x|| ||r_e||: the MFMA sums as up
  // to 2D roundings of up to 2u, the canonical chains and tree, the norms and
  // lo / hi, with room to spare
  const float cb = (float)std::ldexp(4.0 * D + 512.0, -24);
  if (E <= 64)
    route_select_p<1>(d, KS, xb, rtq, npart, part, cb, topk_idx, topk_w, hist, st);
  else if (E <= 128)
    route_select_p<2>(d, KS, xb, rtq, npart, part, cb, topk_idx, topk_w, hist, st);
  else
    route_select_p<4>(d, KS, xb, rtq, npart, part, cb, topk_idx, topk_w, hist, st);
  return hipGetLastError();
}

}  // namespace kmoe_host
