// The steps on either side of the MoE block in a Qwen3 MoE layer
// (kappa/qwen3/block.py:196-207): the pre-FFN RMSNorm that produces the
// block's input, and (in the combine kernels of expert.hip) the residual add
// of its output.
//
// rms_norm (kappa/qwen3/norms.py:10-16) in a canonical order shared with the
// oracle: the squares f32(h)*f32(h), each rounded to float, are summed per
// 64-wide slice in a sequential chain from +0.0f, and the slice sums are
// combined by the same zero-padded pairwise tree as the router logits;
// var = S / D, r = 1 / sqrt(var + eps) with IEEE division and square root, and
// h2 = round_act((f32(h) * r) * f32(scale)).
#include "common.h"
#include "launch.h"
#include "norm.h"

namespace kmoe {

constexpr int kNormWaves = 4;  // tokens per block, one wave each

// 16 bytes (or the run of 16-byte loads) of the scale that go with a piece of the row
template <typename A, typename S>
__device__ __forceinline__ void scale_piece(const S* __restrict__ scale, int piece, float* f) {
  constexpr int n = NormRow<A>::kPiece;
  if constexpr (sizeof(S) == 2 && n == 4) {
    const uint2 v = reinterpret_cast<const uint2*>(scale)[piece];
    f[0] = __uint_as_float(v.x << 16), f[1] = __uint_as_float(v.x & 0xffff0000u);
    f[2] = __uint_as_float(v.y << 16), f[3] = __uint_as_float(v.y & 0xffff0000u);
  } else {
    constexpr int per = NormRow<S>::kPiece;
#pragma unroll
    for (int i = 0; i < n / per; ++i)
      NormRow<S>::unpack(reinterpret_cast<const uint4*>(scale)[piece * (n / per) + i], f + i * per);
  }
}

// One wave per token: wave_rms_factor stages the row in LDS and reduces it,
// then the wave writes round_act((x * r) * scale) from the pieces it still holds.
// Latency: one row's round trip, its 64-step chain and the store (33 MB at 30B-A3B
// T = 4096: 11.7 us; element by element, with the row in LDS as floats, 17 us).
template <typename A, typename S>
__global__ __launch_bounds__(256) void k_rms_norm(int T, int D, float eps, const A* __restrict__ h,
                                                   const S* __restrict__ scale, A* __restrict__ out) {
  using R = NormRow<A>;
  extern __shared__ __attribute__((aligned(16))) uint8_t rows[];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int t = blockIdx.x * kNormWaves + w;
  if (t >= T) return;  // per wave: this kernel has no block-wide barrier
  A* row = reinterpret_cast<A*>(rows + (size_t)w * R::bytes(D));
  const A* src = h + (int64_t)t * D;
  A* dst = out + (int64_t)t * D;
  uint4 v[R::kPieces];
  const float r = wave_rms_factor(src, D, eps, row, v);
  if (R::pieces(src, D) && ((reinterpret_cast<uintptr_t>(dst) | reinterpret_cast<uintptr_t>(scale)) & 15) == 0) {
    const int n = D / R::kPiece;
#pragma unroll
    for (int i = 0; i < R::kPieces; ++i) {
      const int p = lane + 64 * i;
      if (p < n) {
        float f[R::kPiece], sc[R::kPiece];
        R::unpack(v[i], f);
        scale_piece<A, S>(scale, p, sc);
        uint32_t o[4];
#pragma unroll
        for (int j = 0; j < R::kPiece; ++j) f[j] = rms_apply<A>(f[j], r, sc[j]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          if constexpr (sizeof(A) == 2)
            o[j] = (uint32_t)f32_to_bf16_bits(f[2 * j]) | ((uint32_t)f32_to_bf16_bits(f[2 * j + 1]) << 16);
          else
            o[j] = __float_as_uint(f[j]);
        }
        reinterpret_cast<uint4*>(dst)[p] = uint4{o[0], o[1], o[2], o[3]};
      }
    }
    return;
  }
  if constexpr (sizeof(A) == 2) {
    for (int d = lane; d < D; d += 64)
      Act<A>::store(dst, d, rms_apply<A>(Act<A>::load(row, R::at(d)), r, Act<S>::load(scale, d)));
    return;
  }
  for (int base = 0; base < D; base += 64 * R::kBatch) {
    float sc[R::kBatch];
#pragma unroll
    for (int j = 0; j < R::kBatch; ++j) sc[j] = Act<S>::load(scale, min(base + 64 * j + lane, D - 1));
#pragma unroll
    for (int j = 0; j < R::kBatch; ++j) {
      const int d = base + 64 * j + lane;
      if (d < D) Act<A>::store(dst, d, rms_apply<A>(Act<A>::load(row, R::at(d)), r, sc[j]));
    }
  }
}

}  // namespace kmoe

namespace kmoe_host {

using namespace kmoe;


hipError_t launch_rms_norm(const kmoe_desc& d, const void* h, const void* scale, kmoe_dtype scale_dtype, float eps,
                           void* out, hipStream_t st) {
  const int T = (int)d.tokens, D = (int)d.hidden;
  if (T == 0) return hipSuccess;
  const dim3 grid((T + kNormWaves - 1) / kNormWaves);
  const bool act_bf16 = d.act_dtype == KMOE_DTYPE_BF16, s_bf16 = scale_dtype == KMOE_DTYPE_BF16;
  const size_t lds = kNormWaves * (act_bf16 ? NormRow<uint16_t>::bytes(D) : NormRow<float>::bytes(D));
  if (act_bf16 && s_bf16)
    hipLaunchKernelGGL((k_rms_norm<uint16_t, uint16_t>), grid, dim3(64 * kNormWaves), lds, st, T, D, eps,
                       reinterpret_cast<const uint16_t*>(h), reinterpret_cast<const uint16_t*>(scale),
                       reinterpret_cast<uint16_t*>(out));
  else if (act_bf16)
    hipLaunchKernelGGL((k_rms_norm<uint16_t, float>), grid, dim3(64 * kNormWaves), lds, st, T, D, eps,
                       reinterpret_cast<const uint16_t*>(h), reinterpret_cast<const float*>(scale),
                       reinterpret_cast<uint16_t*>(out));
  else if (s_bf16)
    hipLaunchKernelGGL((k_rms_norm<float, uint16_t>), grid, dim3(64 * kNormWaves), lds, st, T, D, eps,
                       reinterpret_cast<const float*>(h), reinterpret_cast<const uint16_t*>(scale),
                       reinterpret_cast<float*>(out));
  else
    hipLaunchKernelGGL((k_rms_norm<float, float>), grid, dim3(64 * kNormWaves), lds, st, T, D, eps,
                       reinterpret_cast<const float*>(h), reinterpret_cast<const float*>(scale),
                       reinterpret_cast<float*>(out));
  return hipGetLastError();
}

}  // namespace kmoe_host
