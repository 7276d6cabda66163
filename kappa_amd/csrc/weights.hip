// Weight-side kernels: the one-time relayout of W8 experts for the gfx950
// kernels, to_compute_dtype (kappa/qwen3/quant.py:34-38) and the per-channel
// int8 quantiser (kappa/qwen3/quant.py:41-48 with a per-channel max-abs).
#include <float.h>

#include "common.h"
#include "expert_dev.h"
#include "launch.h"

namespace kmoe {

__device__ __forceinline__ float scale_at(const void* s, int s_bf16, size_t i) {
  return s_bf16 ? bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(s)[i]) : reinterpret_cast<const float*>(s)[i];
}

// Four rows of four int8 columns (a dword per row) -> the four rows of each column
__device__ __forceinline__ void transpose4x4(const uint32_t* r, uint32_t* c) {
  const uint32_t a = __builtin_amdgcn_perm(r[1], r[0], 0x05010400u);  // r0c0 r1c0 r0c1 r1c1
  const uint32_t b = __builtin_amdgcn_perm(r[3], r[2], 0x05010400u);
  const uint32_t d = __builtin_amdgcn_perm(r[1], r[0], 0x07030602u);  // r0c2 r1c2 r0c3 r1c3
  const uint32_t f = __builtin_amdgcn_perm(r[3], r[2], 0x07030602u);
  c[0] = __builtin_amdgcn_perm(b, a, 0x05040100u);
  c[1] = __builtin_amdgcn_perm(b, a, 0x07060302u);
  c[2] = __builtin_amdgcn_perm(f, d, 0x05040100u);
  c[3] = __builtin_amdgcn_perm(f, d, 0x07060302u);
}

// A stacked int8 matrix [E][Kd][N] into cells of 16 columns x 16 k: dst
// [E][N/16][W][Kd/16][16 col][16 k], matrix `which` of W (w13: gate and up, W = 2;
// w2: W = 1). A thread takes 16 rows of four columns: one dword per row (a wave
// reads 256 consecutive bytes of each row, all 16 rows in flight) and four 16-byte
// stores, 64 consecutive bytes; the waves of a block take consecutive k groups,
// whose cells are consecutive. Bound by HBM: 30B-A3B gate + up + down (1.2 GB moved)
// 235-260 us (4.6-5.1 TB/s). One 16-byte cell per thread from 16 byte loads took
// 516 us.
// Source rows need no alignment.
__global__ __launch_bounds__(256) void k_pack(int Kd, int N, int W, const int8_t* __restrict__ src0,
                                              const int8_t* __restrict__ src1, int8_t* __restrict__ dst) {
  typedef uint32_t __attribute__((aligned(1))) u32_any;
  const int KG = Kd >> 4;
  // blocks over columns (fastest), k groups, matrices (one-dimensional: either extent
  // may exceed a grid's other dimensions)
  const uint32_t nx = ((N >> 2) + 63) >> 6, ny = (KG + 3) >> 2;
  const uint32_t bx = blockIdx.x % nx, bz = blockIdx.x / nx / ny, by = blockIdx.x / nx - bz * ny;
  const int quad = bx * 64 + (threadIdx.x & 63);  // four columns
  const int kg = by * 4 + (threadIdx.x >> 6);
  const int which = W == 2 ? (int)(bz & 1) : 0;
  const int64_t e = W == 2 ? bz >> 1 : bz;
  if (quad * 4 >= N || kg >= KG) return;
  const int8_t* src = (which ? src1 : src0) + (e * Kd + (int64_t)kg * 16) * N + quad * 4;
  uint32_t r[16];
#pragma unroll
  for (int k = 0; k < 16; ++k) r[k] = *reinterpret_cast<const u32_any*>(src + (int64_t)k * N);
  uint32_t c[4][4];  // [k quad][column]
#pragma unroll
  for (int k = 0; k < 4; ++k) transpose4x4(r + 4 * k, c[k]);
  int8_t* cell = dst + (((e * (N >> 4) + (quad >> 2)) * W + which) * KG + kg) * 256 + (quad & 3) * 64;
#pragma unroll
  for (int j = 0; j < 4; ++j) *reinterpret_cast<uint4*>(cell + 16 * j) = uint4{c[0][j], c[1][j], c[2][j], c[3][j]};
}

// s13 [E][I/16][2][16] and s2 [E][D]: the scales as given, in f32 (the kernels
// cast them to bf16 for the gather and fixed_capacity programs,
// kappa/qwen3/quant.py:37, and use them as they are for the ragged program's
// f32 dequantisation, kappa/qwen3/ffn_moe.py:203-205).
__global__ __launch_bounds__(256) void k_pack_scales(int E, int D, int I, const void* __restrict__ gs, int g_bf16,
                                                     int g_pc, const void* __restrict__ us, int u_bf16, int u_pc,
                                                     const void* __restrict__ ds, int d_bf16, int d_pc,
                                                     float* __restrict__ s13, float* __restrict__ s2) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t n13 = (int64_t)E * I * 2;
  if (i < n13) {
    const int col = (int)(i & 15);
    const int which = (int)((i >> 4) & 1);
    const int64_t r = i >> 5;
    const int ig = (int)(r % (I >> 4));
    const int64_t e = r / (I >> 4);
    const int64_t ch = e * I + ig * 16 + col;
    const float v = which ? scale_at(us, u_bf16, u_pc ? ch : 0) : scale_at(gs, g_bf16, g_pc ? ch : 0);
    s13[i] = v;
  } else if (i < n13 + (int64_t)E * D) {
    const int64_t j = i - n13;
    s2[j] = scale_at(ds, d_bf16, d_pc ? j : 0);
  }
}

// out[o, c] = to_compute_dtype(w)[o, c]; for int8 the scale of (o / rows_per_block, c).
template <typename O>
__global__ __launch_bounds__(256) void k_to_compute(int64_t outer, int64_t channels, int64_t rows_per_block,
                                                    const void* __restrict__ v, int wt, const void* __restrict__ s,
                                                    int s_bf16, int per_channel, O* __restrict__ out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= outer * channels) return;
  float r;
  if (wt == 0) {
    r = Act<O>::round(reinterpret_cast<const float*>(v)[i]);
  } else if (wt == 1) {
    r = bf16_bits_to_f32(reinterpret_cast<const uint16_t*>(v)[i]);
  } else {
    const int64_t o = i / channels, c = i - o * channels;
    const float sv = scale_at(s, s_bf16, per_channel ? (size_t)((o / rows_per_block) * channels + c) : 0);
    const float q = (float)reinterpret_cast<const int8_t*>(v)[i];
    r = Act<O>::kBf16 ? round_bf16(q * round_bf16(sv)) : q * sv;
  }
  Act<O>::store(out, i, r);
}

// One quantised value, clip(rint(w / sc), -128, 127), with the IEEE division.
__device__ __forceinline__ int quantize_one(float w, float sc) {
  float r = rintf(w / sc);
  r = fminf(fmaxf(r, -128.0f), 127.0f);
  return (int8_t)r;
}

__device__ __forceinline__ float channel_scale(float amax) {
  const float sc = amax / 127.0f;
  return sc > FLT_MIN ? sc : FLT_MIN;
}

// Per-output-channel quantiser over [E, Kd, N]: a block of 1024 threads per
// (64 columns, expert). A thread owns the 16 bytes of a row at its columns, one
// row of each sweep of the block; the first SW sweeps stay in registers between
// the maximum and the quantisation, so up to SW * 128 rows of bf16 (64 of f32) are
// read from memory once; rows beyond are read again. Column maxima meet by
// shuffles and in LDS.
//
// rint(w / sc) needs the correctly rounded quotient only near a tie: with inv =
// 1 / sc (rounded), the exact w * inv is within 127 * 2^-24 < 7.6e-6 of w / sc, and so
// is the rounded quotient, so wherever w * inv is at most 0.49995 from the nearest
// integer both round to that integer (in [-127, 127]; no clipping). Otherwise
// (1e-4 of the values; NaN and infinities fail the comparison too) the values of
// the load are divided.
//
// 30B-A3B gate, up and down (1.2 GB of bf16 in, 0.6 GB of int8 out) take 500 us
// (3.6 TB/s); one thread per column, which read the column twice and divided every
// element, took 4380 us. Sixteen sweeps leave one block per CU, whose load, reduce
// and store phases follow each other; persistent blocks that request the next
// item's sweeps while storing measured 179 us per matrix against 167.
template <typename Wt, int SW>
__global__ __launch_bounds__(1024, SW == 8 ? 8 : 4) void k_quantize_strip(int E, int Kd, int N,
                                                                          const Wt* __restrict__ w,
                                                                          int8_t* __restrict__ q,
                                                                          float* __restrict__ s) {
  constexpr int VPT = 16 / sizeof(Wt);  // columns per thread
  constexpr int TPR = 64 / VPT;         // threads per row
  constexpr int RPS = 1024 / TPR;       // rows per sweep
  __shared__ float part[16][64];
  __shared__ float scale[64];
  const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
  const int cp = tid % TPR, row0 = tid / TPR;
  // The strips of a 128-byte output line (a pair) run at block indices 8 apart, so on
  // one XCD at about the same time, and its L2 joins their 64-byte halves
  const int strips = (N + 63) >> 6, pairs = (strips + 1) >> 1;
  const int pair = (blockIdx.x >> 4) * 8 + (blockIdx.x & 7), strip = 2 * (pair % pairs) + ((blockIdx.x >> 3) & 1);
  const int64_t e = pair / pairs;
  if (e >= E || strip >= strips) return;
  const int col0 = strip * 64;
  const bool on = col0 + cp * VPT < N;
  // a thread's element offset from (uniform) sweep bases, below 2^31 bytes
  const uint32_t own = (uint32_t)row0 * (uint32_t)N + (uint32_t)(cp * VPT);
  const int64_t step = (int64_t)RPS * N;
  const Wt* we = w + e * Kd * N + col0;
  int8_t* qe = q + e * Kd * N + col0;
  auto load = [&](const Wt* base) { return load_stream16(reinterpret_cast<const int8_t*>(base + own)); };
  auto unpack = [](const uint4& v, float* f) {
    const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (sizeof(Wt) == 2) {
        f[2 * i] = __uint_as_float(d[i] << 16);
        f[2 * i + 1] = __uint_as_float(d[i] & 0xffff0000u);
      } else {
        f[i] = __uint_as_float(d[i]);
      }
    }
  };
  uint4 v[SW];
#pragma unroll
  for (int k = 0; k < SW; ++k) {
    v[k] = uint4{0u, 0u, 0u, 0u};
    if (on && k * RPS + row0 < Kd) v[k] = load(we + k * step);
  }
  float m[VPT], f[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) m[i] = 0.0f;
#pragma unroll
  for (int k = 0; k < SW; ++k) {
    unpack(v[k], f);
#pragma unroll
    for (int i = 0; i < VPT; ++i) m[i] = fmaxf(m[i], fabsf(f[i]));
  }
  for (int k = SW; on && k * RPS + row0 < Kd; ++k) {
    unpack(load(we + k * step), f);
#pragma unroll
    for (int i = 0; i < VPT; ++i) m[i] = fmaxf(m[i], fabsf(f[i]));
  }
#pragma unroll
  for (int o = TPR; o < 64; o <<= 1)
#pragma unroll
    for (int i = 0; i < VPT; ++i) m[i] = fmaxf(m[i], __shfl_xor(m[i], o, 64));
  if (lane < TPR) {
#pragma unroll
    for (int i = 0; i < VPT; ++i) part[wv][cp * VPT + i] = m[i];
  }
  __syncthreads();
  if (tid < 64) {
    float a = part[0][tid];
#pragma unroll
    for (int k = 1; k < 16; ++k) a = fmaxf(a, part[k][tid]);
    const float sc = channel_scale(a);
    scale[tid] = sc;
    if (col0 + tid < N) s[e * N + col0 + tid] = sc;
  }
  __syncthreads();
  float inv[VPT];
#pragma unroll
  for (int i = 0; i < VPT; ++i) inv[i] = 1.0f / scale[cp * VPT + i];
  auto store = [&](const uint32_t* r, int8_t* base) {  // the low bytes of r
    uint32_t o[VPT / 4];
#pragma unroll
    for (int i = 0; i < VPT / 4; ++i)
      o[i] = __builtin_amdgcn_perm(__builtin_amdgcn_perm(r[4 * i + 3], r[4 * i + 2], 0x0c0c0400u),
                                   __builtin_amdgcn_perm(r[4 * i + 1], r[4 * i], 0x0c0c0400u), 0x05040100u);
    if constexpr (VPT == 8)
      *reinterpret_cast<uint2*>(base + own) = uint2{o[0], o[1]};
    else
      *reinterpret_cast<uint32_t*>(base + own) = o[0];
  };
  // the values of one load by the reciprocal; false if one of them needs the division
  auto put = [&](const uint4& raw, int k) {
    constexpr float kMagic = 12582912.0f;  // 1.5 * 2^23: the sum's low bits are the rounded integer
    float x[VPT];
    unpack(raw, x);
    uint32_t r[VPT];
    bool sure = true;
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const float m = __builtin_fmaf(x[i], inv[i], kMagic);
      sure &= fabsf(__builtin_fmaf(x[i], inv[i], -(m - kMagic))) <= 0.49995f;
      r[i] = __float_as_uint(m);
    }
    store(r, qe + k * step);
    return sure;
  };
  auto put_divided = [&](int k) {
    float x[VPT];
    unpack(load(we + k * step), x);
    uint32_t r[VPT];
#pragma unroll
    for (int i = 0; i < VPT; ++i) r[i] = (uint32_t)quantize_one(x[i], scale[cp * VPT + i]);
    store(r, qe + k * step);
  };
  uint32_t again = 0;  // sweeps to divide: read once more and stored over
#pragma unroll
  for (int k = 0; k < SW; ++k) {
    // (keeps the packed words, not their unpacked floats, alive across the barriers)
    asm volatile("" : "+v"(v[k].x), "+v"(v[k].y), "+v"(v[k].z), "+v"(v[k].w));
    if (on && k * RPS + row0 < Kd && !put(v[k], k)) again |= 1u << k;
  }
  for (int k = SW; on && k * RPS + row0 < Kd; ++k)
    if (!put(load(we + k * step), k)) put_divided(k);
  while (again) {
    const int k = __builtin_ctz(again);
    again &= again - 1;
    put_divided(k);
  }
}

// Any width and alignment: one thread per (e, n).
template <typename W>
__global__ __launch_bounds__(256) void k_quantize_pc(int64_t E, int64_t Kd, int64_t N, const W* __restrict__ w,
                                                     int8_t* __restrict__ q, float* __restrict__ s) {
  const int64_t n = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t e = blockIdx.y;
  if (n >= N) return;
  const W* we = w + e * Kd * N + n;
  float amax = 0.0f;
  for (int64_t k = 0; k < Kd; ++k) amax = fmaxf(amax, fabsf(Act<W>::load(we, k * N)));
  const float sc = channel_scale(amax);
  s[e * N + n] = sc;
  int8_t* qe = q + e * Kd * N + n;
  for (int64_t k = 0; k < Kd; ++k) qe[k * N] = (int8_t)quantize_one(Act<W>::load(we, k * N), sc);
}

}  // namespace kmoe

namespace kmoe_host {

using namespace kmoe;

hipError_t launch_prepack(const kmoe_desc& d, const kmoe_weight& gate, const kmoe_weight& up, const kmoe_weight& down,
                          const kmoe_packed_experts& p, hipStream_t st) {
  const int E = (int)d.num_experts, D = (int)d.hidden, I = (int)d.intermediate;
  auto pack = [&](int Kd, int N, int W, const kmoe_weight& w0, const kmoe_weight& w1, void* dst) {
    hipLaunchKernelGGL(k_pack, dim3((unsigned)((int64_t)((N / 4 + 63) / 64) * ((Kd / 16 + 3) / 4) * E * W)), dim3(256), 0,
                       st, Kd, N, W,
                       reinterpret_cast<const int8_t*>(w0.values), reinterpret_cast<const int8_t*>(w1.values),
                       reinterpret_cast<int8_t*>(dst));
    return hipGetLastError();
  };
  hipError_t err = pack(D, I, 2, gate, up, p.w13);
  if (err != hipSuccess) return err;
  err = pack(I, D, 1, down, down, p.w2);
  if (err != hipSuccess) return err;
  const int64_t ns = (int64_t)E * I * 2 + (int64_t)E * D;
  auto bf = [](const kmoe_weight& w) { return w.scale_dtype == KMOE_DTYPE_BF16 ? 1 : 0; };
  auto pc = [](const kmoe_weight& w) { return w.scale_kind == KMOE_SCALE_CHANNEL ? 1 : 0; };
  hipLaunchKernelGGL(k_pack_scales, dim3((unsigned)((ns + 255) / 256)), dim3(256), 0, st, E, D, I, gate.scale,
                     bf(gate), pc(gate), up.scale, bf(up), pc(up), down.scale, bf(down), pc(down),
                     reinterpret_cast<float*>(p.s13), reinterpret_cast<float*>(p.s2));
  return hipGetLastError();
}

hipError_t launch_to_compute_dtype(const kmoe_weight& w, int64_t outer, int64_t channels, int64_t rows_per_block,
                                   kmoe_dtype out_dtype, void* out, hipStream_t st) {
  const int64_t n = outer * channels;
  const unsigned blocks = (unsigned)((n + 255) / 256);
  const int wt = w.dtype == KMOE_DTYPE_F32 ? 0 : (w.dtype == KMOE_DTYPE_BF16 ? 1 : 2);
  const int s_bf16 = (wt == 2 && w.scale_dtype == KMOE_DTYPE_BF16) ? 1 : 0;
  const int pc = (wt == 2 && w.scale_kind == KMOE_SCALE_CHANNEL) ? 1 : 0;
  if (out_dtype == KMOE_DTYPE_BF16)
    hipLaunchKernelGGL((k_to_compute<uint16_t>), dim3(blocks), dim3(256), 0, st, outer, channels, rows_per_block,
                       w.values, wt, w.scale, s_bf16, pc, reinterpret_cast<uint16_t*>(out));
  else
    hipLaunchKernelGGL((k_to_compute<float>), dim3(blocks), dim3(256), 0, st, outer, channels, rows_per_block,
                       w.values, wt, w.scale, s_bf16, pc, reinterpret_cast<float*>(out));
  return hipGetLastError();
}

// The strip quantiser takes rows and outputs it can move 16 (4 or 8) bytes at a time.
template <typename W>
static bool quantize_strip_fits(int64_t E, int64_t Kd, int64_t N, const void* w, const void* q) {
  const int64_t vpt = 16 / sizeof(W);
  return N % vpt == 0 && reinterpret_cast<uintptr_t>(w) % 16 == 0 && reinterpret_cast<uintptr_t>(q) % vpt == 0 &&
         E * ((N + 127) / 128) < ((int64_t)1 << 20) && Kd < ((int64_t)1 << 31) / (int64_t)sizeof(W) / N;
}

template <typename W>
static void quantize_launch(int64_t E, int64_t Kd, int64_t N, const void* w, int8_t* q, float* s, hipStream_t st) {
  const W* wp = reinterpret_cast<const W*>(w);
  if (!quantize_strip_fits<W>(E, Kd, N, w, q)) {
    hipLaunchKernelGGL((k_quantize_pc<W>), dim3((unsigned)((N + 255) / 256), (unsigned)E), dim3(256), 0, st, E, Kd, N,
                       wp, q, s);
    return;
  }
  const int64_t pairs = E * ((N + 127) / 128);
  const dim3 grid((unsigned)((pairs + 7) / 8 * 16));
  // eight sweeps in registers where they hold every row (two blocks per CU), else sixteen
  const int rows = 1024 * (int)(16 / sizeof(W)) / 64;
  if (Kd <= 8 * rows)
    hipLaunchKernelGGL((k_quantize_strip<W, 8>), grid, dim3(1024), 0, st, (int)E, (int)Kd, (int)N, wp, q, s);
  else
    hipLaunchKernelGGL((k_quantize_strip<W, 16>), grid, dim3(1024), 0, st, (int)E, (int)Kd, (int)N, wp, q, s);
}

hipError_t launch_quantize_per_channel(int64_t E, int64_t Kd, int64_t N, const void* w, kmoe_dtype w_dtype, int8_t* q,
                                       float* s, hipStream_t st) {
  if (w_dtype == KMOE_DTYPE_BF16)
    quantize_launch<uint16_t>(E, Kd, N, w, q, s, st);
  else
    quantize_launch<float>(E, Kd, N, w, q, s, st);
  return hipGetLastError();
}

}  // namespace kmoe_host
