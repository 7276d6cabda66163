// SwiGLU experts on plain bf16 weights in the reference layout ([E, D, I] gate
// and up, [E, I, D] down), bf16 activations, on bf16 MFMA.
//
// Reference: as expert.hip, for an unquantised layer (weights are jax arrays of
// x.dtype): _moe_gather_einsum kappa/qwen3/ffn_moe.py:74-104 and
// _moe_fixed_capacity :107-158 on the kChainAct chain, _moe_ragged :174-216 on
// kChainF32, whose f32 h is two bf16 planes per row (hi, lo), both multiplied
// by the weights.
//
// A weight matrix is [k][n] row-major, and an MFMA operand is 8 consecutive k
// of one column per lane. Nothing is relaid out: lane (c = lane % 16, q = lane /
// 16) takes W consecutive columns W c .. W c + W - 1 of the rows k = 8 q .. 8 q + 7
// (16 lanes cover 16 W consecutive columns: 64 or 128 bytes of a row), and one
// v_perm_b32 per dword pairs two rows of one column, which gives the operands
// of W tiles: tile j's column m is column W m + j. The weights are the MFMA's
// first operand, so a lane ends with its token's columns W (4 q + i) + j.
//
// The layout-native kernels (one fmaf chain per output, every assignment
// reading its expert's weights again) took, for gate/up + down of the 30B-A3B
// layer, 1045 + 314 us at T = 4 (gather) and 21.4 + 10.9 ms at T = 1024 (ragged);
// these take 40 + 18 and 196 + 110 us.
#include "common.h"
#include "expert_dev.h"
#include "launch.h"

namespace kmoe {

namespace {

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// eight rows of four columns (8 bytes per row) -> the operands of the four columns
__device__ __forceinline__ void transpose4(const u32x2* r, bf16x8* c) {
  uint32_t lo[8], hi[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    lo[i] = r[i].x;
    hi[i] = r[i].y;
  }
  transpose2(lo, c[0], c[1]);
  transpose2(hi, c[2], c[3]);
}

// 8 bytes at a wave-uniform base and a lane's 32-bit byte offset (no 64-bit
// address per lane and load), nontemporal
__device__ __forceinline__ u32x2 load_stream8(const char* base, uint32_t off) {
  return __builtin_nontemporal_load(reinterpret_cast<const u32x2*>(base + off));
}

constexpr int kW16Waves = 8;  // waves of a decode block, splitting the reduction

// One output of the f32 chain's down product as the layout-native kernel sums it: h =
// hi + lo first, then one chain. The planes meet a weight separately, so an infinite
// weight gives inf - inf (or 0 * inf) where h * inf is infinite: outputs that come out
// NaN are summed again this way. h: a row's hi plane (lo I further), w: the column.
__device__ __forceinline__ float w16_chain(const uint16_t* __restrict__ h, int I, const uint16_t* __restrict__ w,
                                           int D) {
  float acc = 0.0f;
  for (int i = 0; i < I; ++i)
    acc = __builtin_fmaf(bf16_bits_to_f32(h[i]) + bf16_bits_to_f32(h[I + i]), bf16_bits_to_f32(w[(size_t)i * D]), acc);
  return acc;
}

}  // namespace

// ---------------------------------------------------------------------------
// Decode: one block per (64 columns, active expert, 16-row group). Eight waves
// split the reduction (32-deep steps [KC w / 8, KC (w + 1) / 8)); a wave streams
// its rows of the 64 columns straight into registers, NB steps in flight, and
// the partial sums meet in LDS in wave order, so a row's value does not depend
// on the other rows of the batch. Bound by the weight stream: T = 64 1.2 GB in
// ~205 us for both kernels (5.9 TB/s), T = 4 (29 of 128 experts) 182 MB in 38 us.
// The row bases are wave-uniform with one 32-bit lane offset: with a 64-bit
// address per lane and load the kernel needed 162 registers instead of 130 and
// T = 64 took 251 us per layer (now 228). 128 registers keep two blocks on a CU.
// Four waves of the same loads: T = 1 / 64 43 / 226 us; batches of four steps
// in four waves (202 registers): 43 / 226.
// ---------------------------------------------------------------------------
template <int CH>
__global__ __launch_bounds__(64 * kW16Waves, 4) void k_gateup_w16(int D, int I, int E, const uint16_t* __restrict__ x,
                                                               const int32_t* __restrict__ offsets,
                                                               const int32_t* __restrict__ active,
                                                               const int32_t* __restrict__ sorted_token,
                                                               const uint16_t* __restrict__ wg,
                                                               const uint16_t* __restrict__ wu,
                                                               uint16_t* __restrict__ h_sorted, int cap) {
  constexpr int NB = 2;
  __shared__ floatx4 red[kW16Waves][2][4][64];  // [wave][gate, up][tile][lane]
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, q = lane >> 4;
  const int n_active = active[E];
  const int e = active[blockIdx.y < (unsigned)E ? blockIdx.y : 0];
  if ((int)blockIdx.y >= n_active) return;
  const int r0 = offsets[e] + 16 * (int)blockIdx.z;
  const int nrows = min(offsets[e + 1] - offsets[e], cap) - 16 * (int)blockIdx.z;
  if (nrows <= 0) return;
  const int col0 = blockIdx.x * 64;
  const char* const bg = reinterpret_cast<const char*>(wg + (size_t)e * D * I + col0);
  const char* const bu = reinterpret_cast<const char*>(wu + (size_t)e * D * I + col0);
  const uint32_t pitch = 2u * (uint32_t)I, loff = 8u * q * pitch + 8u * c;
  const int KC = D >> 5;
  const int c0 = (KC * wv) / kW16Waves, c1 = (KC * (wv + 1)) / kW16Waves;
  const int tok = sorted_token[r0 + min(c, nrows - 1)];
  const uint16_t* xr = x + (size_t)tok * D + 8 * q;
  floatx4 ag[4], au[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    ag[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    au[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  }
  for (int cb = c0; cb < c1; cb += NB) {
    u32x2 g[NB][8], u[NB][8];
    uint4 a[NB];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if (cb + i < c1) {
#pragma unroll
        for (int r = 0; r < 8; ++r) {
          const size_t o = (size_t)((cb + i) * 32 + r) * pitch;
          g[i][r] = load_stream8(bg + o, loff);
          u[i][r] = load_stream8(bu + o, loff);
        }
        // rows past the group repeat its last row and are not stored
        a[i] = *reinterpret_cast<const uint4*>(xr + (cb + i) * 32);
      }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if (cb + i < c1) {
        bf16x8 fg[4], fu[4];
        transpose4(g[i], fg);
        transpose4(u[i], fu);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          ag[j] = mfma16(fg[j], as_bf16x8(a[i]), ag[j]);
          au[j] = mfma16(fu[j], as_bf16x8(a[i]), au[j]);
        }
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    red[wv][0][j][lane] = ag[j];
    red[wv][1][j][lane] = au[j];
  }
  __syncthreads();
  if (wv >= 4 || c >= nrows) return;
  // wave j finishes tile j: row c, columns 4 (4 q + i) + j
  floatx4 g = red[0][0][wv][lane], u = red[0][1][wv][lane];
#pragma unroll
  for (int w = 1; w < kW16Waves; ++w) {
    g += red[w][0][wv][lane];
    u += red[w][1][wv][lane];
  }
  uint16_t* hr = h_sorted + (size_t)(r0 + c) * (CH == kChainF32 ? 2 * I : I) + col0 + 16 * q + wv;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (CH == kChainAct)
      hr[4 * i] = f32_to_bf16_bits(swiglu<true>(round_bf16(g[i]), round_bf16(u[i])));
    else
      split_bf16(swiglu<false>(g[i], u[i]), hr[4 * i], hr[I + 4 * i]);
  }
}

template <int CH>
__global__ __launch_bounds__(64 * kW16Waves, 4) void k_down_w16(int D, int I, int E, const uint16_t* __restrict__ h_sorted,
                                                             const int32_t* __restrict__ offsets,
                                                             const int32_t* __restrict__ active,
                                                             const uint16_t* __restrict__ wd,
                                                             uint16_t* __restrict__ y_sorted, int cap) {
  constexpr int NB = 3;
  constexpr int PL = CH == kChainF32 ? 2 : 1;  // planes of h
  __shared__ floatx4 red[kW16Waves][4][64];
  const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int c = lane & 15, q = lane >> 4;
  const int n_active = active[E];
  const int e = active[blockIdx.y < (unsigned)E ? blockIdx.y : 0];
  if ((int)blockIdx.y >= n_active) return;
  const int r0 = offsets[e] + 16 * (int)blockIdx.z;
  const int nrows = min(offsets[e + 1] - offsets[e], cap) - 16 * (int)blockIdx.z;
  if (nrows <= 0) return;
  const int col0 = blockIdx.x * 64;
  const char* const bd = reinterpret_cast<const char*>(wd + (size_t)e * I * D + col0);
  const uint32_t pitch = 2u * (uint32_t)D, loff = 8u * q * pitch + 8u * c;
  const int KC = I >> 5;
  const int c0 = (KC * wv) / kW16Waves, c1 = (KC * (wv + 1)) / kW16Waves;
  const uint16_t* hr = h_sorted + (size_t)(r0 + min(c, nrows - 1)) * PL * I + 8 * q;
  floatx4 acc[4];
#pragma unroll
  for (int j = 0; j < 4; ++j) acc[j] = floatx4{0.f, 0.f, 0.f, 0.f};
  for (int cb = c0; cb < c1; cb += NB) {
    u32x2 w[NB][8];
    uint4 a[NB][PL];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if (cb + i < c1) {
#pragma unroll
        for (int r = 0; r < 8; ++r) w[i][r] = load_stream8(bd + (size_t)((cb + i) * 32 + r) * pitch, loff);
#pragma unroll
        for (int p = 0; p < PL; ++p) a[i][p] = *reinterpret_cast<const uint4*>(hr + p * I + (cb + i) * 32);
      }
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      if (cb + i < c1) {
        bf16x8 f[4];
        transpose4(w[i], f);
#pragma unroll
        for (int p = 0; p < PL; ++p)
#pragma unroll
          for (int j = 0; j < 4; ++j) acc[j] = mfma16(f[j], as_bf16x8(a[i][p]), acc[j]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) red[wv][j][lane] = acc[j];
  __syncthreads();
  if (wv >= 4 || c >= nrows) return;
  floatx4 v = red[0][wv][lane];
#pragma unroll
  for (int w = 1; w < kW16Waves; ++w) v += red[w][wv][lane];
  uint16_t* yr = y_sorted + (size_t)(r0 + c) * D + col0 + 16 * q + wv;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (CH == kChainF32 && v[i] != v[i])
      v[i] = w16_chain(h_sorted + (size_t)(r0 + c) * 2 * I, I, wd + (size_t)e * I * D + col0 + 16 * q + wv + 4 * i, D);
    yr[4 * i] = f32_to_bf16_bits(v[i]);
  }
}

// ---------------------------------------------------------------------------
// Prefill: grouped GEMM over (expert, 64-row tile, column tile) work items, the
// items of one expert on one XCD as in k_gemm (expert.hip). A block of four
// waves computes up to 64 rows x 256 weight columns (gate/up: 128 gate and the
// same 128 up columns); wave w owns 64 of them (gate/up: 32 + 32) for all rows.
//
// Both operands reach LDS by direct global->LDS loads in 64-deep chunks, two
// stages each: A (8 KB) as [row][8 x 16 B], pieces swizzled by row; B (32 KB)
// as 8 KB per wave in the order its lanes read it: the rows k = 16 q + s of the
// four lane groups q side by side, so that a fragment row is one contiguous
// 256- or 512-byte LDS read without bank conflicts. 80 KB: two blocks per CU,
// 128 KB of weights in flight or in use on each, which keeps the HBM stream fed
// at a few rows per expert; with 64 rows per tile the loop is bound by LDS
// (A 32 KB + B 32 KB read and 40 KB written per chunk against 32 MFMAs per
// wave).
//
// The k order inside a chunk is k_gemm's: lane group q supplies k = 16 q + 8 st
// + 0..7 in step st, for both operands. Columns past the matrix (its width is a
// multiple of 64, not of the tile) repeat the last ones and are not stored.
// ---------------------------------------------------------------------------
namespace {

constexpr int kW16Rows = 64;
constexpr int kW16A = kW16Rows * 128;  // A stage
constexpr int kW16B = 4 * 8192;        // B stage

struct W16Loads {
  uint32_t avoff[2];     // byte offsets (per lane) of this wave's A loads in src
  const char* b0;        // gate/up: gate columns at chunk 0; down: the wave's columns
  const char* b1;        // gate/up: up columns at chunk 0
  uint32_t bvoff;        // byte offset (per lane) of the wave's B loads
  uint32_t pitch;        // bytes of a weight row
};

template <bool GATEUP, int MT, int CH, int PL>
__device__ __forceinline__ void w16_tile(uint8_t* smem, const W16Loads& gl, int KCW, int wv, int rows, int row0,
                                         int col, bool col_on, const uint16_t* __restrict__ src,
                                         uint16_t* __restrict__ dst, int Ndim) {
  const int lane = threadIdx.x & 63;
  const uint32_t lds0 = lds_addr(smem);
  const uint8_t* const bring = smem + 2 * kW16A + wv * 8192;
  const int KC = PL * KCW;  // A chunks: chunk c is plane c % PL of weight chunk c / PL
  floatx4 acc[MT][4];
#pragma unroll
  for (int mi = 0; mi < MT; ++mi)
#pragma unroll
    for (int g = 0; g < 4; ++g) acc[mi][g] = floatx4{0.f, 0.f, 0.f, 0.f};

  auto issue_a = [&](int c) {
    const uint32_t st = lds0 + (uint32_t)((c & 1) * kW16A + wv * 2048);
    const uint16_t* abase = src + (PL == 2 ? (c & 1) * (KCW * 64) + (c >> 1) * 64 : c * 64);
#pragma unroll
    for (int j = 0; j < 2; ++j) dma16(gl.avoff[j], abase, st + j * 1024);
  };
  auto issue_b = [&](int b) {
    const uint32_t st = lds0 + (uint32_t)(2 * kW16A + (b & 1) * kW16B + wv * 8192);
    const size_t o = (size_t)b * 64 * gl.pitch;
    if (GATEUP) {
      // 16 slots of 64 bytes per load: rows 4 t .. 4 t + 3 of each lane group's 16
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        dma16(gl.bvoff, gl.b0 + o + (size_t)(4 * t) * gl.pitch, st + t * 1024);
        dma16(gl.bvoff, gl.b1 + o + (size_t)(4 * t) * gl.pitch, st + 4096 + t * 1024);
      }
    } else {
      // 8 slots of 128 bytes per load: rows 2 t, 2 t + 1 of each lane group's 16
#pragma unroll
      for (int t = 0; t < 8; ++t) dma16(gl.bvoff, gl.b0 + o + (size_t)(2 * t) * gl.pitch, st + t * 1024);
    }
  };

  // PL = 1: iteration c issues A(c + 1) and B(c + 1) into the stages chunk
  // c - 1 left and waits for both at its end. PL = 2: B(c / 2 + 1) is issued in
  // the even iteration and waited for in the odd one.
  issue_b(0);
  issue_a(0);
  vm_barrier<0>();
  bf16x8 f[2][4];
  for (int c = 0; c < KC; ++c) {
    const int b = PL == 2 ? c >> 1 : c;
    const bool b_next = (PL == 1 || (c & 1) == 0) && b + 1 < KCW;
    if (c + 1 < KC) issue_a(c + 1);
    if (b_next) issue_b(b + 1);
    if (PL == 1 || (c & 1) == 0) {
      const uint8_t* bp = bring + (b & 1) * kW16B;
#pragma unroll
      for (int st = 0; st < 2; ++st) {
        if (GATEUP) {
          uint32_t g[8], u[8];
#pragma unroll
          for (int r = 0; r < 8; ++r) {
            g[r] = *reinterpret_cast<const uint32_t*>(bp + (st * 8 + r) * 256 + 4 * lane);
            u[r] = *reinterpret_cast<const uint32_t*>(bp + 4096 + (st * 8 + r) * 256 + 4 * lane);
          }
          transpose2(g, f[st][0], f[st][1]);
          transpose2(u, f[st][2], f[st][3]);
        } else {
          u32x2 w[8];
#pragma unroll
          for (int r = 0; r < 8; ++r) w[r] = *reinterpret_cast<const u32x2*>(bp + (st * 8 + r) * 512 + 8 * lane);
          transpose4(w, f[st]);
        }
      }
    }
    const uint16_t* As = reinterpret_cast<const uint16_t*>(smem + (c & 1) * kW16A);
#pragma unroll
    for (int st = 0; st < 2; ++st) {
      const int p = 2 * (lane >> 4) + st;
#pragma unroll
      for (int mi = 0; mi < MT; ++mi) {
        const bf16x8 a = *reinterpret_cast<const bf16x8*>(As + a_at<1>(mi * 16 + (lane & 15), p));
#pragma unroll
        for (int g = 0; g < 4; ++g) acc[mi][g] = mfma16(f[st][g], a, acc[mi][g]);
      }
    }
    if (c + 1 < KC) {
      if (PL == 2 && b_next)
        vm_barrier<8>();  // the next weight chunk stays in flight
      else
        vm_barrier<0>();
    }
  }

  bool nan = false;  // of this lane's outputs (the f32 chain's down product)

  // a lane holds row mi * 16 + lane % 16 and, for i, g: gate/up columns 2 (4 q + i)
  // + g (up in tiles 2, 3), down columns 4 (4 q + i) + g, of the wave's columns
  if (!col_on) return;
#pragma unroll
  for (int mi = 0; mi < MT; ++mi) {
    const int row = mi * 16 + (lane & 15);
    if (row >= rows) continue;
    if (GATEUP) {
      uint16_t* drow = dst + (size_t)(row0 + row) * (CH == kChainF32 ? 2 * Ndim : Ndim) + col + 8 * (lane >> 4);
      float hv[8], lv[8];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int g = 0; g < 2; ++g) {
          const float gv = acc[mi][g][i], uv = acc[mi][g + 2][i];
          if (CH == kChainAct) {
            hv[2 * i + g] = swiglu<true>(round_bf16(gv), round_bf16(uv));
          } else {
            const float h = swiglu<false>(gv, uv);
            hv[2 * i + g] = round_bf16(h);
            lv[2 * i + g] = __fsub_rn(h, hv[2 * i + g]);
          }
        }
      *reinterpret_cast<uint4*>(drow) = uint4{pack_bf16x2(hv[0], hv[1]), pack_bf16x2(hv[2], hv[3]),
                                              pack_bf16x2(hv[4], hv[5]), pack_bf16x2(hv[6], hv[7])};
      if (CH == kChainF32)
        *reinterpret_cast<uint4*>(drow + Ndim) = uint4{pack_bf16x2(lv[0], lv[1]), pack_bf16x2(lv[2], lv[3]),
                                                       pack_bf16x2(lv[4], lv[5]), pack_bf16x2(lv[6], lv[7])};
    } else {
      uint16_t* drow = dst + (size_t)(row0 + row) * Ndim + col + 16 * (lane >> 4);
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        uint32_t o[4];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          o[2 * i] = pack_bf16x2(acc[mi][0][2 * hf + i], acc[mi][1][2 * hf + i]);
          o[2 * i + 1] = pack_bf16x2(acc[mi][2][2 * hf + i], acc[mi][3][2 * hf + i]);
        }
        *reinterpret_cast<uint4*>(drow + 8 * hf) = uint4{o[0], o[1], o[2], o[3]};
      }
      if (CH == kChainF32) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int i = 0; i < 4; ++i) nan = nan || acc[mi][g][i] != acc[mi][g][i];
      }
    }
  }
  if (!GATEUP && CH == kChainF32 && nan) {
    // summed again in the chain's order (w16_chain), from what was stored
    for (int row = lane & 15; row < rows; row += 16) {
      uint16_t* y = dst + (size_t)(row0 + row) * Ndim + col + 16 * (lane >> 4);
      for (int j = 0; j < 16; ++j)
        if ((y[j] & 0x7fffu) > 0x7f80u)
          y[j] = f32_to_bf16_bits(w16_chain(src + (size_t)(row0 + row) * PL * KCW * 64, KCW * 64,
                                            reinterpret_cast<const uint16_t*>(gl.b0) + 16 * (lane >> 4) + j, Ndim));
    }
  }
}

}  // namespace

// w0: gate (gate/up) or down; w1: up. src must span fewer than 2^32 bytes, and
// so must one expert's matrix.
template <bool GATEUP, int CH>
__global__ __launch_bounds__(256, 2) void k_gemm_w16(int D, int I, int E, const uint16_t* __restrict__ src,
                                                      const int32_t* __restrict__ offsets,
                                                      const int32_t* __restrict__ sorted_token,
                                                      const uint16_t* __restrict__ w0, const uint16_t* __restrict__ w1,
                                                      uint16_t* __restrict__ dst, int cap) {
  __shared__ __attribute__((aligned(1024))) uint8_t smem[2 * kW16A + 2 * kW16B];
  // set-up scratch inside the ring (no loads are in flight yet)
  int* const mtp = reinterpret_cast<int*>(smem);
  int* const offs = mtp + kMaxExperts + 1;
  int* const wsum = offs + kMaxExperts + 1;
  int* const tok = wsum + 4;
  const int tid = threadIdx.x, lane = tid & 63;
  const int Ndim = GATEUP ? I : D, Kdim = GATEUP ? D : I;
  const int NT = GATEUP ? (I + 127) / 128 : (D + 255) / 256;
  tile_prefix<kW16Rows>(offsets, E, cap, mtp, wsum, offs);
  const int ntiles = mtp[E] * NT;
  const int per = (ntiles + 7) >> 3;
  const int qb = blockIdx.x >> 3;
  if (qb >= per) return;
  const int L = (blockIdx.x & 7) * per + qb;
  if (L >= ntiles) return;
  // L -> (expert, column tile, row tile), row tile fastest; an expert's rows
  // split evenly over its row tiles
  const int e = __builtin_amdgcn_readfirstlane(tile_expert(mtp, E, L / NT));
  const int nmt_e = mtp[e + 1] - mtp[e];
  const int rem = L - mtp[e] * NT;
  const int nt = __builtin_amdgcn_readfirstlane(rem / nmt_e);
  const int mt = rem - nt * nmt_e;
  const int ne = min(offs[e + 1] - offs[e], cap);
  const int tr = (((ne + nmt_e - 1) / nmt_e) + 15) & ~15;
  const int row0 = __builtin_amdgcn_readfirstlane(offs[e] + mt * tr);
  const int rows = __builtin_amdgcn_readfirstlane(min(tr, ne - mt * tr));
  if (tid < kW16Rows) tok[tid] = (tid < rows) ? (GATEUP ? sorted_token[row0 + tid] : row0 + tid) : -1;
  __syncthreads();
  const int wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  constexpr int PL = !GATEUP && CH == kChainF32 ? 2 : 1;
  const int adim = PL * Kdim;
  W16Loads gl;
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    const int r = 8 * (wv * 2 + j) + (lane >> 3);
    const int t = tok[r] >= 0 ? tok[r] : tok[0];
    gl.avoff[j] = ((uint32_t)t * (uint32_t)adim + (uint32_t)(a_piece_at<1>(r, lane & 7) << 3)) * 2u;
  }
  const int width = GATEUP ? 32 : 64;
  const int col_w = nt * (4 * width) + wv * width;
  const bool col_on = col_w < Ndim;
  const int col = min(col_w, Ndim - width);
  gl.pitch = (uint32_t)Ndim * 2u;
  const size_t at = ((size_t)e * Kdim * Ndim + col) * 2;
  gl.b0 = reinterpret_cast<const char*>(w0) + at;
  if (GATEUP) {
    gl.b1 = reinterpret_cast<const char*>(w1) + at;
    gl.bvoff = (uint32_t)(16 * ((lane >> 2) & 3) + (lane >> 4)) * gl.pitch + 16u * (lane & 3);
  } else {
    gl.b1 = gl.b0;
    gl.bvoff = (uint32_t)(16 * ((lane >> 3) & 3) + (lane >> 5)) * gl.pitch + 16u * (lane & 7);
  }
  __syncthreads();  // no wave may start loading into the ring while another still reads tok
  const int KCW = Kdim >> 6;
  switch ((rows + 15) >> 4) {
    case 4:
      w16_tile<GATEUP, 4, CH, PL>(smem, gl, KCW, wv, rows, row0, col, col_on, src, dst, Ndim);
      break;
    case 3:
      w16_tile<GATEUP, 3, CH, PL>(smem, gl, KCW, wv, rows, row0, col, col_on, src, dst, Ndim);
      break;
    case 2:
      w16_tile<GATEUP, 2, CH, PL>(smem, gl, KCW, wv, rows, row0, col, col_on, src, dst, Ndim);
      break;
    default:
      w16_tile<GATEUP, 1, CH, PL>(smem, gl, KCW, wv, rows, row0, col, col_on, src, dst, Ndim);
      break;
  }
}

}  // namespace kmoe

namespace kmoe_host {

using namespace kmoe;

namespace {

template <int CH>
hipError_t w16_stages(const kmoe_desc& d, int family, int stages, const uint16_t* x, const int32_t* offsets,
                      const int32_t* active, const int32_t* sorted_token, const uint16_t* wg, const uint16_t* wu,
                      const uint16_t* wd, uint16_t* hb, uint16_t* yb, int cap, hipStream_t st) {
  const int T = (int)d.tokens, D = (int)d.hidden, E = (int)d.num_experts, K = (int)d.top_k,
            I = (int)d.intermediate;
  const int M = T * K;
  const int slots = M < E ? M : E;
  // the GEMV form up to 64 tokens, as for int8 experts: whole 30B-A3B layers, GEMV
  // against GEMM, T = 1 / 4 / 16 / 64 41 / 76 / 157 / 228 against 75 / 94 / 187 /
  // 255 us. Above 64 tokens it still leads on that shape (T = 65 / 100 234 / 247
  // against 259 / 262 us) and trails on wider or fewer experts (235B-A22B T = 100
  // 938 against 903, 32 experts 116 against 108) and from 150 tokens on (277
  // against 264; T = 220 346 against 267)
  const bool gemv = family != kFamilyGemm;
  const int upper_mt = (M + kW16Rows - 1) / kW16Rows + slots;
  auto grid_for = [&](int NT) { return dim3(((upper_mt * NT + 7) / 8) * 8); };
  if (stages & kStageGateUp) {
    if (gemv)
      hipLaunchKernelGGL((k_gateup_w16<CH>), dim3(I / 64, slots, (T + 15) / 16), dim3(64 * kW16Waves), 0, st, D, I, E,
                         x, offsets, active, sorted_token, wg, wu, hb, cap);
    else
      hipLaunchKernelGGL((k_gemm_w16<true, CH>), grid_for((I + 127) / 128), dim3(256), 0, st, D, I, E, x, offsets,
                         sorted_token, wg, wu, hb, cap);
    hipError_t err = hipGetLastError();
    if (err != hipSuccess) return err;
  }
  if (stages & kStageDown) {
    if (gemv)
      hipLaunchKernelGGL((k_down_w16<CH>), dim3(D / 64, slots, (T + 15) / 16), dim3(64 * kW16Waves), 0, st, D, I, E, hb,
                         offsets, active, wd, yb, cap);
    else
      hipLaunchKernelGGL((k_gemm_w16<false, CH>), grid_for((D + 255) / 256), dim3(256), 0, st, D, I, E, hb, offsets,
                         sorted_token, wd, wd, yb, cap);
    return hipGetLastError();
  }
  return hipSuccess;
}

}  // namespace

bool expert_w16_fits(const kmoe_desc& d, int stages, const void* x, const kmoe_weight* gate, const kmoe_weight* up,
                     const kmoe_weight* down, const void* h_sorted, const void* y_sorted) {
  if (d.act_dtype != KMOE_DTYPE_BF16 || d.hidden % 64 || d.intermediate % 64) return false;
  const uint64_t M = (uint64_t)d.tokens * d.top_k, lim = 1ull << 32;
  const uint64_t hrow = chain_of(d) == kChainF32 ? 2ull * d.intermediate : (uint64_t)d.intermediate;
  if ((uint64_t)d.tokens * d.hidden * 2 >= lim || M * hrow * 2 >= lim || (uint64_t)d.hidden * d.intermediate * 2 >= lim)
    return false;
  auto ok = [](const kmoe_weight* w) { return w && w->dtype == KMOE_DTYPE_BF16 && aligned16(w->values); };
  if (!aligned16(h_sorted)) return false;
  if ((stages & kStageGateUp) && !(ok(gate) && ok(up) && aligned16(x))) return false;
  if ((stages & kStageDown) && !(ok(down) && aligned16(y_sorted))) return false;
  return true;
}

hipError_t launch_expert_w16(const kmoe_desc& d, int chain, int family, int stages, const void* x,
                             const int32_t* offsets, const int32_t* active, const int32_t* sorted_token,
                             const kmoe_weight* gate, const kmoe_weight* up, const kmoe_weight* down, void* h_sorted,
                             void* y_sorted, int cap, hipStream_t st) {
  auto v = [](const kmoe_weight* w) { return w ? reinterpret_cast<const uint16_t*>(w->values) : nullptr; };
  const uint16_t* xb = reinterpret_cast<const uint16_t*>(x);
  uint16_t* hb = reinterpret_cast<uint16_t*>(h_sorted);
  uint16_t* yb = reinterpret_cast<uint16_t*>(y_sorted);
  if (chain == kChainF32)
    return w16_stages<kChainF32>(d, family, stages, xb, offsets, active, sorted_token, v(gate), v(up), v(down), hb, yb,
                                 cap, st);
  return w16_stages<kChainAct>(d, family, stages, xb, offsets, active, sorted_token, v(gate), v(up), v(down), hb, yb,
                               cap, st);
}

}  // namespace kmoe_host
