// Model-side kernels of one decode step (the C5 counterpart of the reference
// runtime's layer_decode, Z/model_hub/LLM.py:208-251, with the rmsnorm /
// rope / silu pieces of Z/model_hub/qwen.py:493-604):
//
//  * decode_stream_kernel (M <= 4), decode_rows_kernel, decode_wide_kernel and
//    decode_linear_kernel:
//    y[m, n] = sum_k x[m, k] * w[n, k] for the few rows m of a decode batch
//    (M <= 16), bf16 in, fp32 accumulate, bf16 out, with an optional RMSNorm of
//    x on the way in and an optional epilogue (residual add, or silu(gate) * up
//    over the two halves of w).  The weights stream once from HBM.
//  * qk_norm_rope_kernel: per-head RMSNorm of q and k, rotate-half RoPE at
//    one position, and the k / v rows written straight into the cache.
//
// Rounding follows the torch restatement: every bf16 tensor of the
// reference is rounded (RNE) where the reference materialises it.
#include "zkv_common.hpp"

#include <algorithm>

namespace zkv {
namespace {

typedef __bf16 bf16x8v_t __attribute__((ext_vector_type(8)));

constexpr int kLinKBlock = 128;  // four MFMA k-chunks of 32
constexpr int kLinMaxM = 16;     // MFMA B columns

enum LinearEpilogue : int { kEpiNone = 0, kEpiResidual = 1, kEpiSiluMul = 2 };

struct LinearParams {
  const uint16_t* x;  // [M, K] bf16, row stride x_ld
  int64_t x_ld;
  const uint16_t* w;  // [N, K] bf16, contiguous rows
  const uint16_t* norm_w;  // [K] bf16 or null
  float eps;
  const uint16_t* res;  // [M, N] bf16 (residual epilogue), row stride res_ld
  int64_t res_ld;
  void* out;  // [M, N] (or [M, N / 2] for silu * up), row stride out_ld
  int64_t out_ld;
  int M, K, N;
  int out_f32;
};

__device__ __forceinline__ float wave_sum(float v) {
  // butterfly over the 64 lanes (every lane ends with the total)
  v += __shfl_xor(v, 32);
  v += __shfl_xor(v, 16);
  v += __shfl_xor(v, 8);
  v += __shfl_xor(v, 4);
  v += __shfl_xor(v, 2);
  v += __shfl_xor(v, 1);
  return v;
}

__device__ __forceinline__ void store_y(const LinearParams& p, int m, int n, float y) {
  if (p.out_f32)
    reinterpret_cast<float*>(p.out)[m * p.out_ld + n] = y;
  else
    reinterpret_cast<uint16_t*>(p.out)[m * p.out_ld + n] = f32_to_bf16_bits(y);
}

// Stages the M x K input rows into LDS (xs), RMS-normalised:
// bf16(x * rsqrt(mean(x^2) + eps) * w).  red: M floats of scratch.
__device__ __forceinline__ void stage_x(const LinearParams& p, uint16_t* xs, float* red) {
  const int nw = blockDim.x >> 6;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int M = p.M, K = p.K;
  const int kv8 = K >> 3;  // 16-byte chunks per row
  // wave m' reduces rows m = m', m' + nw, ... (fixed order: deterministic)
  for (int m = wave; m < M; m += nw) {
    const u32x4_t* xr = reinterpret_cast<const u32x4_t*>(p.x + m * p.x_ld);
    float ss = 0.0f;
    for (int i = lane; i < kv8; i += 64) {
      const u32x4_t v = xr[i];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float lo = __uint_as_float(v[e] << 16), hi = __uint_as_float(v[e] & 0xFFFF0000u);
        ss = ss + lo * lo;
        ss = ss + hi * hi;
      }
    }
    // mean as the sum times 1/K (torch's mean), then rsqrt(mean + eps)
    ss = wave_sum(ss);
    if (lane == 0) red[m] = rsqrtf(ss * (1.0f / static_cast<float>(K)) + p.eps);
  }
  __syncthreads();
  for (int i = tid; i < M * kv8; i += blockDim.x) {
    const int m = i / kv8, k8 = i - m * kv8;
    u32x4_t v = reinterpret_cast<const u32x4_t*>(p.x + m * p.x_ld)[k8];
    const float r = red[m];
    const u32x4_t wv = reinterpret_cast<const u32x4_t*>(p.norm_w)[k8];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float lo = bf16r((__uint_as_float(v[e] << 16) * r) * __uint_as_float(wv[e] << 16));
      const float hi =
          bf16r((__uint_as_float(v[e] & 0xFFFF0000u) * r) * __uint_as_float(wv[e] & 0xFFFF0000u));
      v[e] = (__float_as_uint(lo) >> 16) | (__float_as_uint(hi) & 0xFFFF0000u);
    }
    reinterpret_cast<u32x4_t*>(xs)[i] = v;
  }
  __syncthreads();
}

// M > 4, few tiles, with a norm: one workgroup per tile of 16 output rows (silu *
// up: 8 gate rows and the 8 matching up rows), NW waves splitting the K blocks.  Dynamic LDS: the M x K
// bf16 input rows, then NW x 64 x 4 fp32 partial tiles.
template <int kEpi>
__global__ __launch_bounds__(1024) void decode_linear_kernel(const LinearParams p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  uint16_t* xs = reinterpret_cast<uint16_t*>(lds);
  const int nw = blockDim.x >> 6;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
  const int c = lane & 15, g = lane >> 4;
  const int M = p.M, K = p.K;
  float* red = reinterpret_cast<float*>(lds + static_cast<size_t>(M) * K * 2);
  stage_x(p, xs, red);

  // ---- weight rows of this tile ----
  const int tile = blockIdx.x;
  int row;  // weight row of A row c (or -1 past N)
  if constexpr (kEpi == kEpiSiluMul) {
    const int half = p.N >> 1, j = tile * 8 + (c & 7);
    row = j < half ? (c < 8 ? j : half + j) : -1;
  } else {
    row = tile * 16 + c < p.N ? tile * 16 + c : -1;
  }
  const uint16_t* wr = p.w + static_cast<int64_t>(row < 0 ? 0 : row) * K;
  const bool col_ok = c < M;
  const uint16_t* xr = xs + (col_ok ? c : 0) * K;

  float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
  const int nkb = K / kLinKBlock;
  for (int kb = wave; kb < nkb; kb += nw) {
    u32x4_t a[4], b[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int k = kb * kLinKBlock + 32 * j + 8 * g;
      a[j] = row >= 0 ? *reinterpret_cast<const u32x4_t*>(wr + k) : u32x4_t{0u, 0u, 0u, 0u};
      b[j] = col_ok ? *reinterpret_cast<const u32x4_t*>(xr + k) : u32x4_t{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int j = 0; j < 4; ++j)
      acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v_t, a[j]),
                                                    __builtin_bit_cast(bf16x8v_t, b[j]), acc, 0, 0, 0);
  }

  // ---- sum the waves' partial tiles in wave order, then the epilogue ----
  reinterpret_cast<float4_t*>(red)[wave * 64 + lane] = acc;
  __syncthreads();
  if (wave != 0) return;
  float4_t s = reinterpret_cast<const float4_t*>(red)[lane];
  for (int w = 1; w < nw; ++w) {
    const float4_t t = reinterpret_cast<const float4_t*>(red)[w * 64 + lane];
    s[0] += t[0], s[1] += t[1], s[2] += t[2], s[3] += t[3];
  }
  // lane (c, g) holds rows 4g + i of the tile for batch row c
  if constexpr (kEpi == kEpiSiluMul) {
    // gate rows sit in g < 2, the matching up rows 32 lanes higher
    float up[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      up[i] = __uint_as_float(__builtin_amdgcn_permlane32_swap(__float_as_uint(s[i]), __float_as_uint(s[i]),
                                                               false, false)[1]);
    if (g >= 2 || !col_ok) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int j = tile * 8 + 4 * g + i;
      if (j >= (p.N >> 1)) continue;
      const float gt = bf16r(s[i]), u = bf16r(up[i]);
      const float act = bf16r(gt / (1.0f + expf(-gt)));
      store_y(p, c, j, bf16r(act * u));
    }
  } else {
    if (!col_ok) return;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int n = tile * 16 + 4 * g + i;
      if (n >= p.N) continue;
      float y = bf16r(s[i]);
      if constexpr (kEpi == kEpiResidual) y = bf16r(bf16_to_f32(p.res[c * p.res_ld + n]) + y);
      store_y(p, c, n, y);
    }
  }
}

// M > 4 without a norm (o, down): decode_linear_kernel's sums with nothing
// staged.  The waves of a workgroup split the K blocks (wave w takes blocks w, w
// + nw, ...), so each element of x is used by one wave: it comes from memory
// (the L2) next to its weights, with no barrier before the first weight load.
// A unit is R <= 16 output rows (silu * up: R <= 8 pairs): lanes of the A rows
// past R repeat row R - 1, which moves no more memory, and a row's sum does not
// depend on the unit it is in.
//
// Bound: HBM, behind launch, first latency and last sums.  Against a workgroup
// per 16 rows that stages x in LDS (cold weights, us at M = 6): 2560 x 4096 (o) 9.1
// -> 7.5, 2560 x 9728 (down) 17.1 -> 13.1 (R = 10: 256 units, not 160), 4096 x 12288
// 24.8 -> 23.2, 1024 x 3072 6.5 -> 5.3; silu, 19456 x 2560, M = 16: 51.5 -> 29.0.
// (151936 x 1024, which only a head without its norm would ask for: 58.8 -> 59.9
// at M = 6, 109 -> 76 at M = 16.)

// The sum over kCnt K blocks of a wave, three blocks of loads in flight.  The
// barriers keep the loads where they are: left to itself the compiler sinks them
// to their uses (down 13.1 -> 14.1 us).
template <int kCnt>
__device__ __forceinline__ float4_t row_blocks(const uint16_t* wr, const uint16_t* xr, int wave, int nw) {
  constexpr int kDepth = kCnt < 3 ? kCnt : 3;  // blocks in flight
  float4_t acc = {0.0f, 0.0f, 0.0f, 0.0f};
  if constexpr (kCnt > 0) {
    u32x4_t a[kDepth][4], b[kDepth][4];
    auto load_block = [&](int i) {
      const int k = (wave + i * nw) * kLinKBlock;
#pragma unroll
      for (int j = 0; j < 4; ++j) a[i % kDepth][j] = *reinterpret_cast<const u32x4_t*>(wr + k + 32 * j);
#pragma unroll
      for (int j = 0; j < 4; ++j) b[i % kDepth][j] = *reinterpret_cast<const u32x4_t*>(xr + k + 32 * j);
    };
#pragma unroll
    for (int i = 0; i < kDepth; ++i) load_block(i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int i = 0; i < kCnt; ++i) {
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8v_t, a[i % kDepth][j]),
                                                      __builtin_bit_cast(bf16x8v_t, b[i % kDepth][j]), acc, 0, 0, 0);
      if (i + kDepth < kCnt) load_block(i + kDepth);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  return acc;
}

template <int kEpi, int kCnt>
__global__ __launch_bounds__(1024) void decode_rows_kernel(const LinearParams p, int R) {
  __shared__ float4_t red[16 * 64];
  const int nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4;
  const int K = p.K, N = p.N;
  const int nkb = K / kLinKBlock;
  const bool col_ok = c < p.M;
  const int n0 = blockIdx.x * R;
  // row r of this unit as a row of w (rows past the unit or N repeat the last; not stored)
  auto weight_row = [&](int r) {
    if constexpr (kEpi == kEpiSiluMul)
      return min(n0 + min(r & 7, R - 1), (N >> 1) - 1) + (r < 8 ? 0 : N >> 1);
    else
      return min(n0 + min(r, R - 1), N - 1);
  };
  const uint16_t* wr = p.w + static_cast<int64_t>(weight_row(c)) * K + 8 * g;
  const uint16_t* xr = p.x + min(c, p.M - 1) * p.x_ld + 8 * g;
  uint16_t res[4];  // lane (c, g) ends with rows 4g + i of x row c
  if constexpr (kEpi == kEpiResidual) {
    if (wave == 0) {
#pragma unroll
      for (int i = 0; i < 4; ++i) res[i] = p.res[min(c, p.M - 1) * p.res_ld + weight_row(4 * g + i)];
    }
  }
  // the wave's blocks are all there but for the last: a wave without it takes a
  // straight line of its own (loading some other line in its place costs the load
  // path as much as a block: 6144 x 2560 13.3 us, so 9.7)
  const bool full = wave + (kCnt - 1) * nw < nkb;  // (uniform)
  float4_t acc;
  if (kCnt == 1 || full) {
    asm volatile("; all blocks");  // (unlike the other branch's, so that the loads stay in theirs)
    acc = row_blocks<kCnt>(wr, xr, wave, nw);
  } else {
    asm volatile("; one fewer");
    acc = row_blocks<kCnt - 1>(wr, xr, wave, nw);
  }

  // ---- sum the waves' partial tiles in wave order, then the epilogue ----
  red[wave * 64 + lane] = acc;
  __syncthreads();
  if (wave != 0) return;
  float4_t s = red[lane];
  for (int w = 1; w < nw; ++w) {
    const float4_t t = red[w * 64 + lane];
    s[0] += t[0], s[1] += t[1], s[2] += t[2], s[3] += t[3];
  }
  if constexpr (kEpi == kEpiSiluMul) {
    // gate rows sit in g < 2, the matching up rows 32 lanes higher
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float up = __uint_as_float(__builtin_amdgcn_permlane32_swap(__float_as_uint(s[i]), __float_as_uint(s[i]),
                                                                        false, false)[1]);
      const int r = 4 * g + i, j = n0 + r;
      if (g >= 2 || !col_ok || r >= R || j >= (N >> 1)) continue;
      const float gt = bf16r(s[i]), u = bf16r(up);
      const float act = bf16r(gt / (1.0f + expf(-gt)));
      store_y(p, c, j, bf16r(act * u));
    }
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int r = 4 * g + i, n = n0 + r;
      if (!col_ok || r >= R || n >= N) continue;
      float y = bf16r(s[i]);
      if constexpr (kEpi == kEpiResidual) y = bf16r(bf16_to_f32(res[i]) + y);
      store_y(p, c, n, y);
    }
  }
}

// Stages the M x K input rows into LDS (row stride ld elements), RMS-normalised:
// bf16(x * rsqrt(mean(x^2) + eps) * w).  Wave w of nw takes rows w, w + nw, ...;
// lane l holds 16-byte chunks l, l + 64, ... of a row, summed in that order.
// load(), called ahead of the kernel's weight loads, requests the first kChunks
// chunks (512 kChunks elements) of kRows rows per wave; what is left of a longer
// row is requested behind the weights and waits for them, twice (decode_wide_kernel
// with kChunks 5 and 8, 6144 x 4096, M = 6: 19.5 -> 17.6 us).  The caller
// synchronises after run().
template <int kRows, int kChunks>
struct NormStage {
  u32x4_t xv[kRows][kChunks], wv[kChunks];

  __device__ __forceinline__ void load_row(const LinearParams& p, int r, int m, int lane) {
    const u32x4_t* xr = reinterpret_cast<const u32x4_t*>(p.x + min(m, p.M - 1) * p.x_ld);
#pragma unroll
    for (int j = 0; j < kChunks; ++j) xv[r][j] = xr[min(lane + 64 * j, (p.K >> 3) - 1)];
  }
  __device__ __forceinline__ void load(const LinearParams& p, int wave, int nw, int lane) {
    const int last = (p.K >> 3) - 1;
#pragma unroll
    for (int r = 0; r < kRows; ++r)
      if (r == 0 || wave + r * nw < p.M) load_row(p, r, wave + r * nw, lane);  // (uniform)
#pragma unroll
    for (int j = 0; j < kChunks; ++j)
      wv[j] = reinterpret_cast<const u32x4_t*>(p.norm_w)[min(lane + 64 * j, last)];
  }

  static __device__ __forceinline__ float sum_sq(const u32x4_t v, float ss) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float lo = __uint_as_float(v[e] << 16), hi = __uint_as_float(v[e] & 0xFFFF0000u);
      ss = ss + lo * lo;
      ss = ss + hi * hi;
    }
    return ss;
  }
  static __device__ __forceinline__ u32x4_t normed(u32x4_t v, float r, const u32x4_t w) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float lo = bf16r((__uint_as_float(v[e] << 16) * r) * __uint_as_float(w[e] << 16));
      const float hi = bf16r((__uint_as_float(v[e] & 0xFFFF0000u) * r) * __uint_as_float(w[e] & 0xFFFF0000u));
      v[e] = (__float_as_uint(lo) >> 16) | (__float_as_uint(hi) & 0xFFFF0000u);
    }
    return v;
  }

  __device__ __forceinline__ void norm_row(const LinearParams& p, uint16_t* xs, int ld, int row, int m, int lane) {
    const int kv8 = p.K >> 3;
    const u32x4_t* xr = reinterpret_cast<const u32x4_t*>(p.x + m * p.x_ld);
    float ss = 0.0f;
#pragma unroll
    for (int j = 0; j < kChunks; ++j)
      if (lane + 64 * j < kv8) ss = sum_sq(xv[row][j], ss);
    for (int i = lane + 64 * kChunks; i < kv8; i += 64) ss = sum_sq(xr[i], ss);
    // mean as the sum times 1/K (torch's mean), then rsqrt(mean + eps)
    const float r = rsqrtf(wave_sum(ss) * (1.0f / static_cast<float>(p.K)) + p.eps);
#pragma unroll
    for (int j = 0; j < kChunks; ++j) {
      const int i = lane + 64 * j;
      if (i < kv8) *reinterpret_cast<u32x4_t*>(xs + m * ld + 8 * i) = normed(xv[row][j], r, wv[j]);
    }
    for (int i = lane + 64 * kChunks; i < kv8; i += 64)
      *reinterpret_cast<u32x4_t*>(xs + m * ld + 8 * i) =
          normed(xr[i], r, reinterpret_cast<const u32x4_t*>(p.norm_w)[i]);
  }

  __device__ __forceinline__ void run(const LinearParams& p, uint16_t* xs, int ld, int wave, int nw, int lane) {
#pragma unroll
    for (int row = 0; row < kRows; ++row)
      if (wave + row * nw < p.M) norm_row(p, xs, ld, row, wave + row * nw, lane);
    for (int m = wave + kRows * nw; m < p.M; m += nw) {
      load_row(p, 0, m, lane);
      norm_row(p, xs, ld, 0, m, lane);
    }
  }
};

// ---------------------------------------------------------------------------
// M > 4 and many units: the tiles of decode_linear_kernel as one stream.  A
// unit's K blocks of 128 k form kA * S chains: block kb belongs to chain kb %
// (kA * S), each chain sums its blocks in order in one accumulator, and the
// chains are added in order: decode_linear_kernel's sums (a chain is one of its
// waves), whatever waves work on them.
//
// A workgroup of nw waves is nw / S groups; the S waves of a group share a
// unit, wave `part` of it taking blocks part, part + S, ..., and group g of the
// grid takes units g, g + (groups in the grid), ... (one each for most of a
// layer's projections, which have about as many units as groups fit the chip).
// A block is four loads (4 KiB); each wave keeps four blocks in flight, across
// unit ends and from before the x rows are staged.  The loads are the same on every path: one that some
// path skips makes the compiler wait for the whole stream at each round (past
// a wave's last block they re-read the start of an x row).
//
// The normalised x rows sit in LDS (16 bytes apart in their banks where there is
// room).  kLong: rows of more than 2560 elements, two rows of 4096 per wave
// requested ahead of the weights instead of three of 2560 (249-254 VGPRs
// instead of 204-209: a workgroup of eight waves per CU either way).  Against
// a workgroup per unit, which stages the rows for every unit and waits for them
// before its first weight load (us at M = 6 / 12 / 16): qkv 6144 x 2560 13.4 /
// 15.4 / 19.8 -> 11.3 / 11.5 / 13.0, 6144 x 4096 19.3 / 26.9 / 29.3 -> 17.1 / 17.5 /
// 19.6, gate and up 19456 x 2560 30.9 / 49.5 / 83.8 -> 21.5 / 23.4 / 24.2, 24576 x
// 4096 51.4 / 103 / 111 -> 38.4 / 38.7 / 40.9, head 196 / 312 / 583 -> 142 / 148 /
// 152.  (Slower by 2-3% at M = 5 only, of what was measured: 8192 x 4096 20.2 ->
// 20.6, 9000 x 1536 10.8 -> 11.1.)
// ---------------------------------------------------------------------------
template <int kEpi, int kA, bool kLong>
__global__ __launch_bounds__(512) void decode_wide_kernel(const LinearParams p, int n_units, int S, int xs_ld) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  constexpr int kDepth = 4;  // blocks in flight; a multiple of kA
  uint16_t* xs = reinterpret_cast<uint16_t*>(lds);
  const int M = p.M, K = p.K, N = p.N;
  float4_t* red = reinterpret_cast<float4_t*>(lds + static_cast<size_t>(M) * xs_ld * 2);
  const int nw = blockDim.x >> 6;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int c = lane & 15, g = lane >> 4;
  const int groups = nw / S, part = wave % S;
  const int u0 = blockIdx.x * groups + wave / S, stride = gridDim.x * groups;
  // every group of the workgroup passes the same number of unit ends (the
  // barriers below); units past the end store nothing
  const int n_iter = (n_units - 1 - static_cast<int>(blockIdx.x) * groups) / stride + 1;
  const int cnt = (K / kLinKBlock - part + S - 1) / S;  // this wave's blocks of a unit
  const int rounds = (cnt + kDepth - 1) / kDepth;       // kDepth blocks each, the last with some left out
  const int n_rounds = n_iter * rounds;
  const bool col_ok = c < M;

  // row r of unit u as a row of w (rows past N repeat the last; not stored)
  auto weight_row = [&](int u, int r) {
    if constexpr (kEpi == kEpiSiluMul)
      return min(8 * u + (r & 7), (N >> 1) - 1) + (r < 8 ? 0 : N >> 1);
    else
      return min(16 * u + r, N - 1);
  };
  NormStage<kLong ? 2 : 3, kLong ? 8 : 5> stage;
  stage.load(p, wave, nw, lane);
  float res0[4];  // the first unit's residual: lane (c, g) ends with rows 4g + i of x row c
  if constexpr (kEpi == kEpiResidual) {
#pragma unroll
    for (int i = 0; i < 4; ++i) res0[i] = bf16_to_f32(p.res[min(c, M - 1) * p.res_ld + weight_row(u0, 4 * g + i)]);
  }
  int lu = u0, li = 0;
  const uint16_t* wp;
  auto point = [&]() {
    wp = lu < n_units ? p.w + static_cast<int64_t>(weight_row(lu, c)) * K + 8 * g : p.x + 8 * g;
  };
  point();
  auto load_block = [&](u32x4_t (&a)[4]) {
    const int k = lu < n_units ? (part + li * S) * kLinKBlock : 0;
    const uint16_t* src = li < cnt ? wp + k : p.x + 8 * g;
#pragma unroll
    for (int j = 0; j < 4; ++j) a[j] = *reinterpret_cast<const u32x4_t*>(src + 32 * j);
    if (++li == rounds * kDepth) {
      li = 0;
      lu += stride;
      point();
    }
  };
  u32x4_t wr[kDepth][4];
#pragma unroll
  for (int d = 0; d < kDepth; ++d) load_block(wr[d]);

  stage.run(p, xs, xs_ld, wave, nw, lane);
  __syncthreads();

  float4_t acc[kA] = {};
  int u = u0, ci = 0;
  auto unit_end = [&]() {
    const int uu = u;
    u += stride;
    ci = 0;
    float4_t s = acc[0];
    if (S > 1) {
      // chain i * S + part of this wave; the unit's chains in order
      float4_t* mine = red + (wave - part) * (64 * kA) + lane;
      if (uu != u0) __syncthreads();  // (the last unit's chains have been read)
#pragma unroll
      for (int i = 0; i < kA; ++i) mine[(i * S + part) * 64] = acc[i];
#pragma unroll
      for (int i = 0; i < kA; ++i) acc[i] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
      __syncthreads();
      if (part != 0) return;
      s = mine[0];
      for (int w = 1; w < kA * S; ++w) {
        const float4_t t = mine[w * 64];
        s[0] += t[0], s[1] += t[1], s[2] += t[2], s[3] += t[3];
      }
    } else {
#pragma unroll
      for (int i = 1; i < kA; ++i) s[0] += acc[i][0], s[1] += acc[i][1], s[2] += acc[i][2], s[3] += acc[i][3];
#pragma unroll
      for (int i = 0; i < kA; ++i) acc[i] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
    }
    if (uu >= n_units) return;
    if constexpr (kEpi == kEpiSiluMul) {
      // gate rows sit in g < 2, the matching up rows 32 lanes higher
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float up = __uint_as_float(__builtin_amdgcn_permlane32_swap(__float_as_uint(s[i]), __float_as_uint(s[i]),
                                                                          false, false)[1]);
        const int j = 8 * uu + 4 * g + i;
        if (g >= 2 || !col_ok || j >= (N >> 1)) continue;
        const float gt = bf16r(s[i]), uv = bf16r(up);
        const float act = bf16r(gt / (1.0f + expf(-gt)));
        store_y(p, c, j, bf16r(act * uv));
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int n = 16 * uu + 4 * g + i;
        if (!col_ok || n >= N) continue;
        float y = bf16r(s[i]);
        if constexpr (kEpi == kEpiResidual)
          y = bf16r((uu == u0 ? res0[i] : bf16_to_f32(p.res[c * p.res_ld + n])) + y);
        store_y(p, c, n, y);
      }
    }
  };
  const uint16_t* xl = xs + min(c, M - 1) * xs_ld + 8 * g;
  for (int t = 0; t < n_rounds; ++t) {
#pragma unroll
    for (int d = 0; d < kDepth; ++d) {
      if (ci + d < cnt) {  // (uniform)
        const uint16_t* xp = xl + (part + (ci + d) * S) * kLinKBlock;
#pragma unroll
        for (int j = 0; j < 4; ++j)
          acc[d % kA] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              __builtin_bit_cast(bf16x8v_t, wr[d][j]),
              __builtin_bit_cast(bf16x8v_t, *reinterpret_cast<const u32x4_t*>(xp + 32 * j)), acc[d % kA], 0, 0, 0);
      }
      load_block(wr[d]);
    }
    ci += kDepth;
    if (ci >= cnt) unit_end();
  }
}

// ---------------------------------------------------------------------------
// The same linear for M <= 4 input rows as a weight stream.  A unit of work
// is kR = 4 (or 8) weight rows over all of K (silu * up: kR / 2 gate rows and the
// matching up rows); every wave takes units gw, gw + (waves in the grid), ... and walks
// their (unit, 512-element chunk) items with two items in flight: each item is
// kR loads of 1 KiB of one weight row (64 lanes x 16 B, whole cache lines,
// nontemporal) and, without a norm, the x rows' 16 B.  The loads are the same
// on every path, as in decode_wide_kernel.  With the norm, the workgroup stages
// the normalised x rows in LDS once (the grid is at most a few workgroups per
// CU, so the staging is amortised over many units), its x and norm-weight loads
// ahead of the first weights.  v_dot2_f32_bf16 accumulates w x x in fp32; at
// the unit's last chunk the lanes' partial sums are reduce-scattered with
// shuffles and the epilogue (that of decode_linear_kernel) runs by lane
// quadruples (kR = 8: pairs).  Waves never wait for each other after the staging.
//
// Bound: HBM, behind ~3 us of launch, first latency and last sums.  Qwen3-4B
// projections at M = 4, cold weights, us: a plain read of the weights / with
// loads that some paths skipped (and so every round waiting for all of them) /
// now: qkv 6.6 / 11.6 / 8.7, o 5.2 / 7.9 / 6.9, gate and up 17.1 / 21.1 / 17.8,
// down 9.2 / 13.1 / 13.0, head 120 / 122 / 119.  Units of 8 rows: 9.2, 7.2, 20.9,
// 14.1, 126; of 2 rows: 8.6, 7.1, 18.1, 13.9, 125.
// ---------------------------------------------------------------------------
constexpr int kGemvMaxM = 4;
constexpr int kGemvChunk = 512;  // elements of one row read by one wave instruction
constexpr int kGemvWaves = 4;

typedef __bf16 bf16x2v_t __attribute__((ext_vector_type(2)));

__device__ __forceinline__ bf16x2v_t as_bf16x2(uint32_t v) { return __builtin_bit_cast(bf16x2v_t, v); }

// (each dword named: a bit_cast of an indexed vector element in an unrolled
// loop compiled to four uses of element 0)
__device__ __forceinline__ float dot8(const u32x4_t w, const u32x4_t x, float acc) {
  const uint32_t w0 = w.x, w1 = w.y, w2 = w.z, w3 = w.w;
  const uint32_t x0 = x.x, x1 = x.y, x2 = x.z, x3 = x.w;
  acc = __builtin_amdgcn_fdot2_f32_bf16(as_bf16x2(w0), as_bf16x2(x0), acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(as_bf16x2(w1), as_bf16x2(x1), acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(as_bf16x2(w2), as_bf16x2(x2), acc, false);
  acc = __builtin_amdgcn_fdot2_f32_bf16(as_bf16x2(w3), as_bf16x2(x3), acc, false);
  return acc;
}

// One step of a reduce-scatter over the lanes: lanes whose `bit` is set keep
// the upper half of the N values, the others the lower half, each adding its
// partner's (lane ^ bit) copy of the half it keeps.
template <int N>
__device__ __forceinline__ void rs_step(const float (&v)[N], float (&o)[N / 2], int lane, int bit) {
  const bool hi = lane & bit;
#pragma unroll
  for (int j = 0; j < N / 2; ++j) {
    const float send = hi ? v[j] : v[j + N / 2];
    const float keep = hi ? v[j + N / 2] : v[j];
    o[j] = keep + __shfl_xor(send, bit);
  }
}

// The sum over the 64 lanes of value lane * kV / 64 of the kV per-lane values
// (the same additions for any kV).
template <int kV>
__device__ __forceinline__ float lane_reduce(const float (&acc)[kV], int lane) {
  static_assert(kV == 16 || kV == 32, "4 or 8 rows of 4");
  if constexpr (kV == 32) {
    float a[16], b[8], c[4], d[2], e[1];
    rs_step<32>(acc, a, lane, 32);
    rs_step<16>(a, b, lane, 16);
    rs_step<8>(b, c, lane, 8);
    rs_step<4>(c, d, lane, 4);
    rs_step<2>(d, e, lane, 2);
    return e[0] + __shfl_xor(e[0], 1);
  } else {
    float a[8], b[4], c[2], d[1];
    rs_step<16>(acc, a, lane, 32);
    rs_step<8>(a, b, lane, 16);
    rs_step<4>(b, c, lane, 8);
    rs_step<2>(c, d, lane, 4);
    const float s = d[0] + __shfl_xor(d[0], 2);
    return s + __shfl_xor(s, 1);
  }
}

// 16 bytes of global memory at a wave-uniform base plus a lane's element
// offset, not kept in the caches.  The base is opaque to the compiler: a load
// from a choice of two stays one load instead of one per branch.
__device__ __forceinline__ u32x4_t stream_load(const uint16_t* base, int off) {
  typedef const __attribute__((address_space(1))) uint16_t* gptr_t;
  typedef const __attribute__((address_space(1))) u32x4_t* gptr16_t;
  uint64_t a = reinterpret_cast<uint64_t>(base);
  asm("" : "+s"(a));
  return __builtin_nontemporal_load(reinterpret_cast<gptr16_t>(reinterpret_cast<gptr_t>(a) + off));
}

// kSplit: the narrow projections.  A unit is then worked by the whole
// workgroup, wave w taking chunks w, w + 4, ... (at least one each: the
// launcher uses it for K >= 4 chunks), and the waves' partial sums meet in
// LDS at the unit's end; the workgroups take units blockIdx.x, blockIdx.x +
// gridDim.x, ...
// kD: items in flight; 1 where no wave has a second item (2048 x 2048, M = 1,
// two loads of which the second only re-reads x: 4.8 us, one: 4.15).
template <int kEpi, bool kNorm, bool kSplit, int kR, int kD>
__global__ __launch_bounds__(64 * kGemvWaves) void decode_stream_kernel(const LinearParams p, int n_units) {
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];
  constexpr int kV = kR * kGemvMaxM;       // values per lane: acc[r * 4 + m]
  constexpr int kShift = kR == 8 ? 1 : 2;  // value i ends in lanes i << kShift on
  float* red = reinterpret_cast<float*>(lds);  // kSplit: [waves][64] partial sums
  uint16_t* xs = reinterpret_cast<uint16_t*>(lds + (kSplit ? kGemvWaves * 64 * 4 : 0));  // normalised x [M][K]
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
  const int M = p.M, K = p.K, N = p.N;
  const int n_chunks = (K + kGemvChunk - 1) / kGemvChunk;
  // this wave's units u0, u0 + du, ... and chunks c0, c0 + dc, ... (cnt per unit)
  const int u0 = kSplit ? blockIdx.x : blockIdx.x * kGemvWaves + wave;
  const int du = kSplit ? gridDim.x : gridDim.x * kGemvWaves;
  const int c0 = kSplit ? wave : 0, dc = kSplit ? kGemvWaves : 1;
  const int cnt = kSplit ? (n_chunks - wave + kGemvWaves - 1) / kGemvWaves : n_chunks;
  const int n_my = u0 < n_units ? (n_units - 1 - u0) / du + 1 : 0;
  const int n_items = n_my * cnt;

  // weight row r of a unit (rows past N repeat the last one; not stored)
  auto unit_row = [&](int u, int r) {
    if constexpr (kEpi == kEpiSiluMul) {
      const int half = N >> 1, j = min(u * (kR / 2) + (r % (kR / 2)), half - 1);
      return r < kR / 2 ? j : half + j;
    } else {
      return min(u * kR + r, N - 1);
    }
  };
  NormStage<1, 5> stage;
  if constexpr (kNorm) stage.load(p, wave, kGemvWaves, lane);
  // the first unit's residual (of the lane that stores it)
  const int o_idx = lane >> kShift, o_r = o_idx / kGemvMaxM, o_m = o_idx % kGemvMaxM;
  float res0 = 0.0f;
  if constexpr (kEpi == kEpiResidual)
    res0 = bf16_to_f32(p.res[min(o_m, M - 1) * p.res_ld + unit_row(min(u0, n_units - 1), o_r)]);

  // past the wave's last item the loads re-read the first x row's start;
  // lanes past K re-read the row's last 16 bytes (zeroed before use)
  int lu = u0, lc = c0, li = 0;
  auto load_item = [&](u32x4_t (&wv)[kR], u32x4_t (&xv)[kGemvMaxM]) {
    const bool ok = lu < n_units;
    const int k = ok ? min(lc * kGemvChunk + 8 * lane, K - 8) : 8 * (lane & 15);
#pragma unroll
    for (int r = 0; r < kR; ++r)
      wv[r] = stream_load(ok ? p.w + static_cast<int64_t>(unit_row(lu, r)) * K : p.x, k);
    if constexpr (!kNorm) {
#pragma unroll
      for (int m = 0; m < kGemvMaxM; ++m)
        xv[m] = *reinterpret_cast<const u32x4_t*>(p.x + min(m, M - 1) * p.x_ld + k);
    }
    lc += dc;
    if (++li == cnt) lu += du, lc = c0, li = 0;
  };
  u32x4_t wr[kD][kR], xr[kD][kGemvMaxM];
#pragma unroll
  for (int d = 0; d < kD; ++d) load_item(wr[d], xr[d]);

  if constexpr (kNorm) {
    stage.run(p, xs, K, wave, kGemvWaves, lane);
    __syncthreads();
  }

  float acc[kV];
#pragma unroll
  for (int j = 0; j < kV; ++j) acc[j] = 0.0f;
  int cu = u0, cc = c0, ci = 0;
  // this wave's last chunk of a unit: sums over the lanes (and, split, over
  // the waves), epilogue, fresh accumulators
  auto unit_end = [&]() {
    const int u = cu;
    cu += du, cc = c0, ci = 0;
    float s = lane_reduce(acc, lane);
#pragma unroll
    for (int j = 0; j < kV; ++j) acc[j] = 0.0f;
    if constexpr (kSplit) {
      red[wave * 64 + lane] = s;
      __syncthreads();
      if (wave == 0) {
#pragma unroll
        for (int w = 1; w < kGemvWaves; ++w) s += red[w * 64 + lane];
      }
      __syncthreads();  // red is free for the next unit
      if (wave != 0) return;
    }
    const bool lead = (lane & ((1 << kShift) - 1)) == 0;
    if constexpr (kEpi == kEpiSiluMul) {
      // the up row of gate row r sits kR / 2 rows (32 lanes) higher
      const float up = __shfl_xor(s, 32);
      const int row = u * (kR / 2) + o_r;
      if (lane >= 32 || !lead || o_m >= M || row >= (N >> 1)) return;
      const float gt = bf16r(s), uv = bf16r(up);
      const float act = bf16r(gt / (1.0f + expf(-gt)));
      store_y(p, o_m, row, bf16r(act * uv));
    } else {
      const int row = u * kR + o_r;
      if (!lead || o_m >= M || row >= N) return;
      float y = bf16r(s);
      if constexpr (kEpi == kEpiResidual)
        y = bf16r((u == u0 ? res0 : bf16_to_f32(p.res[o_m * p.res_ld + row])) + y);
      store_y(p, o_m, row, y);
    }
  };
  auto step = [&](u32x4_t (&wv)[kR], u32x4_t (&xv)[kGemvMaxM]) {
    const int k = cc * kGemvChunk + 8 * lane;
    if constexpr (kNorm) {
#pragma unroll
      for (int m = 0; m < kGemvMaxM; ++m)
        xv[m] = *reinterpret_cast<const u32x4_t*>(xs + min(m, M - 1) * K + min(k, K - 8));
    }
    if (cc * kGemvChunk + kGemvChunk > K) {  // (uniform) the chunk ends inside the wave
      const u32x4_t zero = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int r = 0; r < kR; ++r) wv[r] = k < K ? wv[r] : zero;
#pragma unroll
      for (int m = 0; m < kGemvMaxM; ++m) xv[m] = k < K ? xv[m] : zero;
    }
#pragma unroll
    for (int r = 0; r < kR; ++r)
#pragma unroll
      for (int m = 0; m < kGemvMaxM; ++m)
        acc[r * kGemvMaxM + m] = dot8(wv[r], xv[m], acc[r * kGemvMaxM + m]);
    cc += dc;
  };
  // rounds of kD items, refilled while there is a round to refill for, then the
  // last round alone
  int t = 0;
  for (; t + kD < n_items; t += kD) {
#pragma unroll
    for (int d = 0; d < kD; ++d) {
      step(wr[d], xr[d]);
      load_item(wr[d], xr[d]);
      if (++ci == cnt) unit_end();
    }
  }
#pragma unroll
  for (int d = 0; d < kD; ++d) {
    if (t + d < n_items) {
      step(wr[d], xr[d]);
      if (++ci == cnt) unit_end();
    }
  }
}

// ---------------------------------------------------------------------------
// q / k: per-head RMSNorm (bf16 out), then rotate-half RoPE at one position
// (bf16 out); v copied.  One wave per head of one batch row; lane l holds
// channels l and l + 64 (the two halves RoPE pairs).  Heads [0, hq) are q
// (to q_out), [hq, hq + hkv) k and [hq + hkv, hq + 2 hkv) v (to the cache).
// ---------------------------------------------------------------------------
struct QkParams {
  const uint16_t* qkv;  // [bs, (hq + 2 hkv) * 128] bf16, row stride qkv_ld
  int64_t qkv_ld;
  const uint16_t* q_norm;  // [128] bf16
  const uint16_t* k_norm;  // [128] bf16
  float eps;
  const float* cos;  // [64] fp32 (the position's row)
  const float* sin;
  uint16_t* q_out;  // [bs, hq, 128]
  uint16_t* k_dst;  // row of (b, h): k_dst + b * k_sb + h * k_sh
  int64_t k_sb, k_sh;
  uint16_t* v_dst;
  int64_t v_sb, v_sh;
  int bs, hq, hkv;
};

__global__ __launch_bounds__(256) void qk_norm_rope_kernel(const QkParams p) {
  const int heads = p.hq + 2 * p.hkv;
  const int item = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (item >= p.bs * heads) return;
  const int b = item / heads, h = item - b * heads, lane = threadIdx.x & 63;
  const uint16_t* src = p.qkv + b * p.qkv_ld + h * 128;
  const float x1 = bf16_to_f32(src[lane]), x2 = bf16_to_f32(src[lane + 64]);
  if (h >= p.hq + p.hkv) {  // v: straight copy
    uint16_t* dst = p.v_dst + b * p.v_sb + (h - p.hq - p.hkv) * p.v_sh;
    dst[lane] = src[lane];
    dst[lane + 64] = src[lane + 64];
    return;
  }
  const bool is_q = h < p.hq;
  const uint16_t* nw = is_q ? p.q_norm : p.k_norm;
  const float ss = wave_sum(x1 * x1 + x2 * x2);
  const float r = rsqrtf(ss * (1.0f / 128.0f) + p.eps);
  const float n1 = bf16r((x1 * r) * bf16_to_f32(nw[lane]));
  const float n2 = bf16r((x2 * r) * bf16_to_f32(nw[lane + 64]));
  const float cs = p.cos[lane], sn = p.sin[lane];
  const uint16_t y1 = f32_to_bf16_bits(n1 * cs - n2 * sn);
  const uint16_t y2 = f32_to_bf16_bits(n2 * cs + n1 * sn);
  uint16_t* dst = is_q ? p.q_out + (static_cast<int64_t>(b) * p.hq + h) * 128
                       : p.k_dst + b * p.k_sb + (h - p.hq) * p.k_sh;
  dst[lane] = y1;
  dst[lane + 64] = y2;
}

}  // namespace
}  // namespace zkv

using namespace zkv;

extern "C" int zkv_decode_linear(const uint16_t* x, int64_t x_ld, int M, int K, const uint16_t* w, int N,
                                 const uint16_t* norm_w, float eps, const uint16_t* residual, int64_t res_ld,
                                 void* out, int64_t out_ld, int out_f32, int epilogue, zkv_stream_t stream) {
  ZKV_REQUIRE(x && w && out, "zkv_decode_linear: null pointer");
  ZKV_REQUIRE(M >= 1 && M <= kLinMaxM, "zkv_decode_linear: M=%d outside [1, %d]", M, kLinMaxM);
  ZKV_REQUIRE(K > 0 && K % kLinKBlock == 0, "zkv_decode_linear: K=%d is not a positive multiple of %d", K,
              kLinKBlock);
  ZKV_REQUIRE(N > 0, "zkv_decode_linear: N=%d", N);
  ZKV_REQUIRE(epilogue >= kEpiNone && epilogue <= kEpiSiluMul, "zkv_decode_linear: epilogue %d", epilogue);
  ZKV_REQUIRE(epilogue != kEpiResidual || residual, "zkv_decode_linear: residual epilogue without residual");
  ZKV_REQUIRE(epilogue != kEpiSiluMul || N % 2 == 0, "zkv_decode_linear: silu * up needs an even N (%d)", N);
  ZKV_REQUIRE(x_ld >= K && x_ld % 8 == 0 && (reinterpret_cast<uintptr_t>(x) & 15) == 0 &&
                  (reinterpret_cast<uintptr_t>(w) & 15) == 0 &&
                  (norm_w == nullptr || (reinterpret_cast<uintptr_t>(norm_w) & 15) == 0),
              "zkv_decode_linear: x, w and the norm weight need 16-byte aligned rows");
  const size_t x_bytes = static_cast<size_t>(M) * K * 2;
  // units of 16 weight rows (silu * up: 8 gate and 8 up)
  const int n_tiles = epilogue == kEpiSiluMul ? (N / 2 + 7) / 8 : (N + 15) / 16;
  // waves per tile of decode_linear_kernel: enough resident waves to keep the
  // weight stream busy, and few enough blocks per wave that its loads overlap.
  // The x rows and 1 KiB for each of these waves fit the LDS
  const int nkb = K / kLinKBlock;
  int nw = 1;
  while (nw < 16 && nw * 2 <= nkb && static_cast<int64_t>(n_tiles) * nw < 4096) nw *= 2;
  while (nw < 16 && (nkb + nw - 1) / nw > 6) nw *= 2;
  ZKV_REQUIRE(x_bytes + static_cast<size_t>(nw) * 1024 <= 160 * 1024,
              "zkv_decode_linear: M x K = %d x %d needs %zu bytes of LDS (limit 160 KiB)", M, K,
              x_bytes + static_cast<size_t>(nw) * 1024);
  LinearParams p{x, x_ld, w, norm_w, eps, residual, res_ld, out, out_ld, M, K, N, out_f32};
  auto s = reinterpret_cast<hipStream_t>(stream);
  // dynamic LDS above 64 KiB has to be allowed per kernel (once)
#define ZKV_LAUNCH(KERNEL, GRID, BLOCK, LDS, ...)                                                     \
  do {                                                                                                \
    static bool big_lds_set = false;                                                                  \
    if ((LDS) > 64 * 1024 && !big_lds_set) {                                                          \
      if (hipFuncSetAttribute(reinterpret_cast<const void*>(&KERNEL),                                 \
                              hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024) != hipSuccess) \
        return fail(ZKV_EINVAL, "zkv_decode_linear: cannot raise the LDS limit to 160 KiB");          \
      big_lds_set = true;                                                                             \
    }                                                                                                 \
    KERNEL<<<GRID, BLOCK, LDS, s>>>(__VA_ARGS__);                                                     \
  } while (0)
#define ZKV_COMMA ,
  if (M <= kGemvMaxM) {
    // the weight stream; narrow projections (fewer rows than ~2 units per wave
    // of a full chip) split K over the waves of a workgroup
    const int rows = epilogue == kEpiSiluMul ? N / 2 : N;
    const int n_chunks = (K + kGemvChunk - 1) / kGemvChunk;
    const bool split = rows < 8192 && n_chunks >= kGemvWaves && !norm_w;
    // without a norm each item loads the x rows too: units of 8 rows halve that
    // from 40000 weight rows on; 151936 x 2560, M = 1 / 4, us: 4 rows 113 / 124, 8 rows
    // 112 / 113; 65536 x 2048 50.1 / 51.3 and 46.4 / 47.0.  Fewer rows give the waves
    // too few units (36000 x 2048 24.6 / 25.2 and 27.2 / 27.3), one x row and rows of
    // 1024 have little to halve (65536 x 6144 119 and 122 at M = 1; 151936 x 1024 47.4
    // / 48.0 and 48.8 / 48.5), and 8 rows whole multiples of 8 KiB apart meet on the
    // same channels (65536 x 4096 84 / 87 and 110 / 113; silu * up, whose rows are two
    // runs of 4, not: 40000 x 4096 57.7 / 59.8 and 53.4 / 53.4).
    const bool tall = !norm_w && N >= 40000 && K > 1024 && (M >= 2 || K < 4096) &&
                      (K % 4096 != 0 || epilogue == kEpiSiluMul);
    const int R = tall ? 8 : 4;
    const int per_unit = epilogue == kEpiSiluMul ? R / 2 : R;
    const int n_units = (rows + per_unit - 1) / per_unit;
    const int n_groups = split ? n_units : (n_units + kGemvWaves - 1) / kGemvWaves;
    const int grid = std::max(1, std::min(n_groups, 768));
    // one unit and one chunk of it for each wave (a norm's staging hides the rest)
    const bool once = !norm_w && n_groups <= 768 && n_chunks == (split ? kGemvWaves : 1);
    const size_t lds = (split ? kGemvWaves * 64 * 4 : 0) + (norm_w ? x_bytes : 0);
#define ZKV_GEMV_L(E, NORM, SPLIT, R, D)                                                                 \
  ZKV_LAUNCH(decode_stream_kernel<E ZKV_COMMA NORM ZKV_COMMA SPLIT ZKV_COMMA R ZKV_COMMA D>, grid, 64 * kGemvWaves, lds, \
             p, n_units)
#define ZKV_GEMV(E)                                          \
  do {                                                       \
    if (norm_w) ZKV_GEMV_L(E, true, false, 4, 2);            \
    else if (tall) ZKV_GEMV_L(E, false, false, 8, 2);        \
    else if (split && once) ZKV_GEMV_L(E, false, true, 4, 1); \
    else if (split) ZKV_GEMV_L(E, false, true, 4, 2);        \
    else if (once) ZKV_GEMV_L(E, false, false, 4, 1);        \
    else ZKV_GEMV_L(E, false, false, 4, 2);                  \
  } while (0)
    if (epilogue == kEpiNone) ZKV_GEMV(kEpiNone);
    else if (epilogue == kEpiResidual) ZKV_GEMV(kEpiResidual);
    else ZKV_GEMV(kEpiSiluMul);
#undef ZKV_GEMV
#undef ZKV_GEMV_L
    return check_launch("decode_stream_kernel");
  }
  if (norm_w && static_cast<int64_t>(n_tiles) * nkb >= 6144) {
    // 24 MB of weights and more: a workgroup per tile against this stream, M = 6,
    // 4096 x 1024 (2048 blocks) 5.9 and 6.6 us, 6144 x 2048 (6144) 11.6 and 9.2,
    // 6144 x 2560 (7680) 13.4 and 11.3.
    // The nw chains of a unit's sum are nw / S accumulators in each of S waves.  S
    // is the split whose waves take the fewest rounds of kDepth blocks: 2048 waves
    // run at a time, and a wave loads whole rounds.  Fewer waves per unit unless
    // more save a sixteenth: 8192 x 2560, M = 6, S = 2 (128 workgroups) 16.3 us, S = 4
    // (256) 12.8; 4096 x 4096 S = 4 17.0, S = 8 11.8; 24576 x 4096 S = 2 54, S = 4
    // 38.7; the head of 4096, 151936 rows, S = 2 (160 rounds) 237, S = 4 (152) 242.
    // (The first figure of each with the long rows requested late.)
    int S = 0, best = 0;
    for (int t = std::max(nw / 4, 1); t <= std::min(nw, 8); t *= 2) {
      const int turns = static_cast<int>((static_cast<int64_t>(n_tiles) * t + 2047) / 2048);
      const int rounds = turns * (((nkb + t - 1) / t + 3) / 4);
      if (S == 0 || 16 * rounds < 15 * best) best = rounds, S = t;
    }
    // eight waves (six where a unit takes one) stage the rows
    const int per_wave = nw / S;
    int nwv = S == 1 ? 6 : 8;
    // (one unit's chains always fit: the requirement above)
    if (S > 1 && x_bytes + static_cast<size_t>(nwv) * per_wave * 1024 > 160 * 1024) nwv = S;
    const size_t red_bytes = S > 1 ? static_cast<size_t>(nwv) * per_wave * 1024 : 0;
    // x rows 16 bytes apart in their banks where the LDS holds the padding
    const int xs_ld = x_bytes + M * 16 + red_bytes <= 160 * 1024 ? K + 8 : K;
    const size_t lds = static_cast<size_t>(M) * xs_ld * 2 + red_bytes;
    // a workgroup per CU, what the registers allow: one that waits for another's
    // end would stage the rows again
    const int grid = std::min((n_tiles + nwv / S - 1) / (nwv / S), 256);
    const bool long_rows = K > 2560;
#define ZKV_WIDE_L(E, A, L) \
  ZKV_LAUNCH(decode_wide_kernel<E ZKV_COMMA A ZKV_COMMA L>, grid, 64 * nwv, lds, p, n_tiles, S, xs_ld)
#define ZKV_WIDE_A(E, A)                        \
  do {                                          \
    if (long_rows) ZKV_WIDE_L(E, A, true);      \
    else ZKV_WIDE_L(E, A, false);               \
  } while (0)
#define ZKV_WIDE(E)                             \
  do {                                          \
    if (per_wave == 4) ZKV_WIDE_A(E, 4);        \
    else if (per_wave == 2) ZKV_WIDE_A(E, 2);   \
    else ZKV_WIDE_A(E, 1);                      \
  } while (0)
    if (epilogue == kEpiNone) ZKV_WIDE(kEpiNone);
    else if (epilogue == kEpiResidual) ZKV_WIDE(kEpiResidual);
    else ZKV_WIDE(kEpiSiluMul);
#undef ZKV_WIDE
#undef ZKV_WIDE_A
#undef ZKV_WIDE_L
    return check_launch("decode_wide_kernel");
  }
  if (!norm_w) {
    // rows (or pairs) per unit: the number of units is rounded up to whole rounds
    // of 256 CUs (160 tiles of 16 rows leave 96 CUs idle: down at M = 6 17.1 us, in
    // 256 units of 10 rows 13.1)
    const int rows = epilogue == kEpiSiluMul ? N / 2 : N;
    const int units = (n_tiles + 255) / 256 * 256;
    const int R = (rows + units - 1) / units;
    const int grid = (rows + R - 1) / R;
    // at most 8 blocks per wave: the LDS requirement above bounds K at M >= 5
    const int cnt = (nkb + nw - 1) / nw;
#define ZKV_ROWS_CNT(E, C)                                                    \
  case C:                                                                     \
    decode_rows_kernel<E, C><<<grid, 64 * nw, 0, s>>>(p, R);                  \
    break;
#define ZKV_ROWS(E)                                                           \
  switch (cnt) {                                                              \
    ZKV_ROWS_CNT(E, 1) ZKV_ROWS_CNT(E, 2) ZKV_ROWS_CNT(E, 3) ZKV_ROWS_CNT(E, 4) \
    ZKV_ROWS_CNT(E, 5) ZKV_ROWS_CNT(E, 6) ZKV_ROWS_CNT(E, 7) ZKV_ROWS_CNT(E, 8) \
    default:                                                                  \
      return fail(ZKV_EINVAL, "zkv_decode_linear: %d K blocks per wave", cnt); \
  }
    if (epilogue == kEpiNone) ZKV_ROWS(kEpiNone)
    else if (epilogue == kEpiResidual) ZKV_ROWS(kEpiResidual)
    else ZKV_ROWS(kEpiSiluMul)
#undef ZKV_ROWS
#undef ZKV_ROWS_CNT
    return check_launch("decode_rows_kernel");
  }
  const size_t lds = x_bytes + static_cast<size_t>(nw) * 1024;
  if (epilogue == kEpiNone) ZKV_LAUNCH(decode_linear_kernel<kEpiNone>, n_tiles, 64 * nw, lds, p);
  else if (epilogue == kEpiResidual) ZKV_LAUNCH(decode_linear_kernel<kEpiResidual>, n_tiles, 64 * nw, lds, p);
  else ZKV_LAUNCH(decode_linear_kernel<kEpiSiluMul>, n_tiles, 64 * nw, lds, p);
#undef ZKV_COMMA
#undef ZKV_LAUNCH
  return check_launch("decode_linear_kernel");
}

extern "C" int zkv_qk_norm_rope(const uint16_t* qkv, int64_t qkv_ld, int bs, int hq, int hkv,
                                const uint16_t* q_norm, const uint16_t* k_norm, float eps, const float* cos_row,
                                const float* sin_row, uint16_t* q_out, uint16_t* k_dst, int64_t k_sb,
                                int64_t k_sh, uint16_t* v_dst, int64_t v_sb, int64_t v_sh, zkv_stream_t stream) {
  ZKV_REQUIRE(qkv && q_norm && k_norm && cos_row && sin_row && q_out && k_dst && v_dst,
              "zkv_qk_norm_rope: null pointer");
  ZKV_REQUIRE(bs > 0 && hq > 0 && hkv > 0 && qkv_ld >= static_cast<int64_t>(hq + 2 * hkv) * 128,
              "zkv_qk_norm_rope: bad sizes bs=%d hq=%d hkv=%d qkv_ld=%lld", bs, hq, hkv,
              static_cast<long long>(qkv_ld));
  const QkParams p{qkv, qkv_ld, q_norm, k_norm, eps, cos_row, sin_row, q_out, k_dst, k_sb, k_sh,
                   v_dst, v_sb, v_sh, bs, hq, hkv};
  const int items = bs * (hq + 2 * hkv);
  qk_norm_rope_kernel<<<(items + 3) / 4, 256, 0, reinterpret_cast<hipStream_t>(stream)>>>(p);
  return check_launch("qk_norm_rope_kernel");
}
