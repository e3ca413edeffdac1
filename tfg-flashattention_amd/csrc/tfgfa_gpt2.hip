// tfgfa_gpt2.hip - the GPT-2 block around the attention, MI355X (gfx950).
//
// The reference's block (src/py/model_inference.py:96-164) spells its LayerNorm, GELU and
// residual adds out as elementwise operators; each is then a pass over memory of its own, and a
// decode step of a few rows is some 45 launches per layer.  Here:
//   layernorm_kernel    LayerNorm of a row held in one wave's registers, with the residual add
//                       before it and the rounding to bf16 after it where the caller has them;
//   gelu_kernel         the tanh GELU in one pass;
//   cast_kernel         float32 -> bf16 copies of several weights in one launch;
//   linear_rows_kernel  a projection of at most 8 rows read straight from the float32 weights,
//                       with the LayerNorm before it and the bias, GELU and residual after it.
//
// Compiled with NaN semantics kept (unlike the attention kernels): these functions pass
// infinities and NaN through as the elementwise operators do.
#include <hip/hip_runtime.h>

#include <math.h>
#include <stdint.h>

#include <algorithm>

#include "tfgfa.h"
#include "tfgfa_gpt2.h"

namespace tfgpt2 {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 load4(const float* p) { return *reinterpret_cast<const f32x4*>(p); }
__device__ __forceinline__ f32x4 load4(const __bf16* p) {
  return __builtin_convertvector(*reinterpret_cast<const bf16x4*>(p), f32x4);
}
__device__ __forceinline__ void store4(float* p, f32x4 v) { *reinterpret_cast<f32x4*>(p) = v; }
__device__ __forceinline__ void store4(__bf16* p, f32x4 v) {
  *reinterpret_cast<bf16x4*>(p) = __builtin_convertvector(v, bf16x4);
}

template <int kCtrl>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xF, 0xF, false));
}
// Sum over the 16 lanes that are 4 apart, in each of them.
__device__ __forceinline__ float block_sum(float x) {
  x = dpp_add<0x124>(x);  // row of 16: rotated by 4
  x = dpp_add<0x128>(x);  // row of 16: rotated by 8
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);  // rows 0 and 1, rows 2 and 3
  const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}
// Sum over the 64 lanes, in every lane.
__device__ __forceinline__ float wave_sum(float x) {
  x = dpp_add<0xB1>(x);  // quad: lanes 1 apart
  x = dpp_add<0x4E>(x);  // quad: lanes 2 apart
  return block_sum(x);
}

__device__ __forceinline__ float gelu(float x) {
  return 0.5f * x * (1.0f + tanhf(0.7978845608028654f * (x + 0.044715f * (x * x * x))));
}

// Normalises a row held as v[i] = elements 4 * (64 i + lane) .. +3 (those below d; the others are
// zero) in place: two passes over registers, so the variance is that of the centred values.
template <int kV>
__device__ __forceinline__ void normalise_row(f32x4 (&v)[kV], int d, int lane, float eps) {
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < kV; ++i) s += (v[i][0] + v[i][1]) + (v[i][2] + v[i][3]);
  const float inv_d = 1.0f / (float)d;
  const float mean = wave_sum(s) * inv_d;
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < kV; ++i) {
    if (4 * (64 * i + lane) < d) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[i][e] -= mean;
        q = fmaf(v[i][e], v[i][e], q);
      }
    }
  }
  const float r = 1.0f / sqrtf(wave_sum(q) * inv_d + eps);
#pragma unroll
  for (int i = 0; i < kV; ++i) v[i] *= r;
}

// ---------------------------------------------------------------------------------------
// LayerNorm.  Bound: memory (one read of the row, one write); at the some hundred rows of a prompt,
// the latency of a row's chain: its loads, two reductions, its stores.  One wave per row: the row
// stays in registers, and a reduction is 6 cross-lane steps with no barrier.  scale and shift are
// loaded with the row, not after the reductions.  kV * 256 elements per row.
//   613 rows of 1600: 4.9 us to bf16, 5.1 us with the residual (four rows per workgroup,
//   scale and shift loaded where used: 7.2 and 9.3); the operators they stand for: about 32 us a
//   norm, and 86 us for the mixed bf16 + float32 add before the second.
template <int kV, bool kDelta, typename Y>
__global__ __launch_bounds__(64) void layernorm_kernel(
    const float* x, const __bf16* __restrict__ delta, float* sum, const float* __restrict__ scale,
    const float* __restrict__ shift, Y* __restrict__ y, int d, float eps) {
  const int lane = threadIdx.x;
  const long long base = (long long)blockIdx.x * d;
  // Elements past the row are read at its start and zeroed: loads with no branch between them go
  // out together.
  f32x4 v[kV], g[kV], h[kV], dl[kDelta ? kV : 1];
#pragma unroll
  for (int i = 0; i < kV; ++i) {
    const int c = 4 * (64 * i + lane), cc = c < d ? c : 0;
    v[i] = load4(x + base + cc);
    if constexpr (kDelta) dl[i] = load4(delta + base + cc);
  }
#pragma unroll
  for (int i = 0; i < kV; ++i) {
    const int c = 4 * (64 * i + lane), cc = c < d ? c : 0;
    g[i] = load4(scale + cc);
    h[i] = load4(shift + cc);
  }
#pragma unroll
  for (int i = 0; i < kV; ++i) {
    const int c = 4 * (64 * i + lane);
    if constexpr (kDelta) v[i] += dl[i];
    if (c >= d) v[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    if constexpr (kDelta)
      if (c < d) store4(sum + base + c, v[i]);
  }
  normalise_row(v, d, lane, eps);
#pragma unroll
  for (int i = 0; i < kV; ++i) {
    const int c = 4 * (64 * i + lane);
    if (c < d) store4(y + base + c, v[i] * g[i] + h[i]);
  }
}

// ---------------------------------------------------------------------------------------
// GELU.  Bound: memory (4 bytes read and written per value): 613 x 6400 values take 6.5 us, 4.8 TB/s;
// the eight operators they stand for took 46 us.
constexpr int kGeluThreads = 256;
__global__ __launch_bounds__(kGeluThreads) void gelu_kernel(const float* __restrict__ x,
                                                            float* __restrict__ y, long long n) {
  const long long i = ((long long)blockIdx.x * kGeluThreads + threadIdx.x) * 4;
  if (i + 4 <= n) {
    const f32x4 v = load4(x + i);
    store4(y + i, f32x4{gelu(v[0]), gelu(v[1]), gelu(v[2]), gelu(v[3])});
  } else {
    for (long long j = i; j < n; ++j) y[j] = gelu(x[j]);
  }
}

// ---------------------------------------------------------------------------------------
// float32 -> bf16.  Bound: memory.  The arrays are laid end to end in units of 4 values.
constexpr int kMaxCasts = TFGPT2_MAX_CASTS;
constexpr int kCastThreads = 256;
struct Casts {
  const float* src[kMaxCasts];
  __bf16* dst[kMaxCasts];
  long long end[kMaxCasts];  // units of 4 values up to and including array i
  int count;
};
__global__ __launch_bounds__(kCastThreads) void cast_kernel(Casts a) {
  const long long u = (long long)blockIdx.x * kCastThreads + threadIdx.x;
  long long begin = 0;
#pragma unroll
  for (int i = 0; i < kMaxCasts; ++i) {
    if (i < a.count) {
      if (u >= begin && u < a.end[i]) store4(a.dst[i] + 4 * (u - begin), load4(a.src[i] + 4 * (u - begin)));
      begin = a.end[i];
    }
  }
}

// ---------------------------------------------------------------------------------------
// A linear layer on at most 8 rows.
//
// Bound: memory, the float32 weights read once (4 K N bytes); at the sizes of a GPT-2 layer (4 to
// 40 MB per projection) the launch and the latency of the first loads weigh as much.
// v_mfma_f32_4x4x1f32 multiplies 16 independent 4 x 4 blocks with a contraction length of 1.
// Here block b is a piece of the contraction, not of the output: lane l = i + 4b loads 16 bytes of
// weight row i at k = 64 s + 4 b .. +3 (s: a strip of 64), so a wave's load is 4 rows x 256
// contiguous bytes, and four MFMAs (one per element) accumulate
//   D_b[i][j] += w[i][64 s + 4 b + e] * x[j][64 s + 4 b + e];
// the 16 block sums are added at the end.  So 4 weight rows are enough to fill a wave's loads,
// which spreads even N = 768 over 192 workgroups; with 16-row tiles (16x16x4) a projection to
// 1024 outputs would use 64 of the 256 CUs.
//   Lane layout (4x4x1, 16 blocks): A[i] at lane i + 4b; B[j] at lane j + 4b; D[i][j] in register
//   i of lane j + 4b.
// A workgroup owns 4 outputs; its kW waves take the strips in turn, kStrips each in one batch of
// loads (x's rows with them, or first of all the rows to be normalised, so that the norm does not
// wait for the weights), and add their sums in LDS, in a fixed order.  A batch loads without a
// branch (values past K are read at the row's start and zeroed): after one the compiler could not
// count the loads in flight and would wait for the weights before the norm.
//   GPT-2 medium, 4 rows, inside a replayed step (us): norm + query/key/value 6.4 (12.6 MB of
//   weights), output projection 4.8 (4.2 MB), norm + MLP up + GELU 7.3 (16.8 MB, 2.3 TB/s), MLP
//   down 6.8; with two row tiles per workgroup, 8 waves, x read where used and the weights loaded
//   before the rows to be normalised: 14.6, 6.8, 15.2 and 9.5.  The linear layers alone took 3 x 6.9,
//   6.9, 13.0 and 11.4, behind casts of the attention's weights (8 x 2.6), norms and GELU.
constexpr int kTileRows = 4;               // outputs per workgroup and part
constexpr int kNormWaves = 4;              // waves per workgroup with the norm
constexpr int kNormPad = 4;                // floats between the normalised rows in LDS
constexpr int kMaxParts = 3;
constexpr int kNormLdsFloats = 15360;      // M * (K + kNormPad) at most (60 KiB)

struct RowsOut {
  const float* bias[kMaxParts];
  void* y[kMaxParts];
  const float* residual;
  float eps;
};

// kG: groups of 4 rows of x; kV: 256-element pieces of a normalised row (0: no norm); tiles:
// workgroups per part.  The first 14 argument dwords arrive in SGPRs (-amdgpu-kernarg-preload-count):
// what the weight and row loads need.  The bias and the residual are loaded beside the weights, not
// where they are added: a round trip less at the end of a kernel of a few.
template <int kW, int kStrips, int kG, typename X, typename Y, int kV, bool kGelu>
__global__ __launch_bounds__(64 * kW) void linear_rows_kernel(
    const void* __restrict__ x, const float* __restrict__ w0, const float* __restrict__ w1,
    const float* __restrict__ w2, int M, int N, int K, int tiles, const float* __restrict__ ln_scale,
    const float* __restrict__ ln_shift, RowsOut out) {
  extern __shared__ __attribute__((aligned(16))) float xs[];  // kV: M rows of K + kNormPad floats
  __shared__ float red[kW][kG][4][4];                         // [wave][col group][row][col]
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i = lane & 3, b = lane >> 2;
  const int part = blockIdx.x / tiles;
  const int n0 = (blockIdx.x - part * tiles) * kTileRows;
  const float* w = part == 0 ? w0 : part == 1 ? w1 : w2;
  const int nStrips = (K + 63) / 64;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};

  // Column 4 g + i of the operand is row min(4 g + i, M - 1) of x; weight rows past N are row N - 1
  // (neither's sums are stored).
  int col[kG];
#pragma unroll
  for (int g = 0; g < kG; ++g) col[g] = min(4 * g + i, M - 1);
  const float* wrow = w + (long long)min(n0 + i, N - 1) * K;
  f32x4 wv[kStrips], xv[kV ? 1 : kStrips][kG];
  // The batch of strips s0, s0 + kW, ..
  auto load_batch = [&](int s0) {
#pragma unroll
    for (int u = 0; u < kStrips; ++u) {
      const int k = 64 * (s0 + u * kW) + 4 * b, kk = k < K ? k : 0;
      wv[u] = load4(wrow + kk);
      if constexpr (kV == 0) {
#pragma unroll
        for (int g = 0; g < kG; ++g) xv[u][g] = load4(static_cast<const X*>(x) + (long long)col[g] * K + kk);
      }
    }
  };

  if constexpr (kV > 0) {
    // Row m of x by wave m % kW, normalised into LDS.
    f32x4 v[kV], g[kV], h[kV];
    for (int m = wave; m < M; m += kW) {
      const float* xr = static_cast<const float*>(x) + (long long)m * K;
#pragma unroll
      for (int c = 0; c < kV; ++c) {
        const int k = 4 * (64 * c + lane), kk = k < K ? k : 0;
        v[c] = load4(xr + kk);
        g[c] = load4(ln_scale + kk);
        h[c] = load4(ln_shift + kk);
      }
      if (m == wave) load_batch(wave);
#pragma unroll
      for (int c = 0; c < kV; ++c)
        if (4 * (64 * c + lane) >= K) v[c] = zero;
      normalise_row(v, K, lane, out.eps);
#pragma unroll
      for (int c = 0; c < kV; ++c) {
        const int k = 4 * (64 * c + lane);
        if (k < K) *reinterpret_cast<f32x4*>(xs + m * (K + kNormPad) + k) = v[c] * g[c] + h[c];
      }
    }
    if (wave >= M) load_batch(wave);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
  } else {
    load_batch(wave);
  }

  // Thread -> (row m of x, output r of the workgroup's four) of the results.
  const int r = threadIdx.x % kTileRows, m = threadIdx.x / kTileRows, n = n0 + r;
  const bool writes = m < M && n < N;
  const float* bias = part == 0 ? out.bias[0] : part == 1 ? out.bias[1] : out.bias[2];
  const long long at = (long long)m * N + n;
  float add_bias = 0.f, add_residual = 0.f;
  if (writes && bias != nullptr) add_bias = bias[n];
  if (writes && out.residual != nullptr) add_residual = out.residual[at];

  f32x4 acc[kG];
#pragma unroll
  for (int g = 0; g < kG; ++g) acc[g] = zero;
  for (int s0 = wave; s0 < nStrips; s0 += kStrips * kW) {
    if (s0 != wave) load_batch(s0);
#pragma unroll
    for (int u = 0; u < kStrips; ++u) {
      const int k = 64 * (s0 + u * kW) + 4 * b, kk = k < K ? k : 0;
      const f32x4 wu = k < K ? wv[u] : zero;
#pragma unroll
      for (int g = 0; g < kG; ++g) {
        f32x4 xu;
        if constexpr (kV > 0)
          xu = *reinterpret_cast<const f32x4*>(xs + col[g] * (K + kNormPad) + kk);
        else
          xu = xv[u][g];
        if (k >= K) xu = zero;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          acc[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(wu[e], xu[e], acc[g], 0, 0, 0);
      }
    }
  }

  // The 16 blocks of the wave (lanes 4 apart), then the waves.
#pragma unroll
  for (int g = 0; g < kG; ++g)
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const float v = block_sum(acc[g][c]);
      if (lane < 4) red[wave][g][c][lane] = v;
    }
  __syncthreads();
  if (!writes) return;
  float v = 0.f;
#pragma unroll
  for (int ww = 0; ww < kW; ++ww) v += red[ww][m / 4][r][m % 4];
  v += add_bias;
  if (kGelu) v = gelu(v);
  Y* y = static_cast<Y*>(part == 0 ? out.y[0] : part == 1 ? out.y[1] : out.y[2]);
  y[at] = (Y)(v + add_residual);
}

// ---------------------------------------------------------------------------------------
// Host side.

static bool misaligned(const void* p) { return ((uintptr_t)p & 15u) != 0; }

static int launched() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TFGFA_OK : -(int)e;
}

template <int kV, typename Y>
static void launch_norm(const float* x, const __bf16* delta, float* sum, const float* scale,
                        const float* shift, Y* y, long long rows, int d, float eps,
                        hipStream_t stream) {
  const dim3 grid((unsigned)rows), block(64);
  if (delta != nullptr)
    hipLaunchKernelGGL((layernorm_kernel<kV, true, Y>), grid, block, 0, stream, x, delta, sum,
                       scale, shift, y, d, eps);
  else
    hipLaunchKernelGGL((layernorm_kernel<kV, false, Y>), grid, block, 0, stream, x, delta, sum,
                       scale, shift, y, d, eps);
}

struct RowsArgs {
  const void* x;
  const float* ln_scale;
  const float* ln_shift;
  const float* w[kMaxParts];
  int M, N, K, tiles;
  RowsOut out;
};

template <int kW, int kStrips, int kG, typename X, typename Y, int kV, bool kGelu = false>
static void launch_rows(const RowsArgs& a, int parts, hipStream_t stream) {
  const size_t lds = kV ? (size_t)a.M * (a.K + kNormPad) * sizeof(float) : 0;
  hipLaunchKernelGGL((linear_rows_kernel<kW, kStrips, kG, X, Y, kV, kGelu>),
                     dim3((unsigned)(a.tiles * parts)), dim3(64 * kW), lds, stream, a.x, a.w[0],
                     a.w[1], a.w[2], a.M, a.N, a.K, a.tiles, a.ln_scale, a.ln_shift, a.out);
}

// With the norm: 4 waves (more would idle through the norm of 4 rows), the whole width in one
// batch.
template <int kG, typename Y, bool kGelu>
static void launch_rows_norm(const RowsArgs& a, int parts, hipStream_t stream) {
  if (a.K <= 1024)
    launch_rows<kNormWaves, 4, kG, float, Y, 4, kGelu>(a, parts, stream);
  else
    launch_rows<kNormWaves, 8, kG, float, Y, 8, kGelu>(a, parts, stream);
}

// Without: the fewest waves and strips that take the width in one batch, up to 8192; wider ones
// loop.
template <int kG, typename X>
static void launch_rows_plain(const RowsArgs& a, int parts, hipStream_t stream) {
  if (a.K <= 1024)
    launch_rows<8, 2, kG, X, float, 0>(a, parts, stream);
  else if (a.K <= 2048)
    launch_rows<8, 4, kG, X, float, 0>(a, parts, stream);
  else if (a.K <= 4096)
    launch_rows<8, 8, kG, X, float, 0>(a, parts, stream);
  else
    launch_rows<16, 8, kG, X, float, 0>(a, parts, stream);
}

template <int kG>
static void launch_rows_types(const RowsArgs& a, int parts, bool x_bf16, bool y_bf16, bool ln,
                              bool gelu, hipStream_t stream) {
  if (ln && gelu)
    launch_rows_norm<kG, float, true>(a, parts, stream);
  else if (ln && y_bf16)
    launch_rows_norm<kG, __bf16, false>(a, parts, stream);
  else if (ln)
    launch_rows_norm<kG, float, false>(a, parts, stream);
  else if (x_bf16)
    launch_rows_plain<kG, __bf16>(a, parts, stream);
  else
    launch_rows_plain<kG, float>(a, parts, stream);
}

}  // namespace tfgpt2

extern "C" int tfgpt2_layernorm(const float* x, const void* delta, float* sum, const float* scale,
                                const float* shift, void* y, int y_bf16, int64_t rows, int d,
                                float eps, void* hip_stream) {
  using namespace tfgpt2;
  if (rows < 0 || d < 4 || d > TFGPT2_MAX_NORM_DIM || (d & 3)) return TFGFA_ERR_BAD_SHAPE;
  if (y_bf16 != 0 && y_bf16 != 1) return TFGFA_ERR_DTYPE;
  if (rows == 0) return TFGFA_OK;
  if (rows > INT32_MAX) return TFGFA_ERR_TOO_LARGE;
  if (!x || !scale || !shift || !y || (delta != nullptr && sum == nullptr)) return TFGFA_ERR_NULL_POINTER;
  if (misaligned(x) || misaligned(delta) || misaligned(sum) || misaligned(scale) ||
      misaligned(shift) || misaligned(y))
    return TFGFA_ERR_ALIGNMENT;
  const __bf16* dl = static_cast<const __bf16*>(delta);
  const hipStream_t stream = (hipStream_t)hip_stream;
  if (d <= 1024) {
    if (y_bf16)
      launch_norm<4>(x, dl, sum, scale, shift, static_cast<__bf16*>(y), rows, d, eps, stream);
    else
      launch_norm<4>(x, dl, sum, scale, shift, static_cast<float*>(y), rows, d, eps, stream);
  } else {
    if (y_bf16)
      launch_norm<8>(x, dl, sum, scale, shift, static_cast<__bf16*>(y), rows, d, eps, stream);
    else
      launch_norm<8>(x, dl, sum, scale, shift, static_cast<float*>(y), rows, d, eps, stream);
  }
  return launched();
}

extern "C" int tfgpt2_gelu(const float* x, float* y, int64_t n, void* hip_stream) {
  using namespace tfgpt2;
  if (n < 0) return TFGFA_ERR_BAD_SHAPE;
  if (n == 0) return TFGFA_OK;
  const long long blocks = (n + 4LL * kGeluThreads - 1) / (4LL * kGeluThreads);
  if (blocks > INT32_MAX) return TFGFA_ERR_TOO_LARGE;
  if (!x || !y) return TFGFA_ERR_NULL_POINTER;
  if (misaligned(x) || misaligned(y)) return TFGFA_ERR_ALIGNMENT;
  hipLaunchKernelGGL(gelu_kernel, dim3((unsigned)blocks), dim3(kGeluThreads), 0,
                     (hipStream_t)hip_stream, x, y, (long long)n);
  return launched();
}

extern "C" int tfgpt2_cast_bf16(int count, const float* const* src, void* const* dst,
                                const int64_t* n, void* hip_stream) {
  using namespace tfgpt2;
  if (count < 0 || count > kMaxCasts) return TFGFA_ERR_BAD_SHAPE;
  if (count > 0 && (!src || !dst || !n)) return TFGFA_ERR_NULL_POINTER;
  Casts a = {};
  long long units = 0;
  for (int i = 0; i < count; ++i) {
    if (n[i] < 0 || (n[i] & 3)) return TFGFA_ERR_BAD_SHAPE;
    if (n[i] > 0 && (!src[i] || !dst[i])) return TFGFA_ERR_NULL_POINTER;
    if (misaligned(src[i]) || misaligned(dst[i])) return TFGFA_ERR_ALIGNMENT;
    units += n[i] / 4;
    a.src[i] = src[i];
    a.dst[i] = static_cast<__bf16*>(dst[i]);
    a.end[i] = units;
  }
  a.count = count;
  const long long blocks = (units + kCastThreads - 1) / kCastThreads;
  if (blocks > INT32_MAX) return TFGFA_ERR_TOO_LARGE;
  if (blocks == 0) return TFGFA_OK;
  hipLaunchKernelGGL(cast_kernel, dim3((unsigned)blocks), dim3(kCastThreads), 0,
                     (hipStream_t)hip_stream, a);
  return launched();
}

extern "C" int tfgpt2_linear_rows(const void* x, int x_bf16, const float* ln_scale,
                                  const float* ln_shift, float eps, int parts,
                                  const float* const* w, const float* const* bias, int gelu,
                                  const float* residual, void* const* y, int y_bf16, int M, int N,
                                  int K, void* hip_stream) {
  using namespace tfgpt2;
  if (M < 0 || M > TFGPT2_MAX_ROWS || N < 1 || K < 4 || (K & 3) || parts < 1 || parts > kMaxParts)
    return TFGFA_ERR_BAD_SHAPE;
  if ((x_bf16 != 0 && x_bf16 != 1) || (y_bf16 != 0 && y_bf16 != 1) || (gelu != 0 && gelu != 1))
    return TFGFA_ERR_DTYPE;
  const bool ln = ln_scale != nullptr;
  if (ln != (ln_shift != nullptr)) return TFGFA_ERR_NULL_POINTER;
  if (ln && (x_bf16 || K > TFGPT2_MAX_NORM_DIM || (long long)M * (K + kNormPad) > kNormLdsFloats))
    return TFGFA_ERR_BAD_SHAPE;
  if (residual != nullptr && parts != 1) return TFGFA_ERR_BAD_SHAPE;
  if ((y_bf16 && (!ln || gelu)) || (gelu && !ln)) return TFGFA_ERR_DTYPE;
  if (M == 0) return TFGFA_OK;
  const long long tiles = ((long long)N + kTileRows - 1) / kTileRows;
  if (tiles * parts > INT32_MAX) return TFGFA_ERR_TOO_LARGE;
  if (!x || !w || !bias || !y) return TFGFA_ERR_NULL_POINTER;
  RowsArgs a = {};
  for (int p = 0; p < parts; ++p) {
    if (!w[p] || !y[p]) return TFGFA_ERR_NULL_POINTER;
    if (misaligned(w[p]) || misaligned(bias[p]) || misaligned(y[p])) return TFGFA_ERR_ALIGNMENT;
    a.w[p] = w[p];
    a.out.bias[p] = bias[p];
    a.out.y[p] = y[p];
  }
  if (misaligned(x) || misaligned(ln_scale) || misaligned(ln_shift) || misaligned(residual))
    return TFGFA_ERR_ALIGNMENT;
  a.x = x;
  a.ln_scale = ln_scale;
  a.ln_shift = ln_shift;
  a.out.residual = residual;
  a.out.eps = eps;
  a.M = M;
  a.N = N;
  a.K = K;
  a.tiles = (int)tiles;
  const hipStream_t stream = (hipStream_t)hip_stream;
  if (M <= 4)
    launch_rows_types<1>(a, parts, x_bf16 != 0, y_bf16 != 0, ln, gelu != 0, stream);
  else
    launch_rows_types<2>(a, parts, x_bf16 != 0, y_bf16 != 0, ln, gelu != 0, stream);
  return launched();
}
