// tfgfa_gpt2.hip - the GPT-2 block around the attention, MI355X (gfx950).
//
// The reference's block (src/py/model_inference.py:96-164) spells its LayerNorm, GELU and
// residual adds out as elementwise operators; each is then a pass over memory of its own, and a
// decode step of a few rows is some 45 launches per layer.  Here:
//   layernorm_kernel    LayerNorm of a row held in one wave's registers, with the residual add
//                       before it and the rounding to bf16 after it where the caller has them;
//   gelu_kernel         the tanh GELU in one pass.
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

// Sum over the 64 lanes, in every lane.
template <int kCtrl>
__device__ __forceinline__ float dpp_add(float x) {
  return x + __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(x), kCtrl, 0xF, 0xF, false));
}
__device__ __forceinline__ float wave_sum(float x) {
  x = dpp_add<0xB1>(x);   // quad: lanes 1 apart
  x = dpp_add<0x4E>(x);   // quad: lanes 2 apart
  x = dpp_add<0x124>(x);  // row of 16: rotated by 4
  x = dpp_add<0x128>(x);  // row of 16: rotated by 8
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  x = __uint_as_float(r[0]) + __uint_as_float(r[1]);  // rows 0 and 1, rows 2 and 3
  const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return __uint_as_float(q[0]) + __uint_as_float(q[1]);
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
