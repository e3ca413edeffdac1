// tfgfa_gpt2.hip - the GPT-2 block around the attention, MI355X (gfx950).
//
// The reference's block (src/py/model_inference.py:96-164) spells its LayerNorm, GELU and
// residual adds out as elementwise operators; each is then a pass over memory of its own, and a
// decode step of a few rows is some 45 launches per layer.  Here:
//   layernorm_kernel    LayerNorm of a row held in one wave's registers, with the residual add
//                       before it and the rounding to bf16 after it where the caller has them;
//   gelu_kernel         the tanh GELU in one pass;
//   cast_kernel         float32 -> bf16 copies of several weights in one launch;
//   linear_planes_kernel  the MLP's float32 linears on the bf16 matrix units, from exact three-way
//                       splits of both operands;
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
#include "tfgfa_device.h"
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

// A float32 value as three bf16 ones that add up to it exactly: itself rounded to bf16 (8 significant
// bits), the remainder (at most 2^-9 of it, 16 bits) rounded, and the rest (at most 2^-18, 8 bits).  An
// infinity or a NaN stays the first, the others are NaN then.  A finite value that rounds to infinity
// (the top 2^-9 of the float range) has no such split: store_planes truncates it instead (a remainder
// of 16 bits is left all the same), a weight's gives NaN, and plain_sums what the NaN stands for.
// top_pair: two values rounded, packed; drop_lo, drop_hi: what the first and the second leave.
__device__ __forceinline__ uint32_t top_pair(float a, float b) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ float drop_lo(float a, uint32_t top) { return a - __uint_as_float(top << 16); }
__device__ __forceinline__ float drop_hi(float b, uint32_t top) {
  return b - __uint_as_float(top & 0xffff0000u);
}
// Four values into the three planes of a (3, rows, width) array, `plane` elements apart.
__device__ __forceinline__ void store_planes(__bf16* y, long long plane, f32x4 v) {
  typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
#pragma unroll
  for (int p = 0; p < 3; ++p) {
    u32x2 top = {top_pair(v[0], v[1]), top_pair(v[2], v[3])};
    if (p == 0) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const uint32_t bits = __float_as_uint(v[e]), high = (e & 1) ? 0xffff0000u : 0x0000ffffu;
        if ((bits & 0x7fff8000u) == 0x7f7f8000u)  // finite, half a unit or more above bf16's largest
          top[e >> 1] = (top[e >> 1] & ~high) | ((e & 1) ? bits & 0xffff0000u : bits >> 16);
      }
    }
    *reinterpret_cast<u32x2*>(y + p * plane) = top;
    v = f32x4{drop_lo(v[0], top[0]), drop_hi(v[1], top[0]), drop_lo(v[2], top[1]), drop_hi(v[3], top[1])};
  }
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
//   scale and shift loaded where used: 7.2 and 9.3), 6.7 with the residual into planes; the operators
//   they stand for: about 32 us a norm, and 86 us for the mixed bf16 + float32 add before the second.
enum { kOutF32 = 0, kOutBf16 = 1, kOutPlanes = 2 };

template <int kV, bool kDelta, int kOut>
__global__ __launch_bounds__(64) void layernorm_kernel(
    const float* x, const __bf16* __restrict__ delta, float* sum, const float* __restrict__ scale,
    const float* __restrict__ shift, void* __restrict__ y, int d, float eps) {
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
    if (c >= d) continue;
    const f32x4 o = v[i] * g[i] + h[i];
    if (kOut == kOutF32)
      store4(static_cast<float*>(y) + base + c, o);
    else if (kOut == kOutBf16)
      store4(static_cast<__bf16*>(y) + base + c, o);
    else
      store_planes(static_cast<__bf16*>(y) + base + c, (long long)gridDim.x * d, o);
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
// The MLP's float32 linears: y = x w^T + bias for many rows.
//
// Bound: the matrix units.  The float32 MFMA peaks at 157 TFLOP/s (a library GEMM reaches 110-139 of
// it), the bf16 one at 16 times that.  A float32 value is the exact sum of three bf16 values, so a
// product of two is nine bf16 products; the six larger ones are computed (smallest first, float32
// accumulation), the other three are below 2^-26 of the product, less than float32 rounds it by.
// The largest of the six has sums of its own, rounded once per 16 of the contraction (the float32
// GEMM: once per 4), so the result is closer to float64's than the float32 GEMM's: 613 x 1600 -> 6400
// 2.4e-7 (7.1e-7), 613 x 6400 -> 1600 2.8e-7 (1.4e-6), 100 x 3072 -> 768 1.4e-7 (5.0e-7).
// x arrives as three planes, written so by the kernels that produce it; the weights are split in
// registers, 5.5 VALU instructions a value.  A workgroup of 8 waves (2 a SIMD: one wave's splits
// overlap the other's MFMAs) computes 128 rows x 128 outputs, a wave 64 x 32: 12 MFMAs for 12 split
// steps per 16 of the contraction.  Steps of 32 stream into a ring of three 40-KiB slots by direct
// buffer -> LDS loads (24 KiB of planes, 64-B rows with chunk c of row r at c ^ ((r >> 2) & 3); 16 KiB
// of weights, 128-B rows swizzled as swz_k), one barrier a step.
// A grid that leaves CUs idle splits the contraction into S partial sums (choose_k_splits), added in
// order by reduce_kernel.
//   us, with bias (float32 library GEMM): 613 x 1600 -> 6400 82 (114), 613 x 6400 -> 1600 S = 3 86
//   (104), 1000 x 1024 -> 4096 51 (68), 1000 x 4096 -> 1024 S = 4 55 (68), 4096 x 4096 -> 1024 205 (247).
//   Both operands split in registers, 4 waves of 64 x 64 (613 x 1600 -> 6400): 97, 87 with the splits
//   spread between the MFMAs; a single wave a SIMD does not overlap the two.
using tfgfa::head_desc;
using tfgfa::lds_addr;
using tfgfa::lds_transfer;
using tfgfa::swz_k;
using tfgfa::wait_vmcnt;
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef tfgfa::i32x4 i32x4;

// The descriptor moved on by `bytes` (within its rows), the range still ending at the same address.
__device__ __forceinline__ i32x4 advance(i32x4 desc, int bytes) {
  const uint64_t base = ((uint64_t)(uint32_t)desc[1] << 32 | (uint32_t)desc[0]) + (uint32_t)bytes;
  i32x4 d;
  d[0] = (int)(uint32_t)base;
  d[1] = (int)(uint32_t)(base >> 32);
  d[2] = desc[2] - bytes;
  d[3] = desc[3];
  return d;
}

// Four outputs n.. of row m over the contraction's k0..k1 with the products in float32.  Infinities in
// x or w, weights at the top of the float range and overflow meet NaN in the split products where a
// float32 GEMM need not (inf - inf, inf * 0), and a product of first pieces that were rounded up is
// infinite where the float32 one is within 2^-8 of the range's top, so a sum that is not finite is
// computed again; ordinary values never are.
// Ends early where all four are NaN in float32 too (a NaN in x, or in every weight row).
__device__ __forceinline__ f32x4 plain_sums(const __bf16* X, const float* W, int M, int K, int m, int n,
                                            int k0, int k1) {
  f32x4 s = {0.f, 0.f, 0.f, 0.f};
#pragma unroll 1
  for (int k = k0; k < k1; k += 4) {
    f32x4 x = load4(X + (long long)m * K + k);
    const f32x4 x1 = load4(X + ((long long)M + m) * K + k), x2 = load4(X + (2LL * M + m) * K + k);
#pragma unroll
    for (int e = 0; e < 4; ++e)
      if (__builtin_isfinite(x[e])) x[e] += x1[e] + x2[e];
#pragma unroll
    for (int o = 0; o < 4; ++o) {
      const f32x4 w = load4(W + (long long)(n + o) * K + k);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[o] = fmaf(x[e], w[e], s[o]);
    }
    if (__builtin_isnan(s[0]) && __builtin_isnan(s[1]) && __builtin_isnan(s[2]) && __builtin_isnan(s[3])) break;
  }
  return s;
}

constexpr int kTile = 128;  // rows and outputs per workgroup
constexpr int kXBytes = 24 * 1024, kStage = 40 * 1024, kStages = 3;
// What is written: a split's sums; GELU(sums + bias) as planes; sums + bias + residual.
enum { kPartial = 0, kGeluPlanes = 1, kFinal = 2 };

template <int kMode>
__global__ __launch_bounds__(512, 2) void linear_planes_kernel(
    const __bf16* __restrict__ X, const float* __restrict__ W, int M, int N, int K, int tm, int tn,
    int S, int steps, const float* __restrict__ bias, const float* __restrict__ residual,
    void* __restrict__ Yv) {
  __shared__ __attribute__((aligned(1024))) unsigned char ring[kStages * kStage];
  // Workgroups are dealt to the 8 XCDs round-robin: each XCD gets a run of consecutive tiles, row
  // tiles fastest, so the row tiles of one weight tile read it through one L2.
  const int T = tm * tn * S, per = (T + 7) / 8;
  const int t = (blockIdx.x % 8) * per + blockIdx.x / 8;
  if (t >= T) return;
  const int mt = t % tm, nt = t / tm % tn, z = t / (tm * tn);
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wr = wave & 1, wc = wave >> 1;
  const int m0 = mt * 128, n0 = nt * 128;
  const int s0 = z * steps, ns = min(steps, K / 32 - s0);  // this split's steps (at least one)
  // Rows past M of a plane read the next plane's or, past the last, zero; weight rows past N read
  // zero.  None of their sums are stored.
  const i32x4 xd = advance(head_desc(X + (long long)m0 * K, 3 * M - m0, K * 2), s0 * 64);
  const i32x4 wd = advance(head_desc(W + (long long)n0 * K, N - n0, K * 4), s0 * 128);
  int xo[3], wo[2];  // this wave's 3 of the 24 X transfers (plane, 16 rows) and 2 of the 16 W ones (8 rows)
#pragma unroll
  for (int i = 0; i < 3; ++i) {
    const int blk = 3 * wave + i, row = 16 * (blk & 7) + (lane >> 2);
    xo[i] = ((blk >> 3) * M + row) * K * 2 + (((lane & 3) ^ ((row >> 2) & 3)) << 4);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = 8 * (2 * wave + i) + (lane >> 3);
    wo[i] = row * K * 4 + (((lane & 7) ^ swz_k(row)) << 4);
  }
  auto issue = [&](int s, int slot) {
    unsigned char* dst = ring + slot * kStage;
    const i32x4 x = advance(xd, s * 64), w = advance(wd, s * 128);
#pragma unroll
    for (int i = 0; i < 3; ++i) lds_transfer(x, lds_addr(dst + (3 * wave + i) * 1024), xo[i]);
#pragma unroll
    for (int i = 0; i < 2; ++i) lds_transfer(w, lds_addr(dst + kXBytes + (2 * wave + i) * 1024), wo[i]);
  };
  const int r = lane & 31, h = lane >> 5;
  int fx[2], fw[2][2];
#pragma unroll
  for (int c = 0; c < 2; ++c) {
    fx[c] = (64 * wr + r) * 64 + (((2 * c + h) ^ ((r >> 2) & 3)) << 4);
#pragma unroll
    for (int e = 0; e < 2; ++e) fw[c][e] = kXBytes + (32 * wc + r) * 128 + (((4 * c + 2 * h + e) ^ swz_k(r)) << 4);
  }
  // The largest product's sums and the five small ones' apart: the small ones' roundings are then
  // 2^-8 of the large ones', which come once per 16 of the contraction.
  f32x16 acc[2], low[2];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[b][e] = low[b][e] = 0.f;
  typedef f32x4 Raw[2];
  auto read_w = [&](Raw& q, int slot, int c, int e) { q[e] = *reinterpret_cast<const f32x4*>(ring + slot * kStage + fw[c][e]); };
  auto read_x = [&](u32x4 (&q)[2][3], int slot, int c, int k) {  // k: 0..5 = plane * 2 + tile
    const int p = k >> 1, b = k & 1;
    q[b][p] = *reinterpret_cast<const u32x4*>(ring + slot * kStage + p * 8192 + b * 2048 + fx[c]);
  };
  auto split_step = [&](u32x4 (&o)[3], Raw& q, int k) {  // 12 steps: pair k / 3, plane k % 3
    const int pair = k / 3, pl = k % 3, e = pair >> 1, c = 2 * (pair & 1);
    const float x0 = q[e][c], x1 = q[e][c + 1];
    uint32_t v = top_pair(x0, x1);
    asm volatile("" : "+v"(v));
    o[pl][pair] = v;
    if (pl < 2) {
      float r0 = drop_lo(x0, v), r1 = drop_hi(x1, v);
      asm volatile("" : "+v"(r0), "+v"(r1));
      q[e][c] = r0;
      q[e][c + 1] = r1;
    }
  };
  // MFMA i of 12: the six products, smallest first, of the two row tiles.
  auto mma = [&](const u32x4 (&w)[3], const u32x4 (&x)[2][3], int i) {
    constexpr int pw[6] = {2, 0, 1, 1, 0, 0}, px[6] = {0, 2, 1, 0, 1, 0};
    const int p = i >> 1, b = i & 1;
    f32x16& sum = p == 5 ? acc[b] : low[b];
    sum = __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, w[pw[p]]),
                                                  __builtin_bit_cast(bf16x8, x[b][px[p]]), sum, 0, 0, 0);
  };
  // Waits for this wave's loads of a step, `ahead` later steps of 5 loads staying in flight, and for
  // its LDS reads; then for the other waves.
  auto sync = [&](int ahead) {
    if (ahead >= 2)
      wait_vmcnt<10>();
    else if (ahead == 1)
      wait_vmcnt<5>();
    else
      wait_vmcnt<0>();
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  issue(0, 0);
  if (ns > 1) issue(1, 1);
  if (ns > 2) issue(2, 2);
  u32x4 XA[2][3], XB[2][3], WA[3], WB[3];
  Raw R0, R1;
  sync(min(ns - 1, 2));
#pragma unroll
  for (int e = 0; e < 2; ++e) { read_w(R0, 0, 0, e); read_w(R1, 0, 1, e); }
#pragma unroll
  for (int k = 0; k < 6; ++k) read_x(XA, 0, 0, k);
#pragma unroll
  for (int k = 0; k < 12; ++k) split_step(WA, R0, k);
  int slot = 0;
  for (int s = 0; s < ns; ++s) {
    // Chunk 0 (16 of the step's 32), beside the split of chunk 1's weights.
#pragma unroll
    for (int i = 0; i < 12; ++i) {
      mma(WA, XA, i);
      if (i < 6) read_x(XB, slot, 1, i);
      split_step(WB, R1, i);
      __builtin_amdgcn_sched_barrier(0);
    }
    const int next = slot == 2 ? 0 : slot + 1;
    // Step s + 1 has landed in every wave's share, and every read of step s is complete: its slot
    // takes step s + 3.  (After the last step the reads below get an old slot's values: unused.)
    if (s + 1 < ns) {
      sync(min(ns - 2 - s, 1));
      if (s + 3 < ns) issue(s + 3, slot);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int e = 0; e < 2; ++e) read_w(R0, next, 0, e);
#pragma unroll
    for (int i = 0; i < 12; ++i) {
      mma(WB, XB, i);
      if (i < 6) read_x(XA, next, 0, i);
      if (i >= 3)
#pragma unroll
        for (int k = 12 * (i - 3) / 9; k < 12 * (i - 2) / 9; ++k) split_step(WA, R0, k);
      if (i >= 8 && i < 10) read_w(R1, next, 1, i - 8);
      __builtin_amdgcn_sched_barrier(0);
    }
    slot = next;
  }
#pragma unroll
  for (int b = 0; b < 2; ++b) {
    const int m = m0 + 64 * wr + 32 * b + r;
    if (m >= M) continue;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int n = n0 + 32 * wc + 8 * g + 4 * h;
      if (n >= N) continue;
      f32x4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = acc[b][4 * g + e] + low[b][4 * g + e];
      if (!__builtin_isfinite((v[0] + v[1]) + (v[2] + v[3])))  // (also of four large ones: the same again)
        v = plain_sums(X, W, M, K, m, n, s0 * 32, (s0 + ns) * 32);
      if (kMode != kPartial && bias != nullptr) v += load4(bias + n);
      if (kMode == kGeluPlanes) {
        store_planes(static_cast<__bf16*>(Yv) + (long long)m * N + n, (long long)M * N,
                     f32x4{gelu(v[0]), gelu(v[1]), gelu(v[2]), gelu(v[3])});
      } else {
        const long long at = ((long long)z * M + m) * N + n;
        if (kMode == kFinal && residual != nullptr) v += load4(residual + at);
        store4(static_cast<float*>(Yv) + at, v);
      }
    }
  }
}
// y = sum of the S partial sums, + bias, then GELU into planes, or + residual.  Bound: memory.
template <int kMode>
__global__ __launch_bounds__(256) void reduce_kernel(const float* __restrict__ part, int S, long long MN,
                                                     int N, const float* __restrict__ bias,
                                                     const float* __restrict__ residual,
                                                     void* __restrict__ y) {
  const long long i = ((long long)blockIdx.x * 256 + threadIdx.x) * 4;
  if (i >= MN) return;
  f32x4 v = load4(part + i);
  for (int z = 1; z < S; ++z) v += load4(part + z * MN + i);
  if (bias != nullptr) v += load4(bias + i % N);
  if (kMode == kGeluPlanes) {
    store_planes(static_cast<__bf16*>(y) + i, MN, f32x4{gelu(v[0]), gelu(v[1]), gelu(v[2]), gelu(v[3])});
  } else {
    if (residual != nullptr) v += load4(residual + i);
    store4(static_cast<float*>(y) + i, v);
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

// A launch of `blocks` workgroups of `threads` threads is past HIP's limit: 2^32 - 1 threads.
static bool too_many(long long blocks, int threads) { return blocks > (long long)UINT32_MAX / threads; }

static int launched() {
  const hipError_t e = hipGetLastError();
  return e == hipSuccess ? TFGFA_OK : -(int)e;
}

template <int kV, int kOut>
static void launch_norm(const float* x, const __bf16* delta, float* sum, const float* scale,
                        const float* shift, void* y, long long rows, int d, float eps,
                        hipStream_t stream) {
  const dim3 grid((unsigned)rows), block(64);
  if (delta != nullptr)
    hipLaunchKernelGGL((layernorm_kernel<kV, true, kOut>), grid, block, 0, stream, x, delta, sum,
                       scale, shift, y, d, eps);
  else
    hipLaunchKernelGGL((layernorm_kernel<kV, false, kOut>), grid, block, 0, stream, x, delta, sum,
                       scale, shift, y, d, eps);
}

template <int kV>
static void launch_norm_out(const float* x, const __bf16* delta, float* sum, const float* scale,
                            const float* shift, void* y, int out, long long rows, int d, float eps,
                            hipStream_t stream) {
  if (out == kOutF32)
    launch_norm<kV, kOutF32>(x, delta, sum, scale, shift, y, rows, d, eps, stream);
  else if (out == kOutBf16)
    launch_norm<kV, kOutBf16>(x, delta, sum, scale, shift, y, rows, d, eps, stream);
  else
    launch_norm<kV, kOutPlanes>(x, delta, sum, scale, shift, y, rows, d, eps, stream);
}

// Splits of the contraction: the fewest rounds of workgroups (one per CU) times steps, counting a
// split's partial sums as the steps that writing and adding them take.
static int choose_k_splits(long long tiles, int steps, int cu_count) {
  int best = 1;
  long long best_cost = 0;
  for (int s = 1; s <= TFGPT2_MAX_K_SPLITS && (s == 1 || steps / s >= 8); ++s) {
    const long long rounds = (tiles * s + cu_count - 1) / cu_count;
    const long long cost = rounds * ((steps + s - 1) / s + 4) + (s > 1 ? 6 + 2 * s : 0);
    if (s == 1 || cost < best_cost) {
      best = s;
      best_cost = cost;
    }
  }
  return best;
}

// Either launch of a linear on planes is past HIP's limit.
static bool planes_too_large(long long tiles, int M, int N, int S) {
  return too_many((tiles * S + 7) / 8 * 8, 512) ||
         (S > 1 && too_many(((long long)M * N / 4 + 255) / 256, 256));
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
static int plain_waves(int K) { return K <= 4096 ? 8 : 16; }
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
                                const float* shift, void* y, int y_kind, int64_t rows, int d,
                                float eps, void* hip_stream) {
  using namespace tfgpt2;
  if (rows < 0 || d < 4 || d > TFGPT2_MAX_NORM_DIM || (d & 3)) return TFGFA_ERR_BAD_SHAPE;
  if (y_kind < TFGPT2_F32 || y_kind > TFGPT2_PLANES) return TFGFA_ERR_DTYPE;
  if (rows == 0) return TFGFA_OK;
  if (too_many(rows, 64)) return TFGFA_ERR_TOO_LARGE;
  if (!x || !scale || !shift || !y || (delta != nullptr && sum == nullptr)) return TFGFA_ERR_NULL_POINTER;
  if (misaligned(x) || misaligned(delta) || misaligned(sum) || misaligned(scale) ||
      misaligned(shift) || misaligned(y))
    return TFGFA_ERR_ALIGNMENT;
  const __bf16* dl = static_cast<const __bf16*>(delta);
  const hipStream_t stream = (hipStream_t)hip_stream;
  if (d <= 1024)
    launch_norm_out<4>(x, dl, sum, scale, shift, y, y_kind, rows, d, eps, stream);
  else
    launch_norm_out<8>(x, dl, sum, scale, shift, y, y_kind, rows, d, eps, stream);
  return launched();
}

extern "C" int tfgpt2_gelu(const float* x, float* y, int64_t n, void* hip_stream) {
  using namespace tfgpt2;
  if (n < 0) return TFGFA_ERR_BAD_SHAPE;
  if (n == 0) return TFGFA_OK;
  const long long blocks = (n + 4LL * kGeluThreads - 1) / (4LL * kGeluThreads);
  if (too_many(blocks, kGeluThreads)) return TFGFA_ERR_TOO_LARGE;
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
  if (too_many(blocks, kCastThreads)) return TFGFA_ERR_TOO_LARGE;
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
  if (too_many(tiles * parts, 64 * (ln ? kNormWaves : plain_waves(K)))) return TFGFA_ERR_TOO_LARGE;
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

extern "C" int tfgpt2_linear_planes_splits(int M, int N, int K, int cu_count) {
  using namespace tfgpt2;
  if (M < 1 || N < 4 || (N & 3) || K < 32 || K % 32 || cu_count < 1) return 0;
  if (3LL * M * K * 2 > INT32_MAX || (long long)N * K * 4 > INT32_MAX) return 0;
  const long long tiles = (((long long)M + kTile - 1) / kTile) * (((long long)N + kTile - 1) / kTile);
  const int S = choose_k_splits(tiles, K / 32, cu_count);
  if (planes_too_large(tiles, M, N, S)) return planes_too_large(tiles, M, N, 1) ? 0 : 1;
  return S;
}

extern "C" int tfgpt2_linear_planes(const void* x, const float* w, const float* bias, int gelu_planes,
                                    const float* residual, void* y, float* part, int splits, int M,
                                    int N, int K, void* hip_stream) {
  using namespace tfgpt2;
  if (gelu_planes != 0 && gelu_planes != 1) return TFGFA_ERR_DTYPE;
  if (M == 0 && N > 0 && K > 0) return TFGFA_OK;
  if (tfgpt2_linear_planes_splits(M, N, K, 1) == 0) return TFGFA_ERR_BAD_SHAPE;
  if (splits < 1 || splits > TFGPT2_MAX_K_SPLITS || splits > K / 32 || (gelu_planes && residual))
    return TFGFA_ERR_BAD_SHAPE;
  if (!x || !w || !y || (splits > 1 && part == nullptr)) return TFGFA_ERR_NULL_POINTER;
  if (misaligned(x) || misaligned(w) || misaligned(bias) || misaligned(residual) || misaligned(y) ||
      misaligned(part))
    return TFGFA_ERR_ALIGNMENT;
  const int tm = ((long long)M + kTile - 1) / kTile, tn = ((long long)N + kTile - 1) / kTile;
  const int steps = (K / 32 + splits - 1) / splits;
  const int S = (K / 32 + steps - 1) / steps;  // no split without a step
  if (planes_too_large((long long)tm * tn, M, N, S)) return TFGFA_ERR_TOO_LARGE;
  const dim3 grid((unsigned)((tm * tn * S + 7) / 8 * 8));
  const hipStream_t stream = (hipStream_t)hip_stream;
  const __bf16* xp = static_cast<const __bf16*>(x);
  if (S == 1) {
    if (gelu_planes)
      hipLaunchKernelGGL(linear_planes_kernel<kGeluPlanes>, grid, dim3(512), 0, stream, xp, w, M, N,
                         K, tm, tn, 1, steps, bias, residual, y);
    else
      hipLaunchKernelGGL(linear_planes_kernel<kFinal>, grid, dim3(512), 0, stream, xp, w, M, N, K, tm,
                         tn, 1, steps, bias, residual, y);
    return launched();
  }
  hipLaunchKernelGGL(linear_planes_kernel<kPartial>, grid, dim3(512), 0, stream, xp, w, M, N, K, tm,
                     tn, S, steps, bias, residual, static_cast<void*>(part));
  const long long MN = (long long)M * N;
  const dim3 rgrid((unsigned)((MN / 4 + 255) / 256));
  if (gelu_planes)
    hipLaunchKernelGGL(reduce_kernel<kGeluPlanes>, rgrid, dim3(256), 0, stream, part, S, MN, N, bias,
                       residual, y);
  else
    hipLaunchKernelGGL(reduce_kernel<kFinal>, rgrid, dim3(256), 0, stream, part, S, MN, N, bias,
                       residual, y);
  return launched();
}
