// Shared device helpers for the gfx950 kernels: storage types, wavefront reductions, error codes.
//
// Every kernel entry point is `extern "C"`, takes raw device pointers and a hipStream_t and
// returns 0 or one of the TS_ERR_* codes; shapes are validated on the host before any launch.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#define TS_OK 0
#define TS_ERR_DTYPE 1     // dtype code is not one of TS_F32 / TS_BF16
#define TS_ERR_SHAPE 2     // a size the kernel does not take
#define TS_ERR_LAUNCH 3    // hipGetLastError() after the launch was not hipSuccess
#define TS_ERR_ARG 4       // null pointer or inconsistent arguments

#define TS_F32 0
#define TS_BF16 1

#define TS_WAVE 64

// bfloat16 as raw bits; one conversion everywhere: the instruction's (round to nearest even, NaN kept quiet; written out in
// integer instructions and a branch it was a third of the row-wise kernels' code).
struct bf16_t {
  uint16_t bits;
};

__device__ __forceinline__ float to_float(float v) { return v; }
__device__ __forceinline__ float to_float(bf16_t v) { return __uint_as_float(((uint32_t)v.bits) << 16); }

template <typename T>
__device__ __forceinline__ T from_float(float v);

template <>
__device__ __forceinline__ float from_float<float>(float v) {
  return v;
}

template <>
__device__ __forceinline__ bf16_t from_float<bf16_t>(float v) {
  return bf16_t{__builtin_bit_cast(uint16_t, static_cast<__bf16>(v))};  // v_cvt_pk_bf16_f32
}

// Round a 32-bit value to the storage type and back: the value the storage type would hold.
template <typename T>
__device__ __forceinline__ float round_to(float v) {
  return to_float(from_float<T>(v));
}

// Sums and maxima over a wavefront by data-parallel moves between lanes (an instruction each;
// the shuffles the compiler makes of __shfl_xor go through the LDS crossbar and cost six trips of
// some hundred cycles).  Lanes meet in a fixed order: the four of a quad, the two quads of a
// half row, the two halves of a row of 16, then the rows; every lane returns the result.  All 64
// lanes must be active at the call (a lane that is switched off contributes nothing, where a
// shuffle would still read its register): call them from code the whole wavefront runs.
template <int CONTROL, int ROW_MASK>
__device__ __forceinline__ float lanes_moved(float keep, float v) {
  // Lanes of rows outside ROW_MASK, and lanes whose source does not exist, get `keep`.
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(__builtin_bit_cast(int, keep), __builtin_bit_cast(int, v),
                                                               CONTROL, ROW_MASK, 0xF, false));
}

__device__ __forceinline__ float wave_sum(float v) {
  v += lanes_moved<0xB1, 0xF>(0.f, v);   // quad_perm [1,0,3,2]
  v += lanes_moved<0x4E, 0xF>(0.f, v);   // quad_perm [2,3,0,1]
  v += lanes_moved<0x141, 0xF>(0.f, v);  // row_half_mirror
  v += lanes_moved<0x140, 0xF>(0.f, v);  // row_mirror: every lane holds its row's sum
  v += lanes_moved<0x142, 0xA>(0.f, v);  // row_bcast15 into rows 1 and 3
  v += lanes_moved<0x143, 0xC>(0.f, v);  // row_bcast31 into rows 2 and 3: row 3 holds all
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), TS_WAVE - 1));
}

// The same of N values, step by step beside one another; the last lane holds the sums.
template <int N>
__device__ __forceinline__ void wave_sums(float (&v)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] += lanes_moved<0xB1, 0xF>(0.f, v[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] += lanes_moved<0x4E, 0xF>(0.f, v[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] += lanes_moved<0x141, 0xF>(0.f, v[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] += lanes_moved<0x140, 0xF>(0.f, v[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] += lanes_moved<0x142, 0xA>(0.f, v[i]);
#pragma unroll
  for (int i = 0; i < N; ++i) v[i] += lanes_moved<0x143, 0xC>(0.f, v[i]);
}

__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, lanes_moved<0xB1, 0xF>(v, v));
  v = fmaxf(v, lanes_moved<0x4E, 0xF>(v, v));
  v = fmaxf(v, lanes_moved<0x141, 0xF>(v, v));
  v = fmaxf(v, lanes_moved<0x140, 0xF>(v, v));
  v = fmaxf(v, lanes_moved<0x142, 0xA>(v, v));
  v = fmaxf(v, lanes_moved<0x143, 0xC>(v, v));
  return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), TS_WAVE - 1));
}

// Sum over a block of `blockDim.x` threads (a multiple of 64, at most 1024); `scratch` holds at
// least 16 floats of LDS.  Every thread returns the total.
__device__ __forceinline__ float block_sum(float v, float* scratch) {
  const int lane = threadIdx.x & (TS_WAVE - 1);
  const int wave = threadIdx.x / TS_WAVE;
  const int waves = (blockDim.x + TS_WAVE - 1) / TS_WAVE;
  v = wave_sum(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = 0.f;
  for (int w = 0; w < waves; ++w) total += scratch[w];
  return total;
}

// The same bits where the block's threads are known: the wavefronts' sums are on their way together (one by one in a loop each is a trip
// to LDS, 0.5 us for sixteen).  `scratch`: 16-byte aligned, THREADS / 64 floats, read by nobody any more.
template <int THREADS>
__device__ __forceinline__ float block_sum_of(float v, float* scratch) {
  constexpr int WAVES = THREADS / TS_WAVE;
  v = wave_sum(v);
  if ((threadIdx.x & (TS_WAVE - 1)) == 0) scratch[threadIdx.x / TS_WAVE] = v;
  __syncthreads();
  float total = 0.f;
#pragma unroll
  for (int w = 0; w < WAVES; ++w) total += scratch[w];
  return total;
}

__device__ __forceinline__ float block_max(float v, float* scratch) {
  const int lane = threadIdx.x & (TS_WAVE - 1);
  const int wave = threadIdx.x / TS_WAVE;
  const int waves = (blockDim.x + TS_WAVE - 1) / TS_WAVE;
  v = wave_max(v);
  __syncthreads();
  if (lane == 0) scratch[wave] = v;
  __syncthreads();
  float total = scratch[0];
  for (int w = 1; w < waves; ++w) total = fmaxf(total, scratch[w]);
  return total;
}

// A 16-byte load of data that a kernel reads once (weights, cached keys and values): marked
// non-temporal, so that it does not displace what the caches hold for others.  On an MI355X a
// kernel that only reads streams 6.6 to 7.0 TB/s this way against 5.9 to 6.2 with plain loads.
typedef unsigned int ts_u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ ts_u32x4 load_once16(const void* at) {
  return __builtin_nontemporal_load(reinterpret_cast<const ts_u32x4*>(at));
}

// The gated unit of a feed-forward: with g' = min(g, limit) and u' = clamp(u, -limit, limit) where
// limit > 0 (else g' = g, u' = u), g' * sigmoid(steepness * (g' + cubic * g'^3)) * (u' + up_shift).
// silu(g) * u is {1, 0, 0, 0}; the tanh form of GELU, 0.5 g (1 + tanh(c (g + a g^3))), is
// g * sigmoid(2 c (g + a g^3)): {2 sqrt(2 / pi), 0, 0, 0.044715}.
struct GluRule {
  float steepness;
  float limit;
  float up_shift;
  float cubic;
};

// g * sigmoid(x) for |x| up to GATE_NEAR: 2^t of the hardware with t = -x log2(e) rounded, and the quotient by 1 + 2^t of the hardware's reciprocal,
// corrected once by its remainder, into which goes what the rounding of t left (-x - t ln 2, ln 2 in two parts).  Twelve instructions where
// expf and a division of any numbers are 24; relative to 64 bits 3.1e-8 to 3.6e-8 (root mean square over gates of 1 to 80) where those
// were 3.7e-8 to 4.0e-8.  No factor, divisor or quotient is beyond the normal numbers there, but for those of a denormal g.
constexpr float GATE_NEAR = 80.f;
__device__ __forceinline__ float gated_near(float g, float x) {
  const float t = x * -1.44269502f;
  const float left = fmaf(t, 1.90465432e-9f, fmaf(t, -0.693147182f, -x));
  const float e = __builtin_amdgcn_exp2f(t), r = __builtin_amdgcn_rcpf(1.f + e), q = g * r;
  return fmaf(fmaf(-(q * e), left, fmaf(-q, e, g) - q), r, q);
}

// The same beyond (and for NaN): the sigmoid is 1, or e^x, 2^64 times which is a normal number where the result is not 0.
__device__ __forceinline__ float gated_far(float g, float x) {
#pragma clang fp contract(off)  // t is rounded, t + 64 then exact where the sum is below t
  const float y = fmaxf(x, -4000.f), t = y * 1.44269502f;
  const float left = fmaf(t, 1.90465432e-9f, fmaf(t, -0.693147182f, y));
  const float e = __builtin_amdgcn_exp2f(t + 64.f), p = g * e;
  return x > 0.f ? g : (p + fmaf(p, left, fmaf(g, e, -p))) * 5.42101086e-20f;
}

// The operands within the rule's limits, and what the sigmoid is taken of.
__device__ __forceinline__ void glu_limits(float& g, float& u, float& x, GluRule rule) {
  if (rule.limit > 0.f) {
    g = fminf(g, rule.limit);
    u = fminf(fmaxf(u, -rule.limit), rule.limit);
  }
  x = rule.steepness * (rule.cubic != 0.f ? fmaf(rule.cubic * g * g, g, g) : g);
}

__device__ __forceinline__ float gated_unit(float g, float u, GluRule rule) {
  float x;
  glu_limits(g, u, x, rule);
  return (fabsf(x) <= GATE_NEAR ? gated_near(g, x) : gated_far(g, x)) * (u + rule.up_shift);
}

// max(z, 0)^2, the unit of a feed-forward without a gate.
__device__ __forceinline__ float relu_squared(float z) {
  const float r = fmaxf(z, 0.f);
  return r * r;
}

// One rotation, written out so that every kernel rounds it the same way.
__device__ __forceinline__ void rotate_pair(float x1, float x2, float c, float s, float& o1, float& o2) {
  o1 = __builtin_fmaf(x1, c, -(x2 * s));
  o2 = __builtin_fmaf(x2, c, x1 * s);
}

// ---------------------------------------------------------------------------------------------
// RMSNorm.  y = w * round_T(x * rsqrt(mean(x^2) + eps)): the normalised value is rounded to the
// storage type before the gain, as the reference does (layers.py:208).
//
// add_rmsnorm: s = residual + pending (32-bit); residual = s; y = norm(s).  With `rows` the
// kernel reads rows[i] and writes y[i] only (residual untouched): the final norm at the wanted
// positions.
// ---------------------------------------------------------------------------------------------
// The gain: `one_rounding == 0` is the rule above, w * round_T(n); otherwise the whole norm is
// 32-bit arithmetic with one rounding at the end, round_T(n * (gain_offset + w)) (a gain stored
// around zero has gain_offset 1).
template <typename T>
__device__ __forceinline__ float with_gain(float normalised, float gain, float gain_offset, int one_rounding) {
  return one_rounding ? normalised * (gain_offset + gain) : gain * round_to<T>(normalised);
}

static inline int ts_launch_status() { return hipGetLastError() == hipSuccess ? TS_OK : TS_ERR_LAUNCH; }
