// Y[M, N] = X[M, K] * W[N, K]^T (+ bias[N]) in true 32-bit, no reduced-precision mode: the product
// of the true 32-bit path (the reference's F.linear, src/turboserve/engine/model/layers.py:142, at
// dtype float32) and of bfloat16 operands whose K the 16-byte loads of the other products do not divide.
//
// Every output is the sum, in order, of up to four chains, one per range of K (`range_of`: a quarter of K
// rounded up to 64); a chain is fused multiply-adds in the order of k, each rounded once to 32-bit.
// The chains run on the matrix cores: v_mfma_f32_32x32x2_f32 and v_mfma_f32_16x16x4_f32 add their
// two (four) products to the accumulator one after the other, in the order of k, each step a fused
// multiply-add rounded to nearest with denormals kept (a loop of fmaf gives the same bits; compared
// over random, widely spread, denormal and cancelling operands at K of 4 to 3,584).  So a row's
// result depends neither on which other rows are in the batch nor on which of the layouts
// below runs it, they run at the matrix cores' 157 TFLOP/s, twice what unpacked vector
// multiply-adds allow, and a few rows against a long K get four times the wavefronts one chain would.
//
// Microseconds at the 7B shape, one chain of vector multiply-adds (64 x 64 tiles; up to 32 rows one output a thread)
// -> these: gate|up at 8 / 64 / 500 rows 194 -> 88, 765 -> 152, 3,048 -> 961 (141 TFLOP/s); down 220 -> 47, 3,402 -> 119,
// 3,365 -> 486; o 35 -> 12, 581 -> 25, 581 -> 98; q|k|v 41 -> 16, 579 -> 32, 638 -> 121; the head at 8 rows 637 -> 320.
#include "common.hpp"

#include <type_traits>

namespace {

typedef float gp_f32x4 __attribute__((ext_vector_type(4)));
typedef float gp_f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned int gp_u32x2 __attribute__((ext_vector_type(2)));

// A product whose weight rows alternate gate, up and that leaves the gated unit of each two (32-bit, the layouts that stage through LDS).
struct PlainGlu {
  int gated;
  GluRule rule;
};

constexpr int GP_DIES = 8;
constexpr int GP_UNITS = 256;  // compute units of an MI355X

// Four consecutive elements of one row as they lie in memory, and as 32-bit values.
template <typename TIn>
struct Quad;
template <>
struct Quad<float> {
  gp_f32x4 v;
  __device__ __forceinline__ void load(const float* p) { v = *reinterpret_cast<const gp_f32x4*>(p); }
  __device__ __forceinline__ void set(int i, float f) { v[i] = f; }
  __device__ __forceinline__ gp_f32x4 values() const { return v; }
};
template <>
struct Quad<bf16_t> {
  gp_u32x2 v;
  __device__ __forceinline__ void load(const bf16_t* p) { v = *reinterpret_cast<const gp_u32x2*>(p); }
  __device__ __forceinline__ void set(int i, bf16_t f) {
    const unsigned int other = v[i / 2];
    const unsigned int both = i & 1 ? (other & 0xffffu) | ((unsigned int)f.bits << 16) : (other & 0xffff0000u) | f.bits;
    v[i / 2] = both;
  }
  __device__ __forceinline__ gp_f32x4 values() const {
    const unsigned int lo = v[0], hi = v[1];
    return gp_f32x4{__uint_as_float(lo << 16), __uint_as_float(lo & 0xffff0000u), __uint_as_float(hi << 16),
                    __uint_as_float(hi & 0xffff0000u)};
  }
};

inline long ceil_of(long a, long b) { return (a + b - 1) / b; }

// The length of a range of K, the same for every layout: a function of K alone.
__host__ __device__ constexpr int range_of(int k) { return (((k + 3) / 4 + 63) / 64) * 64; }

// Elements k0 + lane_k .. + 3 of a row: one load where VEC (K, the row strides and the base
// addresses are multiples of four elements), else one by one.  Always inside the row: what lies past
// its end is read from its last elements instead and cleared by the caller.
template <bool VEC>
struct RowOffset {  // of a tile's row from its first one, in elements: 32 bits where VEC (K and the row strides below 2^25)
  typedef uint32_t type;
};
template <>
struct RowOffset<false> {
  typedef size_t type;
};
template <bool VEC, typename TIn>
__device__ __forceinline__ void fetch_quad(Quad<TIn>& q, const TIn* base, typename RowOffset<VEC>::type row, int k0, int lane_k, int k) {
  if (VEC) {
    q.load(base + k0 + (row + min(lane_k, k - 4 - k0)));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i) q.set(i, base[k0 + (row + min(lane_k + i, k - 1 - k0))]);
  }
}

// Clear the elements of a quad that lie past the row's end; `left`: how many lie inside.
__device__ __forceinline__ void clear_past(gp_f32x4& v, int left) {
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = i < left ? v[i] : 0.f;
}

// ---------------------------------------------------------------------------------------------
// Many rows: a workgroup of 2 x 2 wavefronts owns 64 TM activation rows by 64 TN weight rows, a
// wavefront TM x TN tiles of 32 x 32.  Bound by the matrix cores (an iteration of BK is BK TM TN / 2
// instructions of 64 cycles a wavefront); loads go out two iterations ahead into one of two sets of registers.
// In LDS every 8 k of a row lie as 0 2 4 6 1 3 5 7: the half of the wavefront that supplies the even
// (odd) k of four consecutive instructions reads them as 16 bytes; rows are 4 floats longer than
// their k, so that sixteen rows' pieces touch every bank once.
template <int TM, int TN, int BK, bool VEC, typename TIn, typename TOut>
__global__ void __launch_bounds__(256)
gemm_plain_kernel(TOut* __restrict__ y, const TIn* __restrict__ x, const TIn* __restrict__ w,
                  const TIn* __restrict__ bias, int m, int n, int k, long x_stride, long y_stride, int m_tiles, int n_tiles) {
  constexpr int BM = 64 * TM, BN = 64 * TN, ROW = BK + 4, QUADS = BK / 4, PASS = 256 / QUADS;
  constexpr int PX = BM / PASS, PW = BN / PASS;
  __shared__ __attribute__((aligned(16))) float lds[2][(BM + BN) * ROW];
  // Workgroup id -> tile: ids go to the eight dies in turn; the tiles of activation rows over one weight
  // tile follow one another on one die and share the weights in its L2.
  const int die = blockIdx.x % GP_DIES, turn = blockIdx.x / GP_DIES;
  const int n_tile = (turn / m_tiles) * GP_DIES + die;
  if (n_tile >= n_tiles) return;  // the whole workgroup leaves together
  const int m0 = (turn % m_tiles) * BM, n0 = n_tile * BN;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int r = lane & 31, half = lane >> 5;
  const int wave_m = wave >> 1, wave_n = wave & 1;

  // A quad's address: the tile's first row (the same for the workgroup) and a 32-bit offset of the row.
  const int quad_k = 4 * (tid % QUADS), quad_row = tid / QUADS;
  const TIn* xbase = x + (size_t)m0 * x_stride;
  const TIn* wbase = w + (size_t)n0 * k;
  typedef typename RowOffset<VEC>::type Row;
  Row xrow[PX], wrow[PW];
#pragma unroll
  for (int i = 0; i < PX; ++i) xrow[i] = (Row)min(quad_row + PASS * i, m - 1 - m0) * (Row)x_stride;
#pragma unroll
  for (int i = 0; i < PW; ++i) wrow[i] = (Row)min(quad_row + PASS * i, n - 1 - n0) * (Row)k;

  struct Set {
    Quad<TIn> x[PX], w[PW];
  };
  const int iters = (k + BK - 1) / BK;
  auto fetch = [&](Set& s, int it) __attribute__((always_inline)) {
    const int k0 = min(it, iters - 1) * BK;
#pragma unroll
    for (int i = 0; i < PX; ++i) fetch_quad<VEC>(s.x[i], xbase, xrow[i], k0, quad_k, k);
#pragma unroll
    for (int i = 0; i < PW; ++i) fetch_quad<VEC>(s.w[i], wbase, wrow[i], k0, quad_k, k);
  };
  const int at = quad_row * ROW + (quad_k & ~7) + (quad_k & 4) / 2;  // of the quad's even k; the odd ones 4 behind
  auto stage = [&](const Set& s, int it, int buf) __attribute__((always_inline)) {
    float* to = lds[buf] + at;
    const int left = k - (it * BK + quad_k);
    auto put = [&](gp_f32x4 v, int row) __attribute__((always_inline)) {
      clear_past(v, left);
      *reinterpret_cast<float2*>(to + row * ROW) = make_float2(v[0], v[2]);
      *reinterpret_cast<float2*>(to + row * ROW + 4) = make_float2(v[1], v[3]);
    };
#pragma unroll
    for (int i = 0; i < PX; ++i) put(s.x[i].values(), PASS * i);
#pragma unroll
    for (int i = 0; i < PW; ++i) put(s.w[i].values(), BM + PASS * i);
  };

  gp_f32x16 acc[TM][TN], sum[TM][TN];  // the range's chain, the ranges before it
#pragma unroll
  for (int a = 0; a < TM; ++a) {
#pragma unroll
    for (int b = 0; b < TN; ++b) {
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.f, sum[a][b][i] = 0.f;
    }
  }
  constexpr int GROUPS = BK / 8;  // eight k at a time
  struct Frags {
    gp_f32x4 x[TM], w[TN];
  };
  auto read = [&](Frags& f, int buf, int g) __attribute__((always_inline)) {
    const float* xs = lds[buf] + (wave_m * 32 * TM + r) * ROW + 4 * half + 8 * g;
    const float* ws = lds[buf] + (BM + wave_n * 32 * TN + r) * ROW + 4 * half + 8 * g;
#pragma unroll
    for (int a = 0; a < TM; ++a) f.x[a] = *reinterpret_cast<const gp_f32x4*>(xs + a * 32 * ROW);
#pragma unroll
    for (int b = 0; b < TN; ++b) f.w[b] = *reinterpret_cast<const gp_f32x4*>(ws + b * 32 * ROW);
  };
  auto multiply = [&](const Frags& f) __attribute__((always_inline)) {
#pragma unroll
    for (int s = 0; s < 4; ++s) {
#pragma unroll
      for (int a = 0; a < TM; ++a) {
#pragma unroll
        for (int b = 0; b < TN; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x2f32(f.x[a][s], f.w[b][s], acc[a][b], 0, 0, 0);
      }
    }
  };

  const int range_iters = range_of(k) / BK;
  int range_end = min(range_iters, iters);
  Set s0, s1;
  fetch(s0, 0);
  fetch(s1, 1);
  stage(s0, 0, 0);
  __syncthreads();
  // Buffer it & 1 holds iteration it, f[0] its first group; `next` holds it + 1 and goes to the other buffer; `free`
  // takes the loads of it + 2 (past the end: the last iteration's again, never read).  A group's fragments are
  // read while the one before it is multiplied, the next iteration's first across the barrier: a wavefront that
  // reaches it has what it reads of this buffer in registers and its part of the other one in LDS.
  Frags f[2];
  read(f[0], 0, 0);
  auto round = [&](int it, Set& next, Set& free) __attribute__((always_inline)) {
    const int buf = it & 1;
    fetch(free, it + 2);
    if (TM * TN > 1) {
      // Sixteen matrix instructions a group: the staging and the loads are asked for between them, a little behind
      // each (500 rows of gate|up 1,194 -> 1,154 us); behind four (tiles of 64 x 64) they are faster in one piece
      // (down at 128 rows 390 us, interleaved 419).
      stage(next, it + 1, buf ^ 1);
#pragma unroll
      for (int g = 0; g + 1 < GROUPS; ++g) {
        read(f[(g + 1) & 1], buf, g + 1);
        multiply(f[g & 1]);
      }
      __builtin_amdgcn_sched_group_barrier(0x100, TM + TN, 0);  // DS read
#pragma unroll
      for (int i = 0; i < 4 * TM * TN * (GROUPS - 1); ++i) {
        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
        __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);  // VALU
        __builtin_amdgcn_sched_group_barrier(0x200, 2, 0);  // DS write
        __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // VMEM read
        __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);  // DS read
      }
    } else {
#pragma unroll
      for (int g = 0; g + 1 < GROUPS; ++g) {
        if (g == GROUPS / 2) stage(next, it + 1, buf ^ 1);
        read(f[(g + 1) & 1], buf, g + 1);
        __builtin_amdgcn_sched_barrier(0);
        multiply(f[g & 1]);
      }
    }
    __syncthreads();
    read(f[GROUPS & 1], buf ^ 1, 0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(f[(GROUPS - 1) & 1]);
    if (it + 1 == range_end) {  // the same for every thread
#pragma unroll
      for (int a = 0; a < TM; ++a) {
#pragma unroll
        for (int b = 0; b < TN; ++b) {
#pragma unroll
          for (int i = 0; i < 16; ++i) sum[a][b][i] += acc[a][b][i], acc[a][b][i] = 0.f;
        }
      }
      range_end = min(range_end + range_iters, iters);
    }
  };
  for (int it = 0; it < iters; it += 2) {
    round(it, s1, s0);
    if (it + 1 >= iters) break;
    round(it + 1, s0, s1);
  }

  // sum[a][b][i]: activation row 32 (wave_m TM + a) + 8 (i / 4) + 4 half + i % 4, weight row 32 (wave_n TN + b) + r.
#pragma unroll
  for (int b = 0; b < TN; ++b) {
    const int col = n0 + (wave_n * TN + b) * 32 + r;
    if (col >= n) continue;
    const float bv = bias ? to_float(bias[col]) : 0.f;
#pragma unroll
    for (int a = 0; a < TM; ++a) {
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int row = m0 + (wave_m * TM + a) * 32 + 8 * (i / 4) + 4 * half + i % 4;
        if (row < m) y[(size_t)row * y_stride + col] = from_float<TOut>(bias ? sum[a][b][i] + bv : sum[a][b][i]);
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Few rows of bfloat16 (up to 32 rows: that four elements divide), or of 32-bit rows that 16-byte loads do not divide: a workgroup owns 16 MT activation rows by 16 NT weight rows, each of its four wavefronts one range of
// K; both operands go straight from memory into registers, AHEAD slices of 64 k in flight, without LDS
// or a barrier before the ranges' sums meet at the end: bound by reading W.
// Lane (r, g) = (lane % 16, lane / 16) loads 16 bytes of row r: elements 4 g .. 4 g + 3 of every 16, 64 bytes of each of
// sixteen rows an instruction; four lane swaps (permlane32/16) turn the 4 x 4 of groups and
// elements round, so that step s of the 16 holds element 4 s + g: the order of k.
// The loads are plain ones: an instruction takes half a line, and marked non-temporal the other half
// came from memory again (32-bit gate|up at 8 rows 152 us, plain 131).
__device__ __forceinline__ void turn_quads(gp_f32x4& v) {
  float e0 = v[0], e1 = v[1], e2 = v[2], e3 = v[3];
  auto swap32 = [](float& a, float& b) __attribute__((always_inline)) {
    const auto s = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(s[0]);
    b = __uint_as_float(s[1]);
  };
  auto swap16 = [](float& a, float& b) __attribute__((always_inline)) {
    const auto s = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
    a = __uint_as_float(s[0]);
    b = __uint_as_float(s[1]);
  };
  swap32(e0, e2);
  swap32(e1, e3);
  swap16(e0, e1);
  swap16(e2, e3);
  v = gp_f32x4{e0, e1, e2, e3};
}

template <int MT, int NT, int AHEAD, bool VEC, typename TIn, typename TOut>
__global__ void __launch_bounds__(256)
gemm_plain_few_rows_kernel(TOut* __restrict__ y, const TIn* __restrict__ x, const TIn* __restrict__ w,
                           const TIn* __restrict__ bias, int m, int n, int k, long x_stride, long y_stride) {
  constexpr int SLICE = 64, QUADS = SLICE / 16;
  __shared__ gp_f32x4 parts[3][MT * NT][64];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);  // the same for the wavefront, and known to be
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16 * NT, m0 = blockIdx.y * 16 * MT;
  const int range = range_of(k), start = wave * range, end = min(start + range, k);  // this wavefront's k (none: start >= end)
  const TIn* xbase = x + (size_t)m0 * x_stride;
  const TIn* wbase = w + (size_t)n0 * k;
  typedef typename RowOffset<VEC>::type Row;
  Row xrow[MT], wrow[NT];
#pragma unroll
  for (int t = 0; t < MT; ++t) xrow[t] = (Row)min(16 * t + r, m - 1 - m0) * (Row)x_stride;
#pragma unroll
  for (int t = 0; t < NT; ++t) wrow[t] = (Row)min(16 * t + r, n - 1 - n0) * (Row)k;

  struct Set {
    Quad<TIn> x[MT][QUADS], w[NT][QUADS];
  };
  gp_f32x4 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a) {
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = gp_f32x4{0.f, 0.f, 0.f, 0.f};
  }
  auto fetch = [&](Set& s, int k0, bool whole) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < QUADS; ++c) {
#pragma unroll
      for (int t = 0; t < NT; ++t) fetch_quad<VEC>(s.w[t][c], wbase, wrow[t], k0, 16 * c + 4 * g, whole ? 0x7fffffff : k);
#pragma unroll
      for (int t = 0; t < MT; ++t) fetch_quad<VEC>(s.x[t][c], xbase, xrow[t], k0, 16 * c + 4 * g, whole ? 0x7fffffff : k);
    }
  };
  auto consume = [&](const Set& s, int left) __attribute__((always_inline)) {  // left: elements of the slice inside the row
#pragma unroll
    for (int c = 0; c < QUADS; ++c) {
      gp_f32x4 xv[MT], wv[NT];
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        xv[t] = s.x[t][c].values();
        if (left < SLICE) clear_past(xv[t], left - 16 * c - 4 * g);
        turn_quads(xv[t]);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        wv[t] = s.w[t][c].values();
        if (left < SLICE) clear_past(wv[t], left - 16 * c - 4 * g);
        turn_quads(wv[t]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int a = 0; a < MT; ++a) {
#pragma unroll
          for (int b = 0; b < NT; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(xv[a][e], wv[b][e], acc[a][b], 0, 0, 0);
        }
      }
    }
  };

  const int slices = start < end ? (end - start) / SLICE : 0;  // whole ones
  if (slices > 0) {
    Set ring[AHEAD];  // slot j: a slice whose number is j modulo AHEAD
    const int last = start + (slices - 1) * SLICE;
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) fetch(ring[j], min(start + j * SLICE, last), true);  // past the end: the last slice again
    int s0 = 0;
    for (; s0 + AHEAD <= slices; s0 += AHEAD) {
#pragma unroll
      for (int j = 0; j < AHEAD; ++j) {
        consume(ring[j], SLICE);
        fetch(ring[j], min(start + (s0 + j + AHEAD) * SLICE, last), true);
      }
    }
#pragma unroll
    for (int j = 0; j < AHEAD; ++j)
      if (s0 + j < slices) consume(ring[j], SLICE);
  }
  if (start + slices * SLICE < end) {  // the rest of a K that is no multiple of 64
    Set rest;
    fetch(rest, start + slices * SLICE, false);
    consume(rest, end - start - slices * SLICE);
  }

  if (wave > 0) {
#pragma unroll
    for (int a = 0; a < MT; ++a) {
#pragma unroll
      for (int b = 0; b < NT; ++b) parts[wave - 1][a * NT + b][lane] = acc[a][b];
    }
  }
  __syncthreads();
  if (wave > 0) return;
  // acc[a][b][i]: activation row m0 + 16 a + 4 g + i, weight row n0 + 16 b + r.
#pragma unroll
  for (int b = 0; b < NT; ++b) {
    const int col = n0 + 16 * b + r;
    if (col >= n) continue;
    const float bv = bias ? to_float(bias[col]) : 0.f;
#pragma unroll
    for (int a = 0; a < MT; ++a) {
      gp_f32x4 sum = gp_f32x4{0.f, 0.f, 0.f, 0.f} + acc[a][b];
#pragma unroll
      for (int p = 1; p < 4; ++p)
        if (p * range < k) sum += parts[p - 1][a * NT + b][lane];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = m0 + 16 * a + 4 * g + i;
        if (row < m) y[(size_t)row * y_stride + col] = from_float<TOut>(bias ? sum[i] + bv : sum[i]);
      }
    }
  }
}

// ---------------------------------------------------------------------------------------------
// Up to 32 rows of bfloat16 whose K or strides four elements do not divide: what bounds them is the number of 2-byte loads, and
// with a wavefront a range of K each of them touches sixteen rows.  Here a workgroup owns 16 x 16 outputs, one a thread, and
// walks K in slices of 64 that travel memory -> registers -> LDS (two buffers, one barrier a slice, two slices of loads
// ahead): a row's slice is 128 bytes of sixteen neighbouring lanes.  The same chains, by vector fused multiply-adds.  The
// layout above -> this one, us at 1 / 16 / 32 rows: 18,944 x 3,583 140 / 226 / 260 -> 104 / 104 / 180, 4,608 x 2,049 60 / 66 / 85
// -> 31 / 31 / 41, 3,584 x 9,001 195 / 192 / 308 -> 104 / 104 / 116, 512 x 511 9.4 / 11.3 / 11.5 -> 7.7 / 8.0 / 8.1.
constexpr int UNEVEN_TILE = 16, UNEVEN_SLICE = 64, UNEVEN_MOST_ROWS = 32;

template <typename TOut>
__global__ void __launch_bounds__(256)
gemm_plain_uneven_kernel(TOut* __restrict__ y, const bf16_t* __restrict__ x, const bf16_t* __restrict__ w,
                         const bf16_t* __restrict__ bias, int m, int n, int k, long x_stride, long y_stride) {
  __shared__ __attribute__((aligned(16))) float lds[2][2][UNEVEN_TILE][UNEVEN_SLICE + 4];  // buffer, operand: x, w
  const int row = threadIdx.x / 16, lane_k = threadIdx.x % 16 * 4;  // of both operands: what this thread fetches of a slice
  const int m0 = blockIdx.y * UNEVEN_TILE, n0 = blockIdx.x * UNEVEN_TILE;
  const bf16_t* const xrow = x + (size_t)min(m0 + row, m - 1) * x_stride;
  const bf16_t* const wrow = w + (size_t)min(n0 + row, n - 1) * k;
  float xr[2][4], wr[2][4];  // set j: a slice whose number is j modulo 2
  auto fetch = [&](int j, int slice) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // past the end the last element again, counted as zero
      const int at = slice * UNEVEN_SLICE + lane_k + i;
      const float a = to_float(xrow[min(at, k - 1)]), b = to_float(wrow[min(at, k - 1)]);
      xr[j][i] = at < k ? a : 0.f;
      wr[j][i] = at < k ? b : 0.f;
    }
  };
  auto stage = [&](int j) __attribute__((always_inline)) {
    *reinterpret_cast<gp_f32x4*>(&lds[j][0][row][lane_k]) = gp_f32x4{xr[j][0], xr[j][1], xr[j][2], xr[j][3]};
    *reinterpret_cast<gp_f32x4*>(&lds[j][1][row][lane_k]) = gp_f32x4{wr[j][0], wr[j][1], wr[j][2], wr[j][3]};
  };
  const int slices = (k + UNEVEN_SLICE - 1) / UNEVEN_SLICE, range = range_of(k) / UNEVEN_SLICE;
  const int out_m = threadIdx.x % 16, out_n = threadIdx.x / 16;  // the output this thread owns
  float acc = 0.f, sum = 0.f;  // the range's chain, the ranges before it
  int range_end = min(range, slices);
  fetch(0, 0);
  fetch(1, 1);
  stage(0);
  __syncthreads();
  auto round = [&](int s, int j) __attribute__((always_inline)) {  // slice s lies in buffer j; every thread walks the same slices
    fetch(j, s + 2);
    const float* a = lds[j][0][out_m];
    const float* b = lds[j][1][out_n];
#pragma unroll 1  // in one piece the compiler reads the whole slice into registers first: 148 of them, three wavefronts a SIMD
    for (int part = 0; part < UNEVEN_SLICE; part += 16) {
#pragma unroll
      for (int kk = part; kk < part + 16; ++kk) acc = fmaf(a[kk], b[kk], acc);  // in the order of k
    }
    if (s + 1 == range_end) {
      sum += acc;
      acc = 0.f;
      range_end = min(range_end + range, slices);
    }
    stage(j ^ 1);  // that buffer was last read in the slice before this one, which every thread has left
    __syncthreads();
  };
  for (int s = 0; s < slices; s += 2) {
    round(s, 0);
    if (s + 1 < slices) round(s + 1, 1);
  }
  const int gm = m0 + out_m, gn = n0 + out_n;
  if (gm < m && gn < n) y[(size_t)gm * y_stride + gn] = from_float<TOut>(bias ? sum + to_float(bias[gn]) : sum);
}

// ---------------------------------------------------------------------------------------------
// The same few rows of 32-bit operands, bound by reading W: whole lines, straight from memory to LDS.  Above, an instruction
// takes 64 bytes of each of sixteen rows and W cannot be marked as read once (4.3 TB/s); here one takes 128 bytes of
// each of eight, non-temporal where one tile of activation rows reads them.  A wavefront stages its own range
// in a ring of its own, SLOTS slices of 32 k (a slot is filled again as soon as its fragments are in registers), so nothing
// meets at a barrier before the ranges' sums.  gate|up at 8 rows 127 -> 88 us (6.1 TB/s), at 32 191 -> 122; the head at 8 441 -> 330
// (6.6 TB/s); down 61 -> 47, o 16.4 -> 12.6, q|k|v 25 -> 18.  Piece p (16 bytes) of row r lies at position p ^ (r / 2 % 8) of the row's eight:
// a piece of sixteen rows touches every bank once.  The same chains, bit for bit.
typedef __attribute__((address_space(3))) float lds_f32;
typedef __attribute__((address_space(3))) gp_f32x4 lds_f32x4;

template <int MT, int NT>
struct Stream {
  static constexpr int SLICE = 32, TILE = 16 * SLICE, LOADS = 2 * (MT + NT);          // of a tile of sixteen rows; of a slice
  static constexpr int SLOTS = 80 * 1024 / (4 * (MT + NT) * TILE * 4);                // two workgroups a compute unit
  static constexpr int WAVE = SLOTS * (MT + NT) * TILE;                               // floats of a wavefront's ring
  static constexpr size_t BYTES = (size_t)4 * WAVE * 4;
  static_assert(SLOTS >= 2 && (SLOTS - 1) * LOADS < 64 && 2 * BYTES <= 160 * 1024, "a ring of at least two slices, counted by vmcnt");
  static_assert(WAVE >= MT * NT * 256, "a wavefront's sums fit its ring");
};

// `to` and `from` are the same memory: __restrict__ keeps the compiler from waiting for every load in flight before every
// read, so it must not see that two reads have one address either: the slot that stream_wait lets be read is a new value to
// it (a slot it could follow, it read once for all rounds; no read moves above it), and a slot's fragments go through an asm
// that waits for them before it is filled again.  An edit has to keep both.
template <int LEFT>
__device__ __forceinline__ void stream_wait(int& slot) {
  asm volatile("s_waitcnt vmcnt(%1)" : "+s"(slot) : "n"(LEFT) : "memory");
}

template <int MT, int NT, bool ONCE>
__device__ __forceinline__ void stream_ranges(lds_f32* __restrict__ to, const lds_f32* __restrict__ from, const float* __restrict__ x,
                                              const float* __restrict__ w, int m, int n, int k, long x_stride,
                                              gp_f32x4 (&acc)[MT][NT]) {
  typedef Stream<MT, NT> S;
  constexpr int SLICE = S::SLICE, TILE = S::TILE, SLOTS = S::SLOTS;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * 16 * NT, m0 = blockIdx.y * 16 * MT;
  const int range = range_of(k), start = wave * range, end = min(start + range, k);  // this wavefront's k
  if (start >= end) return;
  const int count = (end - start + SLICE - 1) / SLICE;
  // A lane loads piece (lane % 8) ^ key of row lane / 8 of eight; the second eight of a tile, whose keys are four further on, piece ^ 4.  Offsets count
  // from a tile's first row: what lies past the last row's end (rows beyond N or M, k beyond the last row's) brings zeros,
  // k beyond another row's end that row's neighbours, cleared below.
  const int row8 = lane >> 3, piece = (lane & 7) ^ (row8 >> 1);
  const size_t wbytes = (size_t)min(n - n0, 16 * NT) * k * 4, xbytes = ((size_t)(min(m - m0, 16 * MT) - 1) * x_stride + k) * 4;
  const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(w + (size_t)n0 * k), 0, (int)wbytes, 0x00027000);
  const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x + (size_t)m0 * x_stride), 0, (int)xbytes, 0x00027000);
  uint32_t woff[2 * NT], xoff[2 * MT];
#pragma unroll
  for (int j = 0; j < 2 * NT; ++j) woff[j] = ((uint32_t)(8 * j + row8) * (uint32_t)k + start + 4 * (piece ^ (j & 1 ? 4 : 0))) * 4;
#pragma unroll
  for (int j = 0; j < 2 * MT; ++j) xoff[j] = ((uint32_t)(8 * j + row8) * (uint32_t)x_stride + start + 4 * (piece ^ (j & 1 ? 4 : 0))) * 4;
  auto fetch = [&](int i, int slot) __attribute__((always_inline)) {
    const uint32_t at = i < count ? (uint32_t)i * (SLICE * 4) : 0x80000000u;  // past the end: outside the buffers, nothing is fetched
    lds_f32* base = to + slot * (MT + NT) * TILE;
#pragma unroll
    for (int j = 0; j < 2 * NT; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wbuf, base + j * (TILE / 2), 16, woff[j] + at, 0, 0, ONCE ? 2 : 0);
#pragma unroll
    for (int j = 0; j < 2 * MT; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xbuf, base + NT * TILE + j * (TILE / 2), 16, xoff[j] + at, 0, 0, 0);
  };
  struct Frags {
    gp_f32x4 x[MT][2], w[NT][2];
  };
  const int key = (r >> 1) & 7;
  auto read = [&](Frags& f, int slot) __attribute__((always_inline)) {
    const lds_f32* base = from + slot * (MT + NT) * TILE + r * SLICE;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int at = 4 * ((4 * c + g) ^ key);
#pragma unroll
      for (int t = 0; t < NT; ++t) f.w[t][c] = *(const lds_f32x4*)(base + t * TILE + at);
#pragma unroll
      for (int t = 0; t < MT; ++t) f.x[t][c] = *(const lds_f32x4*)(base + (NT + t) * TILE + at);
    }
  };
  auto consume = [&](Frags& f, int left) __attribute__((always_inline)) {  // left: elements of the slice inside the row
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int t = 0; t < MT; ++t) {
        if (left < SLICE) clear_past(f.x[t][c], left - 16 * c - 4 * g);
        turn_quads(f.x[t][c]);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if (left < SLICE) clear_past(f.w[t][c], left - 16 * c - 4 * g);
        turn_quads(f.w[t][c]);
      }
#pragma unroll
      for (int e = 0; e < 4; ++e) {
#pragma unroll
        for (int a = 0; a < MT; ++a) {
#pragma unroll
          for (int b = 0; b < NT; ++b) acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(f.x[a][c][e], f.w[b][c][e], acc[a][b], 0, 0, 0);
        }
      }
    }
  };
#pragma unroll
  for (int j = 0; j < SLOTS; ++j) fetch(j, j);
  int slot = 0;
  stream_wait<(SLOTS - 1) * S::LOADS>(slot);
  Frags f[2];
  read(f[0], slot);
  auto round = [&](int i, Frags& now, Frags& next) __attribute__((always_inline)) {
    // `now` is in registers: its slot is free.
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int t = 0; t < NT; ++t) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(now.w[t][c])::"memory");
#pragma unroll
      for (int t = 0; t < MT; ++t) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(now.x[t][c])::"memory");
    }
    fetch(i + SLOTS, slot);
    slot = slot + 1 == SLOTS ? 0 : slot + 1;
    stream_wait<(SLOTS - 1) * S::LOADS>(slot);
    read(next, slot);
    consume(now, SLICE);
  };
  int i = 0;  // the last slice alone may be cut short
  for (; i + 2 < count; i += 2) {
    round(i, f[0], f[1]);
    round(i + 1, f[1], f[0]);
  }
  const int left = end - start - (count - 1) * SLICE;
  if (i + 1 < count) {
    round(i, f[0], f[1]);
    consume(f[1], left);
  } else {
    consume(f[0], left);
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // loads past the end
}

template <int MT, int NT, bool ONCE>
__global__ void __launch_bounds__(256)
gemm_plain_stream_kernel(float* __restrict__ y, const float* __restrict__ x, const float* __restrict__ w,
                         const float* __restrict__ bias, int m, int n, int k, long x_stride, long y_stride, PlainGlu glu) {
  typedef Stream<MT, NT> S;
  extern __shared__ __attribute__((aligned(16))) float ring[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  gp_f32x4 acc[MT][NT];
#pragma unroll
  for (int a = 0; a < MT; ++a) {
#pragma unroll
    for (int b = 0; b < NT; ++b) acc[a][b] = gp_f32x4{0.f, 0.f, 0.f, 0.f};
  }
  lds_f32* mine = (lds_f32*)ring + wave * S::WAVE;
  stream_ranges<MT, NT, ONCE>(mine, mine, x, w, m, n, k, x_stride, acc);
  // The ranges' sums meet in the rings.
#pragma unroll
  for (int a = 0; a < MT; ++a) {
#pragma unroll
    for (int b = 0; b < NT; ++b) *(lds_f32x4*)(mine + ((a * NT + b) * 64 + lane) * 4) = acc[a][b];
  }
  __syncthreads();
  // Wavefront v adds up and stores tiles v, v + 4, ...
  const int r = lane & 15, g = lane >> 4, range = range_of(k);
#pragma unroll
  for (int t = 0; t < MT * NT; ++t) {
    if (t % 4 != wave) continue;
    const int col = blockIdx.x * 16 * NT + 16 * (t % NT) + r;
    if (col >= n) continue;
    gp_f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int p = 0; p < 4; ++p)
      if (p == 0 || p * range < k) sum += *(const lds_f32x4*)((lds_f32*)ring + p * S::WAVE + (t * 64 + lane) * 4);
    const float bv = bias ? bias[col] : 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int row = blockIdx.y * 16 * MT + 16 * (t / NT) + 4 * g + i;
      const float v = bias ? sum[i] + bv : sum[i];
      if (glu.gated) {  // the up value is the next lane's
        const float up = lanes_moved<0xB1, 0xF>(v, v);  // quad_perm [1,0,3,2]
        if (row < m && r % 2 == 0) y[(size_t)row * y_stride + col / 2] = gated_unit(v, up, glu.rule);
      } else if (row < m) {
        y[(size_t)row * y_stride + col] = v;
      }
    }
  }
}

template <int MT, int NT, bool ONCE>
int launch_stream(void* y, const void* x, const void* w, const void* bias, int m, int n, int k, long x_stride, long y_stride,
                  dim3 grid, PlainGlu glu, hipStream_t stream) {
  static bool raised = false;  // per process; the attribute belongs to the kernel
  if (!raised) {
    if (hipFuncSetAttribute((const void*)gemm_plain_stream_kernel<MT, NT, ONCE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)Stream<MT, NT>::BYTES) != hipSuccess)
      return TS_ERR_LAUNCH;
    raised = true;
  }
  hipLaunchKernelGGL((gemm_plain_stream_kernel<MT, NT, ONCE>), grid, dim3(256), (Stream<MT, NT>::BYTES), stream, (float*)y,
                     (const float*)x, (const float*)w, (const float*)bias, m, n, k, x_stride, y_stride, glu);
  return ts_launch_status();
}

// ---------------------------------------------------------------------------------------------
// Many 32-bit rows whose K is a multiple of 32: a workgroup of four wavefronts owns 64 activation rows by 16 NT weight rows, a
// wavefront NT tiles of v_mfma_f32_16x16x4_f32.  Bound by the matrix cores, and by everything that a wavefront has its vector unit do
// meanwhile: a 32-bit matrix instruction holds it (32 cycles alone, 51 with two vector instructions behind each, 70 with seven, where a
// bfloat16 one takes three beside it).  So the loop has none: operands go straight from memory to LDS, SLOTS slices of 32 k ahead, their
// offsets kept; a fragment is read from LDS in the order of k, an element of one k of sixteen rows a time (two tiles an instruction), through eight kept
// addresses; slots are numbers known to the compiler.
// Piece p (16 bytes) of row r lies at position p ^ (r / 2 % 8) of the row's eight: the elements that an instruction reads of sixteen rows touch
// every bank once.  The same chains, bit for bit.
template <int NT>
struct PlainRing {
  static constexpr int SLICE = 32, ROWS = 16 * NT + 64, SLOT = ROWS * SLICE;  // floats of a slice
  static constexpr int WLOADS = (NT + 1) / 2, XLOADS = 2, LOADS = WLOADS + XLOADS;  // of a wavefront, eight rows each
  static constexpr int SLOTS = 4;
  static constexpr size_t BYTES = (size_t)SLOTS * SLOT * 4;
  static_assert(NT >= 2 && (SLOTS - 1) * LOADS < 64 && BYTES <= 160 * 1024, "the ring must fit the LDS of a compute unit, its loads vmcnt");
};

// `to` and `from` are the same memory: __restrict__ keeps the compiler from waiting for every load in flight before every
// read.  What orders them: every read's address has come through the asm behind the wait for its loads (at), and a slot is filled again behind the
// barrier before which every wavefront has what it reads of it in registers.  An edit has to keep both.
template <int NT>
__device__ __forceinline__ void plain_block(lds_f32* __restrict__ to, const lds_f32* __restrict__ from, float* __restrict__ y,
                                            const float* __restrict__ x, const float* __restrict__ w, const float* __restrict__ bias, int m,
                                            int n, int k, long x_stride, long y_stride, int m_tiles, int n_tiles, PlainGlu glu) {
  typedef PlainRing<NT> R;
  constexpr int SLICE = R::SLICE, SLOT = R::SLOT, SLOTS = R::SLOTS, WLOADS = R::WLOADS, XLOADS = R::XLOADS, FRAGS = NT + 1;
  // Workgroup id -> tile: ids go to the eight dies in turn; a die takes an eighth of the tiles, which follow one another over eight tiles of
  // activation rows (512 rows) and then over the weight tiles, so that what runs on a die at once, 8 by 4 tiles, shares both in its L2.
  const int mine = (n_tiles * m_tiles + GP_DIES - 1) / GP_DIES;
  const int place = blockIdx.x % GP_DIES * mine + blockIdx.x / GP_DIES;
  if (place >= n_tiles * m_tiles) return;  // the whole workgroup leaves together
  const int band = place / (8 * n_tiles), in_band = place % (8 * n_tiles), high = min(8, m_tiles - 8 * band);
  const int m0 = (8 * band + in_band % high) * 64, n0 = in_band / high * 16 * NT;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r = lane & 15, g = lane >> 4;

  // A load takes eight rows' slices, a lane piece (lane % 8) ^ key of row lane / 8.  Wavefront v takes the eights v, v + 4, ...; where there is none
  // it loads its last one again.  What lies past the last row's end (rows beyond N or M) brings zeros, which are not stored.
  const int row8 = lane >> 3, piece = (lane & 7) ^ (4 * (wave & 1) + (row8 >> 1));
  const float *const w_rows = w + (size_t)n0 * k, *const x_rows = x + (size_t)m0 * x_stride;
  const size_t w_bytes = ((size_t)(min(n - n0, 16 * NT) - 1) * k + k) * 4, x_bytes = ((size_t)(min(m - m0, 64) - 1) * x_stride + k) * 4;
  int woff[WLOADS], xoff[XLOADS], eight[WLOADS];
#pragma unroll
  for (int j = 0; j < WLOADS; ++j) {
    eight[j] = wave + 4 * j < 2 * NT ? wave + 4 * j : wave + 4 * j - 4;
    woff[j] = ((8 * eight[j] + row8) * k + 4 * piece) * 4;
    asm volatile("" : "+v"(woff[j]));  // kept, not added up again
  }
#pragma unroll
  for (int j = 0; j < XLOADS; ++j) {
    xoff[j] = ((8 * (wave + 4 * j) + row8) * (int)x_stride + 4 * piece) * 4;
    asm volatile("" : "+v"(xoff[j]));
  }
  const int count = k / SLICE;
  // Slice i: its buffers (empty past the end) and its place in them.
  auto buffer = [&](const float* rows, size_t bytes, int i) __attribute__((always_inline)) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(rows), 0, i < count ? (int)bytes : 0, 0x00027000);
  };
  auto place_of = [&](int i) __attribute__((always_inline)) { return i < count ? i * (SLICE * 4) : 0; };
  auto load = [&](int j, int i, int slot) __attribute__((always_inline)) {
    if (j < WLOADS)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer(w_rows, w_bytes, i), to + slot * SLOT + 8 * eight[j] * SLICE, 16, woff[j], place_of(i), 0, 0);
    else
      __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer(x_rows, x_bytes, i), to + slot * SLOT + (16 * NT + 8 * (wave + 4 * (j - WLOADS))) * SLICE,
                                               16, xoff[j - WLOADS], place_of(i), 0, 0);
  };
  // Where this lane's element of four k lies, piece q of the slice, in bytes: of a weight tile's row r, and of its activation rows; in the first two
  // slots and in the last two (an instruction reaches 64 KB beyond its address).
  constexpr int FAR = SLOTS / 2;
  unsigned at[2][2][8];
#pragma unroll
  for (int q = 0; q < 8; ++q) {
    const unsigned base = (unsigned)(uintptr_t)from + 4 * (r * SLICE + 4 * (q ^ ((r >> 1) & 7)) + g);
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      at[f][0][q] = base + 4 * f * FAR * SLOT;
      at[f][1][q] = at[f][0][q] + 4 * (16 * NT + 16 * wave) * SLICE;
    }
  }
  float f[2][4][FRAGS];  // of sixteen k, in steps of four: the weights' fragments, the activations'
  auto read = [&](int half, int e, int t, int slot) __attribute__((always_inline)) {
    const unsigned base = at[slot / FAR][t < NT ? 0 : 1][4 * half + e];
    f[half][e][t] = ((const lds_f32*)(uintptr_t)base)[slot % FAR * SLOT + 16 * (t < NT ? t : 0) * SLICE];
  };
  gp_f32x4 acc[NT], sum[NT];  // the range's chain, the ranges before it
#pragma unroll
  for (int b = 0; b < NT; ++b) acc[b] = sum[b] = gp_f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int i = 0; i < SLOTS; ++i) {
#pragma unroll
    for (int j = 0; j < R::LOADS; ++j) load(j, i, i);
  }
  auto renew = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int q = 0; q < 8; ++q) asm volatile("" : "+v"(at[i][0][q]), "+v"(at[i][1][q])::"memory");
    }
  };
  auto arrive = [&](auto LEFT) __attribute__((always_inline)) {  // with LEFT loads still on their way
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(decltype(LEFT)::value) : "memory");
    renew();
  };
  auto held = [&]() __attribute__((always_inline)) {
    __builtin_amdgcn_s_waitcnt(0xc07f);  // lgkmcnt(0), one wait instead of one for each
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
      for (int t = 0; t < FRAGS; ++t) asm volatile("" : "+v"(f[1][e][t]));
    }
  };
  arrive(std::integral_constant<int, (SLOTS - 1) * R::LOADS>{});
#pragma unroll
  for (int e = 0; e < 4; ++e) {
#pragma unroll
    for (int t = 0; t < FRAGS; ++t) read(0, e, t, 0);
  }
  const int range_slices = range_of(k) / SLICE;
  int range_end = min(range_slices, count);
  // 4 NT instructions over one half's fragments, the other half's read beside them in the order in which they are wanted.
  auto multiply = [&](int half, int read_slot, auto LOADING, int i, int free) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
#pragma unroll
      for (int b = 0; b < NT; ++b) {
        acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(f[half][e][b], f[half][e][NT], acc[b], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < FRAGS; ++t)
          if (t / 2 * NT / ((FRAGS + 1) / 2) == b) read(half ^ 1, e, t, read_slot);
        if constexpr (decltype(LOADING)::value) {
#pragma unroll
          for (int j = 0; j < R::LOADS; ++j)
            if (j * 4 * NT / R::LOADS == e * NT + b) load(j, i, free);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };
  // Slice `it` lies in slot SLOT_NOW, its first half's fragments are in registers.
  auto round = [&](int it, auto SLOT_NOW) __attribute__((always_inline)) {
    constexpr int slot = decltype(SLOT_NOW)::value, next = (slot + 1) % SLOTS;
    multiply(0, slot, std::false_type{}, 0, 0);
    // This wavefront has all of slice `it` in registers, and its loads of it + 1 have landed; behind the barrier both hold for the workgroup.
    held();
    arrive(std::integral_constant<int, (SLOTS - 2) * R::LOADS>{});
    multiply(1, next, std::true_type{}, it + SLOTS, slot);
    if (it + 1 == range_end) {  // the same for every thread
#pragma unroll
      for (int b = 0; b < NT; ++b) sum[b] += acc[b], acc[b] = gp_f32x4{0.f, 0.f, 0.f, 0.f};
      range_end = min(range_end + range_slices, count);
    }
  };
  static_assert(SLOTS == 4, "a turn of the loop goes once round the ring");
  for (int it = 0; it < count; it += SLOTS) {
    round(it, std::integral_constant<int, 0>{});
    if (it + 1 >= count) break;
    round(it + 1, std::integral_constant<int, 1>{});
    if (it + 2 >= count) break;
    round(it + 2, std::integral_constant<int, 2>{});
    if (it + 3 >= count) break;
    round(it + 3, std::integral_constant<int, 3>{});
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // loads past the end

  // sum[b][i]: activation row 16 wave + r, weight row 16 b + 4 g + i.
  const int row = m0 + 16 * wave + r;
  if (row >= m) return;
#pragma unroll
  for (int b = 0; b < NT; ++b) {
    const int col = n0 + 16 * b + 4 * g;
    if (col >= n) continue;
    if (bias) {
#pragma unroll
      for (int i = 0; i < 4; ++i) sum[b][i] += bias[col + i];
    }
    if (glu.gated) {
      *reinterpret_cast<float2*>(y + (size_t)row * y_stride + col / 2) =
          make_float2(gated_unit(sum[b][0], sum[b][1], glu.rule), gated_unit(sum[b][2], sum[b][3], glu.rule));
    } else {
      *reinterpret_cast<gp_f32x4*>(y + (size_t)row * y_stride + col) = sum[b];
    }
  }
}

template <int NT>
__global__ void __launch_bounds__(256, 2)
gemm_plain_block_kernel(const float* __restrict__ x, const float* __restrict__ w, int x_stride, int m, int n, int k, int m_tiles, int n_tiles,
                        float* __restrict__ y, const float* __restrict__ bias, long y_stride, PlainGlu glu) {
  extern __shared__ __attribute__((aligned(16))) float block_ring[];
  plain_block<NT>((lds_f32*)block_ring, (const lds_f32*)block_ring, y, x, w, bias, m, n, k, x_stride, y_stride, m_tiles, n_tiles, glu);
}

template <int NT>
int launch_plain_block(void* y, const void* x, const void* w, const void* bias, int m, int n, int k, long x_stride, long y_stride,
                       PlainGlu glu, hipStream_t stream) {
  static bool raised = false;  // per process; the attribute belongs to the kernel
  if (!raised) {
    if (hipFuncSetAttribute((const void*)gemm_plain_block_kernel<NT>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)PlainRing<NT>::BYTES) != hipSuccess)
      return TS_ERR_LAUNCH;
    raised = true;
  }
  const long m_tiles = ceil_of(m, 64), n_tiles = ceil_of(n, 16 * NT), ids = ceil_of(m_tiles * n_tiles, GP_DIES) * GP_DIES;
  if (ids > 0x7fffffffL) return TS_ERR_SHAPE;
  hipLaunchKernelGGL((gemm_plain_block_kernel<NT>), dim3((unsigned)ids), dim3(256), (PlainRing<NT>::BYTES), stream, (const float*)x,
                     (const float*)w, (int)x_stride, m, n, k, (int)m_tiles, (int)n_tiles, (float*)y, (const float*)bias, y_stride, glu);
  return ts_launch_status();
}

// Which layout runs a product: the one whose workgroups are through soonest, a round of one on every compute unit at a time.
// Half microseconds at K = 3,584, measured over q|k|v, o, gate|up and the head of the 7B shape at 1 to 2,048 rows (all
// grow with K alike): a round of workgroups of 16 x 16 outputs whose operands go through LDS takes 9.5 us (read straight from
// memory 13), of 16 x 32 17.5 (24), 32 x 16 15 (22), 32 x 32 24.5 (37) (more weight rows a wavefront read the
// activations less often, fewer give more workgroups), of 64 x 64 70, of 128 x 128 240, and the first round a little more.  Where the block
// layout takes the operands: a round of 64 x 16 NT 13 NT, 3 more where a compute unit holds one (NT 7 and more); 64 x 64 and 128 x 128
// are not asked for there (500 rows, us, before -> NT: gate|up 1,145 -> 961, down 671 -> 486, o 131 -> 99, q|k|v 187 -> 121; 128 rows of o 42 -> 31).
enum PlainKind { FEW_1_1, FEW_1_2, FEW_2_1, FEW_2_2, TILES_64, TILES_128, BLOCK };  // BLOCK + NT

inline int plain_kind(int m, int n, bool stream_reads, bool block) {
  static const struct {
    PlainKind kind;
    int rows, cols, start[2], round[2];  // straight from memory, through LDS
  } layouts[] = {{FEW_1_1, 16, 16, {6, 6}, {26, 19}}, {FEW_1_2, 16, 32, {0, 2}, {48, 35}}, {FEW_2_1, 32, 16, {6, 8}, {44, 30}},
                 {FEW_2_2, 32, 32, {0, 4}, {74, 49}}, {TILES_64, 64, 64, {24, 10}, {130, 140}}, {TILES_128, 128, 128, {0, 0}, {470, 480}}};
  int best = TILES_128;
  long least = -1, filled = 1L << 40;
  for (const auto& l : layouts) {
    if (l.cols < 64 ? ceil_of(m, l.rows) > 65535 : block) continue;  // more tiles of rows than their grids take
    const long workgroups = ceil_of(m, l.rows) * ceil_of(n, l.cols);
    const long cost = l.start[stream_reads] + l.round[stream_reads] * ceil_of(workgroups, GP_UNITS);
    if (least < 0 || cost < least) best = l.kind, least = cost, filled = l.start[1] + l.round[1] * max(workgroups, (long)GP_UNITS) / GP_UNITS;
  }
  // A last round of the few rows' layouts that is nearly empty is nearly over at once (48 rows of 4,608, 432 workgroups of 16 x 32: 26 us, one
  // round of 64 x 32 32).  No tile of the block layout is through before 64, so what is sooner is not compared.
  for (int nt = 2; block && nt <= 9 && filled > 64; ++nt) {
    const long rounds = ceil_of(ceil_of(ceil_of(m, 64) * ceil_of(n, 16 * nt), GP_DIES), GP_UNITS / GP_DIES);
    const long cost = 8 + rounds * (26 * nt + (nt == 2 ? 4 : nt < 7 ? 0 : 6));
    if (cost < filled) best = BLOCK + nt, filled = cost;
  }
  return best;
}

template <typename TIn, typename TOut>
int launch_plain(void* y, const void* x, const void* w, const void* bias, int m, int n, int k, long x_stride,
                 long y_stride, int tile, PlainGlu glu, hipStream_t stream) {
  const size_t quad = 4 * sizeof(TIn);
  const bool vec = k % 4 == 0 && x_stride % 4 == 0 && (uintptr_t)x % quad == 0 && (uintptr_t)w % quad == 0 &&
                   x_stride < (1L << 25) && k < (1 << 25);
  // 32-bit operands whose rows lie within the 31 bits of a buffer's offsets go through LDS.
  const bool stream_reads = sizeof(TIn) == 4 && vec && x_stride < (1L << 24) && k < (1 << 24);
#define TS_PLAIN_ARGS (TOut*)y, (const TIn*)x, (const TIn*)w, (const TIn*)bias, m, n, k, x_stride, y_stride
#define TS_PLAIN_TILED(T, BK, V)                                                                                      \
  do {                                                                                                               \
    const int m_tiles = (int)ceil_of(m, 64 * T), n_tiles = (int)ceil_of(n, 64 * T);                                  \
    const long ids = ceil_of(n_tiles, GP_DIES) * GP_DIES * m_tiles;                                                  \
    if (ids > 0x7fffffffL) return TS_ERR_SHAPE;                                                                      \
    hipLaunchKernelGGL((gemm_plain_kernel<T, T, BK, V, TIn, TOut>), dim3((unsigned)ids), dim3(256), 0, stream,       \
                       TS_PLAIN_ARGS, m_tiles, n_tiles);                                                             \
  } while (0)
#define TS_PLAIN_FEW(MT, NT, AHEAD)                                                                                   \
  do {                                                                                                               \
    dim3 grid((unsigned)ceil_of(n, 16 * NT), (unsigned)ceil_of(m, 16 * MT));                                         \
    if (stream_reads)                                                                                                \
      return grid.y == 1 ? launch_stream<MT, NT, true>(y, x, w, bias, m, n, k, x_stride, y_stride, grid, glu, stream)     \
                         : launch_stream<MT, NT, false>(y, x, w, bias, m, n, k, x_stride, y_stride, grid, glu, stream);   \
    if (vec && sizeof(TIn) == 2)                                                                                     \
      hipLaunchKernelGGL((gemm_plain_few_rows_kernel<MT, NT, AHEAD, sizeof(TIn) == 2, TIn, TOut>), grid, dim3(256),  \
                         0, stream, TS_PLAIN_ARGS);                                                                  \
    else                                                                                                             \
      hipLaunchKernelGGL((gemm_plain_few_rows_kernel<MT, NT, 2, false, TIn, TOut>), grid, dim3(256), 0, stream,      \
                         TS_PLAIN_ARGS);                                                                             \
  } while (0)
  if constexpr (sizeof(TIn) == 2) {  // (32-bit: 3,584 x 3,583 at 16 rows 41 us by the layouts below, 51 by this one)
    if (!vec && m <= UNEVEN_MOST_ROWS) {
      const dim3 grid((unsigned)ceil_of(n, UNEVEN_TILE), (unsigned)ceil_of(m, UNEVEN_TILE));
      hipLaunchKernelGGL((gemm_plain_uneven_kernel<TOut>), grid, dim3(256), 0, stream, TS_PLAIN_ARGS);
      return ts_launch_status();
    }
  }
  // The block layout's stores and loads are 16 bytes, its slices whole, its tiles' rows within 31 bits of the first one.
  const bool block = stream_reads && k % 32 == 0 && n % 4 == 0 && y_stride % (glu.gated ? 2 : 4) == 0 && (uintptr_t)y % 16 == 0 && x_stride < (1L << 21) &&
                     k < (1 << 21);
  if ((tile != 0 && (!block || tile < 2 || tile > 9)) || (glu.gated && !block)) return TS_ERR_SHAPE;
  const int kind = tile ? BLOCK + tile : plain_kind(m, n, stream_reads, block);
  if constexpr (sizeof(TIn) == 4 && sizeof(TOut) == 4) {
#define TS_PLAIN_BLOCK(NT) \
  if (kind == BLOCK + NT) return launch_plain_block<NT>(y, x, w, bias, m, n, k, x_stride, y_stride, glu, stream)
    TS_PLAIN_BLOCK(2);
    TS_PLAIN_BLOCK(3);
    TS_PLAIN_BLOCK(4);
    TS_PLAIN_BLOCK(5);
    TS_PLAIN_BLOCK(6);
    TS_PLAIN_BLOCK(7);
    TS_PLAIN_BLOCK(8);
    TS_PLAIN_BLOCK(9);
#undef TS_PLAIN_BLOCK
  }
  switch (kind) {
    case FEW_1_1:
      TS_PLAIN_FEW(1, 1, 3);
      break;
    case FEW_1_2:
      TS_PLAIN_FEW(1, 2, 3);
      break;
    case FEW_2_1:
      TS_PLAIN_FEW(2, 1, 3);
      break;
    case FEW_2_2:
      TS_PLAIN_FEW(2, 2, 2);
      break;
    case TILES_64:
      if (vec) TS_PLAIN_TILED(1, 32, true); else TS_PLAIN_TILED(1, 32, false);
      break;
    case TILES_128:
      if (vec) TS_PLAIN_TILED(2, 16, true); else TS_PLAIN_TILED(2, 16, false);
      break;
  }
#undef TS_PLAIN_FEW
#undef TS_PLAIN_TILED
#undef TS_PLAIN_ARGS
  return ts_launch_status();
}

}  // namespace

// dtype: type of x, w and bias.  out_f32 != 0: y is float whatever dtype is.  tile: 0, or 2 to 9, tiles of 64 x 16 tile outputs by the block
// layout, where it takes the operands.
// gated != 0 (32-bit, n and k multiples of 4 and 32, operands and strides on 16 bytes): y is [m, n / 2], the gated unit (common.hpp) of rows that
// alternate gate, up.
extern "C" int ts_gemm_plain(void* y, const void* x, const void* w, const void* bias, int m, int n,
                             int k, long x_stride, long y_stride, int dtype, int out_f32, int tile, int gated, float steepness, float limit,
                             float up_shift, float cubic, hipStream_t stream) {
  if (m == 0 || n == 0) return TS_OK;
  if (!y || !x || !w || k < 1 || x_stride < k || y_stride < (gated ? n / 2 : n)) return TS_ERR_ARG;
  if (ceil_of(m, 64) > 65535) return TS_ERR_SHAPE;
  const PlainGlu glu = {gated != 0, {steepness, limit, up_shift, cubic}};
  if (dtype == TS_F32) return launch_plain<float, float>(y, x, w, bias, m, n, k, x_stride, y_stride, tile, glu, stream);
  if (dtype != TS_BF16) return TS_ERR_DTYPE;
  if (tile != 0 || gated) return TS_ERR_SHAPE;
  if (out_f32) return launch_plain<bf16_t, float>(y, x, w, bias, m, n, k, x_stride, y_stride, 0, glu, stream);
  return launch_plain<bf16_t, bf16_t>(y, x, w, bias, m, n, k, x_stride, y_stride, 0, glu, stream);
}
