// States that decay by one number per head and token: per head and request a 32-bit state S [N, P] that every token
// takes as
//     S <- a S + w B x^T        y = S^T C,
// with x [P] of the head, B and C [N] of the head's group (heads / groups neighbouring heads share one).  Three rules
// make a and w:
//   selective  dt = softplus(d + dt_bias), a = exp(-exp(A_log) dt), w = dt; y gets D x added   (a selective state space)
//   fixed      a is one number per head, w = 1                                                   (retention)
//   gated      log input gate i = cap tanh((i' + i_bias) / cap), log forget gate f = log sigmoid(cap tanh((f' + f_bias) /
//              cap)), a running maximum m (it starts at 0) that keeps the exponentials small: m' = max(f + m, i), a = exp(f +
//              m - m'), w = exp(i - m').  Beside S a sum n [N] takes every token as n <- a n + w B, and n . C and m' leave
//              with y: the read-out's denominator.  n is one more column of the state, whose x is 1.
// a, w, S, n, m, y and everything between them are 32-bit.  A column's N elements of the state lie side by side in the
// slot ([P][N]); n and m lie in slots of their own.
//
// x, B and C are columns of the rows `u` (type U, 32-bit partial sums where a projection left such); d, i' and f' are H
// columns each of the fused projection `proj` [T, width] of the run's type, or `splits` 32-bit partial sums.
//
// ts_decaying_walk    per (request, head, stretch of columns): the request's tokens one behind the other, the state in
//                     registers.  Single tokens, short portions, and every 32-bit run.
// Long portions of bfloat16 runs are cut into pieces of SS_PIECE tokens that run side by side on the matrix cores.  With
// c_i the sum of log a over the piece's tokens up to and including i, token j's write weighs w_j exp(s_j - t_i) at token i:
// s = t = -c for the first two rules; s_j = i_j - c_j, t_i = max(m before the piece, s_1 .. s_i), w = 1 for the third
// (m_i = c_i + t_i).  No exponent is above zero.  With t_0 what the state before the piece stands against (0, or m),
//     S_end = exp(t_0 - t_last) S_before + sum_j w_j exp(s_j - t_last) B_j x_j^T
//     y_i   = exp(t_0 - t_i) S_before^T C_i + sum_{j <= i} w_j exp(s_j - t_i) (C_i . B_j) x_j,
// (the blocked form of Dao and Gu, "Transformers are SSMs: Generalized Models and Efficient Algorithms Through
// Structured State Space Duality"), in two or three launches: ts_decaying_pass (the state before each piece, a request's
// pieces one behind the other; what the last one leaves goes to the slot), or where those would be too many rounds of workgroups or too few
// workgroups ts_decaying_pieces mode 0 (every piece's own S_end from a zero state, the pieces side by side) and ts_decaying_carry (the states
// before the pieces, elementwise); then ts_decaying_pieces mode 1 (y).  x, B and C are bfloat16 numbers, so C . B is exact products summed in 32-bit; every other factor is a
// 32-bit number that is cut into three bfloat16 numbers whose sum it is exactly, and the three products are summed
// in 32-bit: nothing of the recurrence is rounded to 16 bits.
//
// ts_heads_finish: every head's y (over its denominator) divided by its root mean square, times a gain, times a gate,
// rounded once; it also leaves the running maximum of a request's last token in the request's slot.
//
// ts_gated_group_norm: y silu(z), every one of `parts` equal parts of a row divided by its own root mean square, times
// a gain, rounded once.
#include "vec.hpp"

#include <type_traits>

#define SS_PIECE 128
#define SS_STRETCH 32
#define SS_PARTS 8  // lanes that share a column of the state in the walk

#define SS_SELECTIVE 0
#define SS_FIXED 1
#define SS_GATED 2
#define SS_NEVER -1e30  // the exponent of a token that is not there

typedef __bf16 ss_bf16x8 __attribute__((ext_vector_type(8)));
typedef float ss_f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int ss_u32x2 __attribute__((ext_vector_type(2)));

template <typename P>
__device__ __forceinline__ float ss_input(const P* p, int splits, size_t stride) {
  if (splits == 1) return to_float(p[0]);
  float s = 0.f;
  for (int first = 0; first < splits; first += 8) {
    float v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) v[j] = to_float(p[(size_t)min(first + j, splits - 1) * stride]);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (first + j < splits) s += v[j];
  }
  return s;
}

// Two at once, twice as many loads in flight.
template <typename P>
__device__ __forceinline__ void ss_input_two(const P* p, const P* q, int splits, size_t stride, float& a, float& b) {
  if (splits == 1) {
    a = to_float(p[0]);
    b = to_float(q[0]);
    return;
  }
  a = b = 0.f;
  for (int first = 0; first < splits; first += 8) {
    float v[8], w[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      v[j] = to_float(p[(size_t)min(first + j, splits - 1) * stride]);
      w[j] = to_float(q[(size_t)min(first + j, splits - 1) * stride]);
    }
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (first + j < splits) {
        a += v[j];
        b += w[j];
      }
  }
}

// The same of VEC neighbouring elements.
template <typename P, int VEC>
__device__ __forceinline__ void ss_input_vec(const P* p, int splits, size_t stride, float (&v)[VEC]) {
  load_vec<P, VEC>(p, v);
  for (int first = 1; first < splits; first += 8) {
    float more[8][VEC];
#pragma unroll
    for (int j = 0; j < 8; ++j) load_vec<P, VEC>(p + (size_t)min(first + j, splits - 1) * stride, more[j]);
#pragma unroll
    for (int j = 0; j < 8; ++j)
      if (first + j < splits) {
#pragma unroll
        for (int e = 0; e < VEC; ++e) v[e] += more[j][e];
      }
  }
}

__device__ __forceinline__ float ss_softplus(float z) { return z > 20.f ? z : log1pf(expf(z)); }

// Where a token's vectors lie in its row of `u`: x of head h from x_at + h P on, B and C of group g from b_at + g N and
// c_at + g N on.
struct SsRows {
  int splits;
  long stride;
  int width;
  int x_at, b_at, c_at;
};

// What a and w are made from: the H columns of the projection from `first` on (gated: 2 H, i' then f'), and a number
// or two per head (selective: dt_bias, A_log; fixed: the decays; gated: the two gates' biases).
struct SsGates {
  int splits;
  long stride;
  int width;
  int first;
  const float* one;
  const float* two;
  float cap;
};

__device__ __forceinline__ float ss_capped(float z, float cap) { return cap * tanhf(z / cap); }

__device__ __forceinline__ float ss_log_sigmoid(float z) { return fminf(z, 0.f) - log1pf(expf(-fabsf(z))); }

// The log gates of head h at row t.
template <typename P>
__device__ __forceinline__ void ss_log_gates(const P* proj, const SsGates& gates, int t, int h, int heads, float& in, float& forget) {
  const P* row = proj + (size_t)t * gates.width + gates.first + h;
  float i, f;
  ss_input_two(row, row + heads, gates.splits, gates.stride, i, f);
  in = ss_capped(i + gates.one[h], gates.cap);
  forget = ss_log_sigmoid(ss_capped(f + gates.two[h], gates.cap));
}

// ---------------------------------------------------------------------------------------------
// the walk
// ---------------------------------------------------------------------------------------------

// NR: state rows a thread holds (of every stretch of 4 SS_PARTS rows the four from 4 part on); COLS: columns of a
// workgroup; BATCH: tokens staged in LDS at a time.  norm [T, H, 2] (gated): n . C and the running maximum.
template <typename U, typename P, int RULE, int NR, int BATCH, int COLS>
__global__ void __launch_bounds__(SS_PARTS * COLS, NR <= 32 ? 5 : 2)
decaying_walk_kernel(float* __restrict__ state, const int* __restrict__ state_slots, const int* __restrict__ query_start_loc, int first_seq,
                     int heads, int groups, int n, int p, float* __restrict__ y, float* __restrict__ norm, float* __restrict__ sums,
                     const float* __restrict__ tops, const U* __restrict__ u, SsRows rows, const P* __restrict__ proj, SsGates gates,
                     const float* __restrict__ skip, float scale) {
  // (Fourteen words of arguments lie in registers at the start: what the state's loads want comes first.)
  constexpr int ROWS = SS_PARTS * NR, THREADS = SS_PARTS * COLS;
  __shared__ __attribute__((aligned(16))) float bs[BATCH][ROWS];
  __shared__ __attribute__((aligned(16))) float cs[BATCH][ROWS];
  __shared__ float xs[BATCH][COLS];
  __shared__ float ws[BATCH], as[BATCH], ms[BATCH];
  const int seq = first_seq + blockIdx.x, h = blockIdx.y, g = h / (heads / groups);
  const int tid = threadIdx.x, part = tid % SS_PARTS, col_in = tid / SS_PARTS;
  const int c0 = blockIdx.z * COLS, c = c0 + col_in;
  const bool summing = RULE == SS_GATED && c == p;  // the column of n
  const bool live = c < p || summing;
  int row0 = query_start_loc[seq], row_end = query_start_loc[seq + 1];
  const size_t b_at = (size_t)rows.b_at + (size_t)g * n, c_at = (size_t)rows.c_at + (size_t)g * n, x_at = (size_t)rows.x_at + (size_t)h * p;
  int slot = state_slots[seq];
  // The other arguments, the rows and the slot come with one wait.
  asm volatile("" : "+s"(slot), "+s"(row0), "+s"(row_end) : "s"(u), "s"(proj), "s"(gates.one), "s"(gates.two), "s"(skip), "s"(rows.stride), "s"(rows.width), "s"(gates.stride), "s"(gates.width));
  const int count = row_end - row0;
  const size_t owner = (size_t)slot * heads + h;
  float* held = summing ? sums + owner * n : state + (owner * p + (live ? c : 0)) * n;
  const bool quads = n % 4 == 0;
  float s[NR];
  // The loads are unconditional (rows past N, columns past P: others of the same state, dropped below), so that they are on their way
  // together: with a branch about each the compiler waited for one before it asked for the next.
  if (quads) {
#pragma unroll
    for (int x = 0; x < NR / 4; ++x) {
      const int d = x * 4 * SS_PARTS + part * 4;
      const float4 v = *reinterpret_cast<const float4*>(held + (d < n ? d : 0));
      s[4 * x] = v.x; s[4 * x + 1] = v.y; s[4 * x + 2] = v.z; s[4 * x + 3] = v.w;
    }
  } else {
#pragma unroll
    for (int e = 0; e < NR; ++e) {
      const int d = e / 4 * 4 * SS_PARTS + part * 4 + e % 4;
      s[e] = held[d < n ? d : 0];
    }
  }
  if (n < ROWS) {
#pragma unroll
    for (int e = 0; e < NR; ++e) s[e] = e / 4 * 4 * SS_PARTS + part * 4 + e % 4 < n ? s[e] : 0.f;
  }
  float rate = 0.f, d_skip = 0.f, top = 0.f;
  if (RULE == SS_SELECTIVE) d_skip = skip[h];
  if (RULE == SS_FIXED) rate = gates.one[h];
  if (RULE == SS_GATED) top = tops[owner];
  for (int base = 0; base < count; base += BATCH) {
    const int batch = min(BATCH, count - base);
    if (base > 0) __syncthreads();  // the batch before is done with what is staged
    // The gates are the third wavefront's, x the last ones', B and C begin with the first: a step of one token waits for them side by side.
    const int lane = tid - 2 * TS_WAVE;
    if (RULE == SS_SELECTIVE && lane >= 0 && lane < batch) {
      const float one = gates.one[h], two = gates.two[h];  // beside the gates' inputs: asked for before, they were waited for first
      const float dt = ss_softplus(ss_input(proj + (size_t)(row0 + base + lane) * gates.width + gates.first + h, gates.splits, gates.stride) + one);
      ws[lane] = dt;
      as[lane] = expf(-expf(two) * dt);
    }
    if (RULE == SS_FIXED && lane >= 0 && lane < batch) {
      ws[lane] = 1.f;
      as[lane] = rate;
    }
    if (RULE == SS_GATED && lane >= 0 && lane < TS_WAVE) {  // lane j takes token j's gates; the maximum passes from token to token
      float in, forget;
      ss_log_gates(proj, gates, row0 + base + min(lane, batch - 1), h, heads, in, forget);
      for (int j = 0; j < batch; ++j) {
        const float i = __shfl(in, j), f = __shfl(forget, j), next = fmaxf(f + top, i);
        if (lane == j) {
          ws[j] = expf(i - next);
          as[j] = expf(f + top - next);
          ms[j] = next;
        }
        top = next;
      }
    }
    for (int i = THREADS - 1 - tid; i < batch * COLS; i += THREADS) {
      const int j = i / COLS, cc = c0 + i % COLS;
      float v = RULE == SS_GATED && cc == p ? 1.f : 0.f;
      if (cc < p) v = ss_input(u + (size_t)(row0 + base + j) * rows.width + x_at + cc, rows.splits, rows.stride);
      xs[j][i % COLS] = v;
    }
    for (int i = tid; i < batch * ROWS; i += THREADS) {
      const int j = i / ROWS, d = i % ROWS;
      const U* row = u + (size_t)(row0 + base + j) * rows.width;
      float vb = 0.f, vc = 0.f;
      if (d < n) ss_input_two(row + b_at + d, row + c_at + d, rows.splits, rows.stride, vb, vc);
      bs[j][d] = vb;
      cs[j][d] = vc;
    }
    __syncthreads();
    for (int j = 0; j < batch; ++j) {
      const float a = as[j], xv = xs[j][col_in], dx = ws[j] * xv;
      float r[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int x = 0; x < NR / 4; ++x) {
        const float4 b4 = *reinterpret_cast<const float4*>(&bs[j][x * 4 * SS_PARTS + part * 4]);
        const float4 c4 = *reinterpret_cast<const float4*>(&cs[j][x * 4 * SS_PARTS + part * 4]);
        const int i = 4 * x;
        s[i] = fmaf(a, s[i], b4.x * dx); s[i + 1] = fmaf(a, s[i + 1], b4.y * dx);
        s[i + 2] = fmaf(a, s[i + 2], b4.z * dx); s[i + 3] = fmaf(a, s[i + 3], b4.w * dx);
        r[0] = fmaf(s[i], c4.x, r[0]); r[1] = fmaf(s[i + 1], c4.y, r[1]);
        r[2] = fmaf(s[i + 2], c4.z, r[2]); r[3] = fmaf(s[i + 3], c4.w, r[3]);
      }
      float sum = (r[0] + r[1]) + (r[2] + r[3]);
      // Over the eight lanes of the column.
      sum += lanes_moved<0xB1, 0xF>(0.f, sum);
      sum += lanes_moved<0x4E, 0xF>(0.f, sum);
      sum += lanes_moved<0x141, 0xF>(0.f, sum);
      if (live && part == 0) {
        const size_t at = (size_t)(row0 + base + j) * heads + h;
        if (summing) {
          norm[2 * at] = sum * scale;
          norm[2 * at + 1] = ms[j];
        } else {
          y[at * p + c] = RULE == SS_SELECTIVE ? fmaf(d_skip, xv, sum) : sum * scale;
        }
      }
    }
  }
  if (!live || count < 1) return;
#pragma unroll
  for (int x = 0; x < NR / 4; ++x) {
    const int d = x * 4 * SS_PARTS + part * 4;
    if (quads) {
      if (d < n) *reinterpret_cast<float4*>(held + d) = make_float4(s[4 * x], s[4 * x + 1], s[4 * x + 2], s[4 * x + 3]);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (d + e < n) held[d + e] = s[4 * x + e];
    }
  }
}

// ---------------------------------------------------------------------------------------------
// a step of single tokens with the convolution in front
// ---------------------------------------------------------------------------------------------

// The selective walk of one token a request whose x, B and C are a convolution of four taps over columns of the projection, with a bias or
// without, through silu, rounded to T (short_conv.hip: `held` [slots, 3, channels], oldest first; the same bits): every workgroup convolves the
// channels that it reads, 288 of them at 128 rows, while its part of the state travels, and a launch of 4 us between two that wait for it falls
// away.  A channel of x belongs to one workgroup, which moves it on in `held`; those of B and C, which all heads of a group read, are
// moved on by the launch behind this one (gated_group_norm_few_kernel).  proj: `splits` 32-bit partial sums, at most BATCH.
struct SsConv {
  const void* taps;  // [channels, 4] of T: x of every head, B of every group, C
  const void* bias;  // [channels] of T, or null
  int first;         // their first column of the projection
  int silu;
};

template <typename T, int NR, int BATCH>
__global__ void __launch_bounds__(256)
selective_token_kernel(float* __restrict__ state, const int* __restrict__ state_slots, const float* __restrict__ proj, float* __restrict__ held, int width,
                       int heads, int groups, int n, int p, int splits, size_t stride, SsConv conv, int dt_at, const float* __restrict__ dt_bias,
                       const float* __restrict__ a_log, const float* __restrict__ skip, float* __restrict__ y) {
  constexpr int THREADS = 256, COLS = THREADS / SS_PARTS, ROWS = SS_PARTS * NR, ITEMS = 2 * ROWS + COLS, ROUNDS = (ITEMS + THREADS - 1) / THREADS;
  __shared__ __attribute__((aligned(16))) float us[ITEMS];  // B, C, x
  __shared__ float weight, decay;
  const int t = blockIdx.x, h = blockIdx.y, g = h / (heads / groups);
  const int tid = threadIdx.x, part = tid % SS_PARTS, col_in = tid / SS_PARTS;
  const int c0 = blockIdx.z * COLS, c = c0 + col_in;
  const bool live = c < p;
  const int channels = heads * p + 2 * groups * n;
  const int slot = state_slots[t];
  float* const own = state + (((size_t)slot * heads + h) * p + (live ? c : 0)) * n;
  float* const kept = held + (size_t)slot * 3 * channels;
  const float* const row = proj + (size_t)t * width;
  // Everything is asked for at once, unconditionally (rows past N, columns past P: others', dropped below).
  float s[NR];
#pragma unroll
  for (int x = 0; x < NR / 4; ++x) {
    const int d = x * 4 * SS_PARTS + part * 4;
    const float4 v = *reinterpret_cast<const float4*>(own + (d < n ? d : 0));
    s[4 * x] = v.x; s[4 * x + 1] = v.y; s[4 * x + 2] = v.z; s[4 * x + 3] = v.w;
  }
  float in[ROUNDS][BATCH], old[ROUNDS][3];
  T taps[ROUNDS][4], add[ROUNDS];
  int channel[ROUNDS];
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int i = tid + THREADS * r;
    if (i >= ITEMS) break;
    const int d = i < 2 * ROWS ? i % ROWS : 0;
    channel[r] = i >= 2 * ROWS ? h * p + min(c0 + i - 2 * ROWS, p - 1) : heads * p + ((i < ROWS ? 0 : groups) + g) * n + min(d, n - 1);
#pragma unroll
    for (int j = 0; j < BATCH; ++j) in[r][j] = row[(size_t)min(j, splits - 1) * stride + conv.first + channel[r]];
#pragma unroll
    for (int j = 0; j < 3; ++j) old[r][j] = kept[(size_t)j * channels + channel[r]];
#pragma unroll
    for (int j = 0; j < 4; ++j) taps[r][j] = ((const T*)conv.taps)[(size_t)channel[r] * 4 + j];
    if (conv.bias) add[r] = ((const T*)conv.bias)[channel[r]];
  }
  const float d_skip = skip[h];
  if (tid == 3 * TS_WAVE) {  // (the last wavefront convolves no x, whatever NR: beside it dt took 0.7 us of a step with state rows of 64)
    const float one = dt_bias[h], two = a_log[h];
    const float dt = ss_softplus(ss_input(row + dt_at + h, splits, stride) + one);
    weight = dt;
    decay = expf(-expf(two) * dt);
  }
#pragma unroll
  for (int r = 0; r < ROUNDS; ++r) {
    const int i = tid + THREADS * r;
    if (i >= ITEMS) break;
    float mine = splits == 1 ? in[r][0] : 0.f + in[r][0];
#pragma unroll
    for (int j = 1; j < BATCH; ++j) mine = j < splits ? mine + in[r][j] : mine;
    float v = 0.f;
#pragma unroll
    for (int j = 0; j < 3; ++j) v = fmaf(to_float(taps[r][j]), old[r][j], v);
    v = fmaf(to_float(taps[r][3]), mine, v);
    if (conv.bias) v += to_float(add[r]);
    if (conv.silu) v = v / (1.f + expf(-v));
    us[i] = i < 2 * ROWS && i % ROWS >= n ? 0.f : to_float(from_float<T>(v));
    if (i >= 2 * ROWS && c0 + i - 2 * ROWS < p) {
      kept[channel[r]] = old[r][1];
      kept[(size_t)channels + channel[r]] = old[r][2];
      kept[(size_t)2 * channels + channel[r]] = mine;
    }
  }
  if (n < ROWS) {
#pragma unroll
    for (int e = 0; e < NR; ++e) s[e] = e / 4 * 4 * SS_PARTS + part * 4 + e % 4 < n ? s[e] : 0.f;
  }
  __syncthreads();
  const float a = decay, xv = us[2 * ROWS + col_in], dx = weight * xv;
  float r[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int x = 0; x < NR / 4; ++x) {
    const float4 b4 = *reinterpret_cast<const float4*>(&us[x * 4 * SS_PARTS + part * 4]);
    const float4 c4 = *reinterpret_cast<const float4*>(&us[ROWS + x * 4 * SS_PARTS + part * 4]);
    const int i = 4 * x;
    s[i] = fmaf(a, s[i], b4.x * dx); s[i + 1] = fmaf(a, s[i + 1], b4.y * dx);
    s[i + 2] = fmaf(a, s[i + 2], b4.z * dx); s[i + 3] = fmaf(a, s[i + 3], b4.w * dx);
    r[0] = fmaf(s[i], c4.x, r[0]); r[1] = fmaf(s[i + 1], c4.y, r[1]);
    r[2] = fmaf(s[i + 2], c4.z, r[2]); r[3] = fmaf(s[i + 3], c4.w, r[3]);
  }
  float sum = (r[0] + r[1]) + (r[2] + r[3]);
  sum += lanes_moved<0xB1, 0xF>(0.f, sum);
  sum += lanes_moved<0x4E, 0xF>(0.f, sum);
  sum += lanes_moved<0x141, 0xF>(0.f, sum);
  if (!live) return;
  if (part == 0) y[((size_t)t * heads + h) * p + c] = fmaf(d_skip, xv, sum);
#pragma unroll
  for (int x = 0; x < NR / 4; ++x) {
    const int d = x * 4 * SS_PARTS + part * 4;
    if (d < n) *reinterpret_cast<float4*>(own + d) = make_float4(s[4 * x], s[4 * x + 1], s[4 * x + 2], s[4 * x + 3]);
  }
}

// ---------------------------------------------------------------------------------------------
// pieces side by side on the matrix cores
// ---------------------------------------------------------------------------------------------

struct SsPiece {
  int seq;    // request of the step
  int first;  // first row
  int count;  // rows, at most SS_PIECE
  int pad;
};

// v = the sum of three bfloat16 numbers, exactly (each takes the next eight bits of the mantissa); returned as bits in
// the upper halves of the words.
__device__ __forceinline__ void ss_cut(float v, uint32_t& top, uint32_t& mid, uint32_t& low) {
  top = __float_as_uint(v) & 0xffff0000u;
  const float r1 = v - __uint_as_float(top);
  mid = __float_as_uint(r1) & 0xffff0000u;
  low = __float_as_uint(r1 - __uint_as_float(mid));
}

// The upper halves of two words side by side.
__device__ __forceinline__ uint32_t ss_pair(uint32_t lower, uint32_t upper) { return __builtin_amdgcn_perm(upper, lower, 0x07060302u); }

__device__ __forceinline__ ss_f32x4 ss_mfma(ts_u32x4 a, ts_u32x4 b, ss_f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(ss_bf16x8, a), __builtin_bit_cast(ss_bf16x8, b), c, 0, 0, 0);
}

// What a piece's tokens need of the decays: w, and the exponents s and t as two 32-bit numbers each (formed in 64-bit, so
// that a difference of two of them is good to 32-bit however long the piece has decayed).  Where s = t it is kept once.
template <int RULE>
struct SsSteps {
  static constexpr int OWN = RULE == SS_GATED ? SS_PIECE : 1;
  float w[SS_PIECE];
  float top[SS_PIECE];  // s
  float low[SS_PIECE];
  float to_top[OWN];    // t
  float to_low[OWN];
  float m[OWN];         // the running maximum
  float total;          // the sum of log a over the piece
  __device__ __forceinline__ float t_top(int i) const { return RULE == SS_GATED ? to_top[i] : top[i]; }
  __device__ __forceinline__ float t_low(int i) const { return RULE == SS_GATED ? to_low[i] : low[i]; }
  // s_j - t_i, and t_r - t_i.
  __device__ __forceinline__ float from(int j, int i) const { return (top[j] - t_top(i)) + (low[j] - t_low(i)); }
  __device__ __forceinline__ float passed(int r, int i) const { return (t_top(r) - t_top(i)) + (t_low(r) - t_low(i)); }
};

// What the projection says of a wavefront's two tokens a lane, 2 l and 2 l + 1 (rows beyond the piece: its last one's).
template <int RULE>
struct SsInputs {
  float head_one, head_two;            // the head's own
  float one[2];                        // d; i'
  float two[RULE == SS_GATED ? 2 : 1]; // f'
};

// For several pieces at once, so that their loads are on their way together.
template <int RULE, int COUNT, typename P>
__device__ __forceinline__ void ss_inputs(SsInputs<RULE> (&in)[COUNT], const P* proj, const SsGates& gates, int h, int heads, const SsPiece (&pieces)[COUNT]) {
#pragma unroll
  for (int x = 0; x < COUNT; ++x) {
    in[x].head_one = gates.one[h];
    in[x].head_two = RULE == SS_FIXED ? 0.f : gates.two[h];
  }
  if (RULE == SS_FIXED) return;
  const P* column = proj + gates.first + h;
  const int lane = threadIdx.x % TS_WAVE;
  if (gates.splits == 1) {
    P raw[COUNT][2][RULE == SS_GATED ? 2 : 1];
#pragma unroll
    for (int x = 0; x < COUNT; ++x)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const P* row = column + (size_t)(pieces[x].first + min(2 * lane + e, pieces[x].count - 1)) * gates.width;
        raw[x][e][0] = row[0];
        if (RULE == SS_GATED) raw[x][e][RULE == SS_GATED ? 1 : 0] = row[heads];
      }
#pragma unroll
    for (int x = 0; x < COUNT; ++x)
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        in[x].one[e] = to_float(raw[x][e][0]);
        if (RULE == SS_GATED) in[x].two[RULE == SS_GATED ? e : 0] = to_float(raw[x][e][RULE == SS_GATED ? 1 : 0]);
      }
    return;
  }
#pragma unroll
  for (int x = 0; x < COUNT; ++x)
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const P* row = column + (size_t)(pieces[x].first + min(2 * lane + e, pieces[x].count - 1)) * gates.width;
      if (RULE == SS_GATED) ss_input_two(row, row + heads, gates.splits, gates.stride, in[x].one[e], in[x].two[RULE == SS_GATED ? e : 0]);
      else in[x].one[e] = ss_input(row, gates.splits, gates.stride);
    }
}

template <int CONTROL, int ROW_MASK>
__device__ __forceinline__ double ss_moved(double keep, double v) {  // lanes_moved of 64 bits
  const uint64_t k = __builtin_bit_cast(uint64_t, keep), b = __builtin_bit_cast(uint64_t, v);
  const uint32_t low = __builtin_amdgcn_update_dpp((int)(uint32_t)k, (int)(uint32_t)b, CONTROL, ROW_MASK, 0xF, false);
  const uint32_t high = __builtin_amdgcn_update_dpp((int)(uint32_t)(k >> 32), (int)(uint32_t)(b >> 32), CONTROL, ROW_MASK, 0xF, false);
  return __builtin_bit_cast(double, (uint64_t)high << 32 | low);
}

// What `join` makes of a lane's value and those of the lanes before it (`none`: of no lane), in registers: every other wavefront of the
// workgroup waits for the decays, and each of the six steps through LDS took some 200 clocks.
template <typename Join>
__device__ __forceinline__ double ss_running(double v, Join join, double none) {
  v = join(ss_moved<0x111, 0xF>(none, v), v);  // row_shr 1, 2, 4, 8: the lanes before it in its row of 16
  v = join(ss_moved<0x112, 0xF>(none, v), v);
  v = join(ss_moved<0x114, 0xF>(none, v), v);
  v = join(ss_moved<0x118, 0xF>(none, v), v);
  v = join(ss_moved<0x142, 0xA>(none, v), v);  // row_bcast15 into rows 1 and 3, row_bcast31 into rows 2 and 3
  return join(ss_moved<0x143, 0xC>(none, v), v);
}

// By one wavefront: lane l takes the tokens 2 l and 2 l + 1 (beyond the piece: nothing decays, nothing is added).
// `floor`: what t starts from (gated).
template <int RULE>
__device__ __forceinline__ void ss_steps(SsSteps<RULE>& at, const SsInputs<RULE>& inputs, const SsGates& gates, double floor, int count) {
  const int lane = threadIdx.x % TS_WAVE;
  float w[2];
  double gone[2], in[2] = {0., 0.};  // log a; the log input gate
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const bool there = 2 * lane + e < count;
    if (RULE == SS_SELECTIVE) {
      w[e] = there ? ss_softplus(inputs.one[e] + inputs.head_one) : 0.f;
      gone[e] = -(double)expf(inputs.head_two) * (double)w[e];
    } else if (RULE == SS_FIXED) {
      w[e] = there ? 1.f : 0.f;
      gone[e] = there ? log((double)inputs.head_one) : 0.;
    } else {
      w[e] = there ? 1.f : 0.f;
      gone[e] = there ? (double)ss_log_sigmoid(ss_capped(inputs.two[RULE == SS_GATED ? e : 0] + inputs.head_two, gates.cap)) : 0.;
      in[e] = (double)ss_capped(inputs.one[e] + inputs.head_one, gates.cap);
    }
  }
  const double own = gone[0] + gone[1];
  const double sum = ss_running(own, [](double before, double v) { return before + v; }, 0.);
  const double c[2] = {sum - own + gone[0], sum};
  double s[2] = {-c[0], -c[1]};
  if (RULE == SS_GATED) {
#pragma unroll
    for (int e = 0; e < 2; ++e) s[e] = 2 * lane + e < count ? in[e] + s[e] : SS_NEVER;
    const double most = ss_running(fmax(s[0], s[1]), [](double before, double v) { return fmax(v, before); }, (double)SS_NEVER);
    const double before = __shfl_up(most, 1);
    const double t[2] = {fmax(fmax(lane > 0 ? before : SS_NEVER, s[0]), floor), fmax(most, floor)};
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float top = (float)t[e];
      at.to_top[2 * lane + e] = top;
      at.to_low[2 * lane + e] = (float)(t[e] - (double)top);
      at.m[2 * lane + e] = (float)(c[e] + t[e]);
    }
  }
#pragma unroll
  for (int e = 0; e < 2; ++e) {
    const float top = (float)s[e];
    at.w[2 * lane + e] = w[e];
    at.top[2 * lane + e] = top;
    at.low[2 * lane + e] = (float)(s[e] - (double)top);
  }
  if (lane == TS_WAVE - 1) at.total = (float)c[1];
}

// Rows 4 q .. 4 q + 3 (from row r0 of u, rows beyond `count` zero) of the eight columns from `col` on, turned: element
// (column e, row i) of the result.
__device__ __forceinline__ void ss_load_rows(const bf16_t* u, size_t u_width, int first, int r0, int count, size_t col, bool in, ts_u32x4 (&raw)[4]) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    raw[i] = ts_u32x4{0u, 0u, 0u, 0u};
    if (in && r0 + i < count) raw[i] = *reinterpret_cast<const ts_u32x4*>(u + (size_t)(first + r0 + i) * u_width + col);
  }
}

__device__ __forceinline__ uint32_t ss_half(ts_u32x4 v, int e) { return e & 1 ? v[e / 2] & 0xffff0000u : v[e / 2] << 16; }  // as the bits of a float

// Where mode 0 keeps token j of row r in LDS.  Rows are SS_STRETCH + 8 apart; the four chunks of eight tokens change
// places by the row's group of eight, and groups of 32 rows are 16 words further apart: so the threads that turn tokens
// and rows over, whose rows are eight apart, write to different banks.
__device__ __forceinline__ int ss_place(int r, int j) {
  return r * (SS_STRETCH + 8) + (r >> 5) * 32 + ((((j >> 3) ^ (r >> 3)) & 3) << 3) + (j & 7);
}

constexpr int ss_rows_size(int rows) { return rows * (SS_STRETCH + 8) + ((rows + 31) >> 5) * 32; }

// Mode 0.  NK: stretches of 32 state rows; PT: stretches of 16 columns.  A wavefront owns every fourth stretch of 16
// state rows and all columns: S_end^T (rows n, columns p) = sum over j of B^T (exact, LDS, tokens side by side) times
// the weighted x (three planes, LDS).  The piece is taken in stretches of
// SS_STRETCH tokens, so that four workgroups and more fit a compute unit.
// piece_state [pieces][H][P (gated: + 1, n)][N]; piece_decay [pieces][H]: the product of the piece's decays (gated: [..][2], the
// sum of log a, and the piece's own m).
template <typename P, int RULE, int NK, int PT>
__global__ void __launch_bounds__(256)
decaying_piece_state_kernel(float* __restrict__ piece_state, float* __restrict__ piece_decay, const bf16_t* __restrict__ u, SsRows rows,
                            const P* __restrict__ proj, SsGates gates, const SsPiece* __restrict__ pieces, int heads, int groups, int n,
                            int p) {
  constexpr int NP = 32 * NK, PP = 16 * PT;
  constexpr int TILES = (2 * NK + 3) / 4;  // stretches of 16 state rows a wavefront owns
  extern __shared__ __attribute__((aligned(16))) uint16_t ss_lds[];
  uint16_t* bt = ss_lds;                          // NP rows: B, tokens side by side
  uint16_t* const xw[3] = {ss_lds + ss_rows_size(NP), ss_lds + ss_rows_size(NP) + ss_rows_size(PP),
                           ss_lds + ss_rows_size(NP) + 2 * ss_rows_size(PP)};  // PP rows each: the weighted x in three planes
  __shared__ SsSteps<RULE> steps;
  __shared__ __attribute__((aligned(16))) float ends[RULE == SS_GATED ? SS_STRETCH : 4];  // the stretch's weights at the piece's end
  const int item = blockIdx.x, h = blockIdx.y, g = h / (heads / groups);
  const SsPiece piece = pieces[item];
  const int tid = threadIdx.x, wave = tid / TS_WAVE, lane = tid % TS_WAVE;
  const int lo = lane % 16, quad = lane / 16;
  const int c0 = blockIdx.z * PP;
  const size_t u_width = rows.width;
  const size_t b_at = (size_t)rows.b_at + (size_t)g * n, x_at = (size_t)rows.x_at + (size_t)h * p + c0;
  const bool summing = RULE == SS_GATED && blockIdx.z == 0;  // this workgroup also makes the piece's n, thread d row d
  float own_sum = 0.f;
  if (wave == 0) {
    SsInputs<RULE> in[1];
    const SsPiece one[1] = {piece};
    ss_inputs<RULE>(in, proj, gates, h, heads, one);
    ss_steps<RULE>(steps, in[0], gates, SS_NEVER, piece.count);
  }
  const size_t columns = RULE == SS_GATED ? p + 1 : p;
  ss_f32x4 acc[TILES][PT];
#pragma unroll
  for (int a = 0; a < TILES; ++a)
#pragma unroll
    for (int b = 0; b < PT; ++b) acc[a][b] = ss_f32x4{0.f, 0.f, 0.f, 0.f};
  for (int j0 = 0; j0 < piece.count; j0 += SS_STRETCH) {
    __syncthreads();  // the steps are there; the stretch before has been read
    for (int i = tid; i < (SS_STRETCH / 4) * (NP / 8); i += 256) {
      const int q = i / (NP / 8), d = (i % (NP / 8)) * 8;
      ts_u32x4 raw[4];
      ss_load_rows(u, u_width, piece.first, j0 + 4 * q, piece.count, b_at + d, d < n, raw);
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const ss_u32x2 four = {ss_pair(ss_half(raw[0], e), ss_half(raw[1], e)), ss_pair(ss_half(raw[2], e), ss_half(raw[3], e))};
        *reinterpret_cast<ss_u32x2*>(&bt[ss_place(d + e, 4 * q)]) = four;
      }
    }
    for (int i = tid; i < (SS_STRETCH / 2) * (PP / 8); i += 256) {  // two tokens by eight columns a thread
      const int q = i / (PP / 8), d = (i % (PP / 8)) * 8;
      ts_u32x4 raw[2];
      float w[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int j = j0 + 2 * q + k;
        raw[k] = ts_u32x4{0u, 0u, 0u, 0u};
        if (c0 + d < p && j < piece.count) raw[k] = *reinterpret_cast<const ts_u32x4*>(u + (size_t)(piece.first + j) * u_width + x_at + d);
        w[k] = steps.w[j] * expf(steps.from(j, SS_PIECE - 1));
        if (RULE == SS_GATED && d == 0) ends[2 * q + k] = w[k];
      }
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        uint32_t top[2], mid[2], low[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) ss_cut(w[k] * __uint_as_float(ss_half(raw[k], e)), top[k], mid[k], low[k]);
        const int at = ss_place(d + e, 2 * q);
        *reinterpret_cast<uint32_t*>(&xw[0][at]) = ss_pair(top[0], top[1]);
        *reinterpret_cast<uint32_t*>(&xw[1][at]) = ss_pair(mid[0], mid[1]);
        *reinterpret_cast<uint32_t*>(&xw[2][at]) = ss_pair(low[0], low[1]);
      }
    }
    __syncthreads();
    if (summing && tid < NP) {
#pragma unroll
      for (int j = 0; j < SS_STRETCH; j += 8) {
        const ts_u32x4 row = *reinterpret_cast<const ts_u32x4*>(&bt[ss_place(tid, j)]);
#pragma unroll
        for (int e = 0; e < 8; ++e) own_sum = fmaf(ends[j + e], __uint_as_float(ss_half(row, e)), own_sum);
      }
    }
    ts_u32x4 bf[TILES];
#pragma unroll
    for (int a = 0; a < TILES; ++a)
      bf[a] = *reinterpret_cast<const ts_u32x4*>(&bt[ss_place(16 * min(wave + 4 * a, 2 * NK - 1) + lo, 8 * quad)]);
#pragma unroll
    for (int plane = 2; plane >= 0; --plane)  // (the small planes first)
#pragma unroll
      for (int b = 0; b < PT; ++b) {
        const ts_u32x4 xf = *reinterpret_cast<const ts_u32x4*>(&xw[plane][ss_place(16 * b + lo, 8 * quad)]);
#pragma unroll
        for (int a = 0; a < TILES; ++a) acc[a][b] = ss_mfma(bf[a], xf, acc[a][b]);
      }
  }
#pragma unroll
  for (int a = 0; a < TILES; ++a) {
    const int d = 16 * (wave + 4 * a) + 4 * quad;
#pragma unroll
    for (int b = 0; b < PT; ++b) {
      const int c = c0 + 16 * b + lo;
      if (d < n && c < p)
        *reinterpret_cast<ss_f32x4*>(piece_state + (((size_t)item * heads + h) * columns + c) * n + d) = acc[a][b];
    }
  }
  if (summing && tid < n) piece_state[(((size_t)item * heads + h) * columns + p) * n + tid] = own_sum;
  if (blockIdx.z == 0 && tid == 0) {
    const size_t at = (size_t)item * heads + h;
    if (RULE == SS_GATED) {
      piece_decay[2 * at] = steps.total;
      piece_decay[2 * at + 1] = steps.m[SS_PIECE - 1];
    } else {
      piece_decay[at] = expf(steps.total);
    }
  }
}

// Between the modes.  A thread takes four neighbouring elements of a head's state (gated: or of n) through its request's
// pieces, and leaves what the pieces start from (gated: also m before each, in piece_top; the slot's own m stays until the
// finish, since every workgroup here reads it).
struct SsCarry {
  int slot_seq;
  int first;
  int count;
  int pad;
};

template <int RULE>
__global__ void __launch_bounds__(256)
decaying_carry_kernel(float* __restrict__ state, float* __restrict__ sums, const float* __restrict__ tops, const int* __restrict__ state_slots,
                      const SsCarry* __restrict__ carries, float* __restrict__ piece_state, const float* __restrict__ piece_decay,
                      float* __restrict__ piece_top, int heads, int n, int p) {
  const SsCarry carry = carries[blockIdx.x];
  const int h = blockIdx.y;
  const int e = 4 * (blockIdx.z * blockDim.x + threadIdx.x);
  const int own_state = n * p, per_head = RULE == SS_GATED ? own_state + n : own_state;
  if (e >= per_head) return;
  const size_t owner = (size_t)state_slots[carry.slot_seq] * heads + h;
  float* slot = RULE == SS_GATED && e >= own_state ? sums + owner * n + (e - own_state) : state + owner * own_state + e;
  float4 s = *reinterpret_cast<const float4*>(slot);
  float top = RULE == SS_GATED ? tops[owner] : 0.f;
  constexpr int AHEAD = 8;  // pieces in flight
  for (int i0 = 0; i0 < carry.count; i0 += AHEAD) {
    float4 own[AHEAD];
    float decay[AHEAD], most[AHEAD];
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      const size_t at = (size_t)(carry.first + min(i0 + i, carry.count - 1)) * heads + h;
      own[i] = *reinterpret_cast<const float4*>(piece_state + at * per_head + e);
      if (RULE == SS_GATED) {
        decay[i] = piece_decay[2 * at];
        most[i] = piece_decay[2 * at + 1];
      } else {
        decay[i] = piece_decay[at];
      }
    }
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) {
      if (i0 + i < carry.count) {
        const size_t at = (size_t)(carry.first + i0 + i) * heads + h;
        *reinterpret_cast<float4*>(piece_state + at * per_head + e) = s;
        float a = decay[i], w = 1.f;
        if (RULE == SS_GATED) {
          if (e == 0) piece_top[at] = top;
          const float next = fmaxf(decay[i] + top, most[i]);
          a = expf(decay[i] + top - next);
          w = expf(most[i] - next);
          top = next;
        }
        s.x = fmaf(a, s.x, w * own[i].x); s.y = fmaf(a, s.y, w * own[i].y);
        s.z = fmaf(a, s.z, w * own[i].z); s.w = fmaf(a, s.w, w * own[i].w);
      }
    }
  }
  *reinterpret_cast<float4*>(slot) = s;
}

// Four 16-bit numbers of sixteen lanes turned over: lane i reads row i / 4, columns 4 (i % 4) .. + 3 of a tile of 4 x 16 and gets column
// i, rows 0 .. 3.
typedef short ss_i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) ss_i16x4 ss_lds_i16x4;
typedef __attribute__((address_space(3))) uint16_t ss_lds_u16;
typedef __attribute__((address_space(3))) uint32_t ss_lds_u32;
typedef __attribute__((address_space(3))) ts_u32x4 ss_lds_u32x4;
__device__ __forceinline__ ts_u32x4 ss_read_turned(const ss_lds_u16* first, const ss_lds_u16* second) {
  const ss_u32x2 a = __builtin_bit_cast(ss_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((ss_lds_i16x4*)first));
  const ss_u32x2 b = __builtin_bit_cast(ss_u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((ss_lds_i16x4*)second));
  return ts_u32x4{a[0], a[1], b[0], b[1]};
}

// Workgroups go to the eight dies in turn: those of neighbouring heads, which share B and C, to one of them and its L2 (`turn`: a workgroup's
// number among the heads', which the grid counts first).
__device__ __forceinline__ int ss_head(int turn, int heads) { return heads % 8 == 0 ? turn % 8 * (heads / 8) + turn / 8 : turn; }

// The state before every piece, and behind the last.  A workgroup takes a request's pieces one behind the other, with ROWS rows by COLS
// columns of a head's state in the registers of its first four wavefronts: the piece's own S_end^T (rows n, columns p) = sum over j of B^T
// (exact) times the weighted x (three planes) on the matrix cores, then S = exp(t_0 - t_last) S + S_end.  So the pieces' own ends never go
// through memory and no launch puts them together.  The other four wavefronts bring the next piece to LDS meanwhile: B straight from
// memory, as its rows lie (the reads turn it over; LDS takes 30 bytes a cycle from registers, twice that from memory), x weighted and
// cut; its rows have travelled for two pieces.  The gates of up to sixteen pieces are made at the start.
// What bounds it is LDS, some 1,200 cycles a piece: so a wavefront multiplies 32 rows, and a workgroup has all rows of few columns, whose x
// it alone weighs.  16 pieces of 64 heads of 128 x 64, whose states before the pieces are 34 MB: 22.5 us where the pieces' own ends
// side by side and a launch that puts them together take 32; one piece 6.6 against 12.8 (alone, in a graph).
// piece_state [pieces][H][P (gated: + 1, n)][N]; piece_top [pieces][H] (gated): m before each piece.  The slot's own m stays until the
// finish, since every workgroup here reads it.
// The wavefronts that ask for loads to LDS read nothing of what those bring, so no wait of the compiler's own stands in their way.
#define SS_TABLE 16
template <typename P, int RULE, int ROWS>
__device__ __forceinline__ void
decaying_pass(ss_lds_u16* lds, SsSteps<RULE>* steps, float (*ends)[SS_PIECE], float* decay_of, float* most_of,
              float* __restrict__ state, float* __restrict__ sums, const float* __restrict__ tops, const int* __restrict__ state_slots,
              const SsCarry* __restrict__ carries, const SsPiece* __restrict__ pieces, float* __restrict__ piece_state,
              float* __restrict__ piece_top, const bf16_t* __restrict__ u, SsRows rows, const P* __restrict__ proj, SsGates gates, int heads,
              int groups, int n, int p) {
  constexpr int WAVES = 8, HALF = 256, COLS = 2048 / ROWS, EACH = SS_TABLE / WAVES;
  // In LDS: two pieces of x, [3 planes][tokens][COLS], then three of B, [tokens][ROWS].
  constexpr int X_PLANE = SS_PIECE * COLS, X_PIECE = 3 * X_PLANE, B_PIECE = SS_PIECE * ROWS, CHUNKS = ROWS / 8;
  constexpr int X_ITEMS = X_PLANE / 8 / HALF, B_LOADS = B_PIECE / 8 / HALF;  // of eight elements, 16 bytes
  const SsCarry carry = carries[blockIdx.y];
  if (carry.count < 1) return;
  // The request's pieces are SS_PIECE rows each, one behind the other, but for the last one's.
  const int first_row = pieces[carry.first].first, last_count = pieces[carry.first + carry.count - 1].count;
  auto piece_of = [&](int i) __attribute__((always_inline)) {
    const int at = min(i, carry.count - 1);
    return SsPiece{0, first_row + SS_PIECE * at, at == carry.count - 1 ? last_count : SS_PIECE, 0};
  };
  const int h = ss_head(blockIdx.x, heads), g = h / (heads / groups), slices = (n + ROWS - 1) / ROWS;
  const int n0 = (int)blockIdx.z % slices * ROWS, c0 = (int)blockIdx.z / slices * COLS;
  const int tid = threadIdx.x % HALF, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / TS_WAVE), lane = threadIdx.x % TS_WAVE;
  const int lo = lane % 16, quad = lane / 16;
  const bool brings = wave >= WAVES / 2;
  const int u_width = rows.width;
  const size_t owner = (size_t)state_slots[carry.slot_seq] * heads + h;
  const int columns = RULE == SS_GATED ? p + 1 : p;
  // Where a token's row of x and its chunk of eight elements of B lie: the reads of four tokens by sixteen columns of each of four
  // groups of eight tokens touch every bank twice.
  auto x_row = [](int t) __attribute__((always_inline)) { return COLS == 16 ? (t & ~12) | (t & 4) << 1 | (t & 8) >> 1 : t; };
  auto b_chunk = [](int t, int chunk) __attribute__((always_inline)) { return chunk ^ ((((t & 3) | (t >> 1 & 4)) << 1) & (CHUNKS - 1)); };

  // -- the wavefronts that bring: B of a piece on its way to LDS (tokens beyond the piece: zeros), x on its way to registers, and from there
  int b_off[B_LOADS];
#pragma unroll
  for (int y = 0; y < B_LOADS; ++y) {
    const int item = tid + HALF * y, t = item / CHUNKS, chunk = b_chunk(t, item % CHUNKS);
    b_off[y] = (t * u_width + (n0 + 8 * chunk < n ? 8 * chunk : 0)) * 2;
  }
  const uint16_t* const b_from = reinterpret_cast<const uint16_t*>(u) + rows.b_at + (size_t)g * n + n0;
  const uint16_t* const x_from = reinterpret_cast<const uint16_t*>(u) + rows.x_at + (size_t)h * p;
  auto fetch_b = [&](const SsPiece piece, int slot) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t buffer = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(b_from + (size_t)piece.first * u_width), 0,
                                                                            ((piece.count - 1) * u_width + min(n - n0, ROWS)) * 2, 0x00027000);
#pragma unroll
    for (int y = 0; y < B_LOADS; ++y)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(buffer, lds + 2 * X_PIECE + slot * B_PIECE + (HALF * y + TS_WAVE * (wave % 4)) * 8, 16, b_off[y], 0, 0, 0);
  };
  struct Part {
    ts_u32x4 x[X_ITEMS];
  };
  auto fetch_x = [&](Part& part, const SsPiece piece) __attribute__((always_inline)) {
#pragma unroll
    for (int y = 0; y < X_ITEMS; ++y) {
      // (Unconditional, of the piece's last row or the first columns where nothing is there, whose weight is 0 or whose result is not stored.)
      const int item = tid + HALF * y, t = min(item / (COLS / 8), piece.count - 1), c = c0 + item % (COLS / 8) * 8;
      part.x[y] = *reinterpret_cast<const ts_u32x4*>(x_from + (size_t)(piece.first + t) * u_width + (c < p ? c : 0));
    }
  };
  auto put = [&](int i, const Part& part) __attribute__((always_inline)) {
#pragma unroll
    for (int y = 0; y < X_ITEMS; ++y) {
      const int item = tid + HALF * y, t = item / (COLS / 8), d = item % (COLS / 8) * 8;
      const float w = ends[i % SS_TABLE][t];
      const ts_u32x4 x = RULE == SS_GATED && c0 + d == p ? ts_u32x4{0x3f80u, 0u, 0u, 0u} : part.x[y];  // (n: x is 1)
      ts_u32x4 planes[3];
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        uint32_t top[2], mid[2], low[2];
#pragma unroll
        for (int k = 0; k < 2; ++k) ss_cut(w * __uint_as_float(k ? x[e] & 0xffff0000u : x[e] << 16), top[k], mid[k], low[k]);
        planes[0][e] = ss_pair(top[0], top[1]);
        planes[1][e] = ss_pair(mid[0], mid[1]);
        planes[2][e] = ss_pair(low[0], low[1]);
      }
#pragma unroll
      for (int plane = 0; plane < 3; ++plane)
        *(ss_lds_u32x4*)(lds + i % 2 * X_PIECE + plane * X_PLANE + x_row(t) * COLS + d) = planes[plane];
    }
  };
  Part ahead[2];
  if (brings) {
    fetch_x(ahead[0], piece_of(0));
    fetch_b(piece_of(0), 0);
    fetch_x(ahead[1], piece_of(1));
    fetch_b(piece_of(1), 1);
  }

  // -- the wavefronts that multiply: tiles of rows n0 + row0 + 16 a + 4 quad .. + 3, column c
  const int row0 = 32 * (wave % 4 % (ROWS / 32)), col0 = 16 * (wave % 4 / (ROWS / 32));
  const int c = c0 + col0 + lo;
  const size_t step = (size_t)heads * columns * n;
  ss_f32x4 held[2];
  bool live[2];
  float *slot[2], *before[2];
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int d = n0 + row0 + 16 * a + 4 * quad;
    live[a] = !brings && d < n && c < columns;
    slot[a] = RULE == SS_GATED && c == p ? sums + owner * n + d : state + (owner * p + c) * n + d;
    before[a] = piece_state + ((size_t)carry.first * heads + h) * columns * n + (size_t)c * n + d;
    held[a] = ss_f32x4{0.f, 0.f, 0.f, 0.f};
    if (live[a]) held[a] = *reinterpret_cast<const ss_f32x4*>(slot[a]);
  }
  float top = RULE == SS_GATED ? tops[owner] : 0.f;

  // All LDS accesses done, then the workgroup's barrier (the fence of __syncthreads would wait for the loads, too).
  auto meet = []() __attribute__((always_inline)) {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // Of piece i, whose x and B lie in LDS.
  auto multiply = [&](int i, int slot_b) __attribute__((always_inline)) {
    const int x_now = i % 2 * X_PIECE, b_now = 2 * X_PIECE + slot_b * B_PIECE;
    constexpr int STEPS = SS_PIECE / 32;
    ts_u32x4 bf[STEPS][2], xf[STEPS][3];
#pragma unroll
    for (int k = 0; k < STEPS; ++k) {
      const int t = 32 * k + 8 * quad + lo / 4;
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        const int chunk = row0 / 8 + 2 * a + lo % 4 / 2;
        const ss_lds_u16* b = lds + b_now + lo % 2 * 4;
        bf[k][a] = ss_read_turned(b + t * ROWS + 8 * b_chunk(t, chunk), b + (t + 4) * ROWS + 8 * b_chunk(t + 4, chunk));
      }
#pragma unroll
      for (int plane = 0; plane < 3; ++plane) {
        const ss_lds_u16* x = lds + x_now + plane * X_PLANE + col0 + 4 * (lo % 4);
        xf[k][plane] = ss_read_turned(x + x_row(t) * COLS, x + x_row(t + 4) * COLS);
      }
    }
    float a_of = decay_of[i % SS_TABLE], w_of = 1.f;
    const float most = RULE == SS_GATED ? most_of[i % SS_TABLE] : 0.f;
    ss_f32x4 own[2] = {ss_f32x4{0.f, 0.f, 0.f, 0.f}, ss_f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
    for (int k = 0; k < STEPS; ++k)
#pragma unroll
      for (int plane = 2; plane >= 0; --plane)  // (the small planes first)
#pragma unroll
        for (int a = 0; a < 2; ++a) own[a] = ss_mfma(bf[k][a], xf[k][plane], own[a]);
    if (RULE == SS_GATED) {
      if (threadIdx.x == 0 && blockIdx.z == 0) piece_top[(size_t)(carry.first + i) * heads + h] = top;
      const float decay = a_of, after = fmaxf(decay + top, most);
      a_of = expf(decay + top - after);
      w_of = expf(most - after);
      top = after;
    }
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      if (live[a]) *reinterpret_cast<ss_f32x4*>(before[a]) = held[a];
      before[a] += step;
#pragma unroll
      for (int e = 0; e < 4; ++e) held[a][e] = fmaf(a_of, held[a][e], w_of * own[a][e]);
    }
  };
  int slot_b = 0;  // of the piece whose turn it is
  for (int i0 = 0; i0 < carry.count; i0 += SS_TABLE) {
    const int batch = min(SS_TABLE, carry.count - i0);
    if (i0 > 0) meet();  // the table's readers are done
    if (wave < batch) {  // pieces wave, wave + 8, ..
      SsPiece of[EACH];
      SsInputs<RULE> in[EACH];
#pragma unroll
      for (int x = 0; x < EACH; ++x) of[x] = piece_of(i0 + min(wave + WAVES * x, batch - 1));
      ss_inputs<RULE>(in, proj, gates, h, heads, of);
#pragma unroll
      for (int x = 0; x < EACH; ++x) {
        const int i = wave + WAVES * x;
        if (i >= batch) break;
        SsSteps<RULE>& at = steps[wave];
        __builtin_amdgcn_wave_barrier();  // (a wavefront's accesses to LDS are in order)
        ss_steps<RULE>(at, in[x], gates, SS_NEVER, of[x].count);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int e = 0; e < 2; ++e) ends[i][2 * lane + e] = at.w[2 * lane + e] * expf(at.from(2 * lane + e, SS_PIECE - 1));
        if (lane == 0) {
          decay_of[i] = RULE == SS_GATED ? at.total : expf(at.total);
          most_of[i] = RULE == SS_GATED ? at.m[RULE == SS_GATED ? SS_PIECE - 1 : 0] : 0.f;
        }
      }
    }
    meet();
    const int until = i0 + batch;
    if (brings) {
      // Behind a piece's barrier the slots of the piece before are free, x and B.  B of piece i has landed when no more than what has been asked
      // for behind it at least, x and B of one turn, is on its way (what the next turn of the loop takes is not asked for later, and the scheduler
      // moves nothing over its barriers).
      auto bring = [&](int i, Part& part) __attribute__((always_inline)) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(B_LOADS + X_ITEMS) : "memory");
        meet();
        const int free_b = slot_b == 0 ? 2 : slot_b - 1;
        slot_b = slot_b == 2 ? 0 : slot_b + 1;
        fetch_b(piece_of(i + 2), free_b);
        if (i + 1 < until) {
          put(i + 1, part);
          fetch_x(part, piece_of(i + 3));
        }
        __builtin_amdgcn_sched_barrier(0);
      };
      put(i0, ahead[0]);
      fetch_x(ahead[0], piece_of(i0 + 2));
      __builtin_amdgcn_sched_barrier(0);
      int i = i0;
      for (; i + 1 < until; i += 2) {  // (no way out between the two: the compiler would count the loads of one of them alone)
        bring(i, ahead[1]);
        bring(i + 1, ahead[0]);
      }
      if (i < until) bring(i, ahead[1]);
    } else {
      for (int i = i0; i < until; ++i) {
        meet();
        multiply(i, slot_b);
        slot_b = slot_b == 2 ? 0 : slot_b + 1;
      }
    }
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
    if (live[a]) *reinterpret_cast<ss_f32x4*>(slot[a]) = held[a];
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // what has been asked for past the end must not come into another workgroup's LDS
}

template <typename P, int RULE, int ROWS>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2)))
decaying_pass_kernel(float* __restrict__ state, float* __restrict__ sums, const float* __restrict__ tops, const int* __restrict__ state_slots,
                     const SsCarry* __restrict__ carries, const SsPiece* __restrict__ pieces, float* __restrict__ piece_state,
                     float* __restrict__ piece_top, const bf16_t* __restrict__ u, SsRows rows, const P* __restrict__ proj, SsGates gates,
                     int heads, int groups, int n, int p) {
  extern __shared__ __attribute__((aligned(16))) uint16_t ss_lds[];
  __shared__ SsSteps<RULE> steps[8];
  __shared__ __attribute__((aligned(16))) float ends[SS_TABLE][SS_PIECE];  // the tokens' weights at their piece's end
  __shared__ float decay_of[SS_TABLE], most_of[SS_TABLE];
  decaying_pass<P, RULE, ROWS>((ss_lds_u16*)ss_lds, steps, ends, decay_of, most_of, state, sums, tops, state_slots, carries,
                               pieces, piece_state, piece_top, u, rows, proj, gates, heads, groups, n, p);
}

// Mode 1.  Wavefront w owns the tokens of the stretches w and 7 - w of sixteen (together they see as many tokens as any
// other's two).  Everything is computed turned, y^T (rows p, columns i): the weights (C_i . B_j) exp(c_i - c_j) dt_j come
// out of one product with token i on the lane and four tokens j in its registers, which is what the next product wants of
// its second operand if the tokens j are counted in that order; they never leave the registers.
// Of the tokens j before the stretch the factor is exp(t_r - t_i) times w_j exp(s_j - t_r), r the last token before
// the stretch: the first is applied to a stretch's sums once, the second comes from a table that the workgroup makes once
// (`before`: both exponents are at most zero, so nothing overflows however strong the decays are).
// n . C (gated) is the same sum without x: of the weights that a lane holds, and of n before the piece against C.
// Its loads were eight trips to memory one behind the other, and the others waited for what the first wavefront makes of the decays; C and the
// state go out together, B and x before the last of the state's products (us, 64 heads of 128 x 64: one piece 15.9 -> 12.8, 512 tokens 16.8 ->
// 14.1, 2,000 30.3 -> 27.2, 4,096 56.6 -> 47.6).  With four workgroups a unit LDS bounds it: 96 KB written and 430 KB read each.
template <typename P, int RULE, int NK, int PT>
__global__ void __launch_bounds__(256, NK <= 4 ? 4 : 2)
decaying_piece_out_kernel(float* __restrict__ y, float* __restrict__ norm, const float* __restrict__ piece_state,
                          const float* __restrict__ piece_top, const bf16_t* __restrict__ u, SsRows rows, const P* __restrict__ proj,
                          SsGates gates, const float* __restrict__ skip, float scale, const SsPiece* __restrict__ pieces, int heads,
                          int groups, int n, int p) {
  constexpr int NP = 32 * NK, PP = 16 * PT, SROW = NP + 8, XROW = SS_PIECE + 4, HALF = SS_PIECE / 2;
  extern __shared__ __attribute__((aligned(16))) uint16_t ss_lds[];
  uint16_t* planes = ss_lds;           // [2][PP][SROW]: the state before the piece, its two lower planes, then its upper one
  uint16_t* br = ss_lds;               // then [HALF][SROW]: B of half the tokens at a time
  uint16_t* xt = ss_lds + HALF * SROW; // and [PP][XROW]: x, tokens side by side
  __shared__ __attribute__((aligned(16))) SsSteps<RULE> steps;
  __shared__ __attribute__((aligned(16))) float before[SS_PIECE / 16][SS_PIECE];  // [stretch of i][j]
  const int item = blockIdx.x, h = blockIdx.y, g = h / (heads / groups);
  const SsPiece piece = pieces[item];
  const int tid = threadIdx.x, wave = tid / TS_WAVE, lane = tid % TS_WAVE;
  const int lo = lane % 16, quad = lane / 16;
  const int c0 = blockIdx.z * PP;
  const size_t u_width = rows.width;
  const size_t b_at = (size_t)rows.b_at + (size_t)g * n, c_at = (size_t)rows.c_at + (size_t)g * n, x_at = (size_t)rows.x_at + (size_t)h * p + c0;
  const int tiles[2] = {wave, 7 - wave};
  const bool summing = RULE == SS_GATED && blockIdx.z == 0;
  const float enter = RULE == SS_GATED ? piece_top[(size_t)item * heads + h] : 0.f;  // t before the piece
  SsInputs<RULE> in[1];
  // What one wavefront makes of the decays, all wait for: its loads go ahead of the others, whose queue is 4,000 clocks long, and the makers of a
  // compute unit's workgroups (256 apart) are on different SIMDs.
  const int maker = (blockIdx.y * gridDim.x + blockIdx.x) / 256 % 4;
  if (wave == maker) {
    const SsPiece one[1] = {piece};
    ss_inputs<RULE>(in, proj, gates, h, heads, one);
  }
  const size_t head_state = ((size_t)item * heads + h) * (RULE == SS_GATED ? p + 1 : p);
  const float* entering = piece_state + (head_state + c0) * n;
  auto row_bytes = [&](size_t at, int i, int d) __attribute__((always_inline)) {  // sixteen of a token's row
    return *reinterpret_cast<const ts_u32x4*>(u + (size_t)(piece.first + min(i, piece.count - 1)) * u_width + at + d);
  };
  // What the first products read is asked for at once (whatever lies past the sizes as the last one's, and dropped).
  constexpr int ITEMS = (PP * (NP / 8) + 255) / 256, B_ITEMS = HALF * (NP / 8) / 256, X_ITEMS = HALF * (PP / 8) / 256;
  ss_f32x4 raw[ITEMS][2];
#pragma unroll
  for (int x = 0; x < ITEMS; ++x) {
    const int i = tid + 256 * x, c = i / (NP / 8), d = (i % (NP / 8)) * 8;
    const float* at = entering + (size_t)min(c, p - 1 - c0) * n + (d < n ? d : 0);
    raw[x][0] = *reinterpret_cast<const ss_f32x4*>(at);
    raw[x][1] = *reinterpret_cast<const ss_f32x4*>(at + 4);
  }
  ts_u32x4 cf[2][NK];  // C of the wavefront's tokens: columns i, eight state rows a lane
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      const int i = 16 * tiles[a] + lo, d = 32 * k + 8 * quad;
      cf[a][k] = row_bytes(c_at, i, d < n ? d : 0);
    }
  __builtin_amdgcn_sched_barrier(0);
  if (wave == maker) ss_steps<RULE>(steps, in[0], gates, enter, piece.count);
  float sum_of[2] = {0.f, 0.f};  // this lane's share of n . C of its tokens
  ss_f32x4 acc[PT][2];
#pragma unroll
  for (int b = 0; b < PT; ++b)
#pragma unroll
    for (int a = 0; a < 2; ++a) acc[b][a] = ss_f32x4{0.f, 0.f, 0.f, 0.f};
  ts_u32x4 upper[ITEMS];  // the upper plane of what the thread has read of the state, while the lower ones are multiplied
#pragma unroll
  for (int x = 0; x < ITEMS; ++x) {
    const int i = tid + 256 * x, c = i / (NP / 8), d = (i % (NP / 8)) * 8;
    const bool held = c0 + c < p && d < n;
    ts_u32x4 middle, lower;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      uint32_t top[2], mid[2], low[2];
#pragma unroll
      for (int k = 0; k < 2; ++k) ss_cut(held ? raw[x][e / 2][2 * (e % 2) + k] : 0.f, top[k], mid[k], low[k]);
      upper[x][e] = ss_pair(top[0], top[1]);
      middle[e] = ss_pair(mid[0], mid[1]);
      lower[e] = ss_pair(low[0], low[1]);
    }
    if (i >= PP * (NP / 8)) continue;
    *reinterpret_cast<ts_u32x4*>(&planes[c * SROW + d]) = middle;
    *reinterpret_cast<ts_u32x4*>(&planes[(PP + c) * SROW + d]) = lower;
  }
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int k = 0; k < NK; ++k)
      if (16 * tiles[a] + lo >= piece.count || 32 * k + 8 * quad >= n) cf[a][k] = ts_u32x4{0u, 0u, 0u, 0u};
  __syncthreads();
#pragma unroll 1
  for (int i = tid; i < SS_PIECE / 16 * SS_PIECE; i += 256) {
    const int tile = i / SS_PIECE, j = i % SS_PIECE, r = 16 * tile - 1;
    if (j <= r) before[tile][j] = steps.w[j] * __expf(steps.from(j, r));
  }
  auto multiply_state = [&](int plane) __attribute__((always_inline)) {
#pragma unroll
    for (int k = 0; k < NK; ++k)
#pragma unroll
      for (int b = 0; b < PT; ++b) {
        const ts_u32x4 sf = *reinterpret_cast<const ts_u32x4*>(&planes[(plane * PP + 16 * b + lo) * SROW + 32 * k + 8 * quad]);
#pragma unroll
        for (int a = 0; a < 2; ++a) acc[b][a] = ss_mfma(sf, cf[a][k], acc[b][a]);
      }
  };
  multiply_state(1);
  multiply_state(0);
  __syncthreads();
#pragma unroll
  for (int x = 0; x < ITEMS; ++x) {
    const int i = tid + 256 * x, c = i / (NP / 8), d = (i % (NP / 8)) * 8;
    if (i < PP * (NP / 8)) *reinterpret_cast<ts_u32x4*>(&planes[c * SROW + d]) = upper[x];
  }
  // B of half of the tokens at a time, and x of all: the first half's are on their way while the upper plane is multiplied.
  ts_u32x4 bs[B_ITEMS], xs[X_ITEMS][2];
  auto fetch_b = [&](int half) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < B_ITEMS; ++x) {
      const int i = tid + 256 * x, j = half * HALF + i / (NP / 8), d = (i % (NP / 8)) * 8;
      bs[x] = row_bytes(b_at, j, d < n ? d : 0);
    }
  };
  auto put_b = [&](int half) __attribute__((always_inline)) {
#pragma unroll
    for (int x = 0; x < B_ITEMS; ++x) {
      const int i = tid + 256 * x, j = i / (NP / 8), d = (i % (NP / 8)) * 8;
      *reinterpret_cast<ts_u32x4*>(&br[j * SROW + d]) = half * HALF + j < piece.count && d < n ? bs[x] : ts_u32x4{0u, 0u, 0u, 0u};
    }
  };
  fetch_b(0);
#pragma unroll
  for (int x = 0; x < X_ITEMS; ++x)  // two tokens by eight columns a thread
#pragma unroll
    for (int k = 0; k < 2; ++k) {
      const int i = tid + 256 * x, j = 2 * (i / (PP / 8)) + k, d = (i % (PP / 8)) * 8;
      xs[x][k] = row_bytes(x_at, j, c0 + d < p ? d : 0);
    }
  __builtin_amdgcn_sched_barrier(0);
  __syncthreads();
  multiply_state(0);
  if (summing) {
    const float* held = piece_state + (head_state + p) * n;
#pragma unroll
    for (int k = 0; k < NK; ++k) {
      const int d = 32 * k + 8 * quad;
      if (d >= n) continue;
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const float v = held[d + e];
#pragma unroll
        for (int a = 0; a < 2; ++a) sum_of[a] = fmaf(v, __uint_as_float(ss_half(cf[a][k], e)), sum_of[a]);
      }
    }
  }
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int r = 16 * tiles[a] - 1;
    const float by = tiles[a] > 0 ? expf((enter - steps.t_top(r)) - steps.t_low(r)) : 1.f;
#pragma unroll
    for (int b = 0; b < PT; ++b) acc[b][a] *= by;
    sum_of[a] *= by;
  }
  __syncthreads();  // the planes have been read: their place takes what follows
  put_b(0);
#pragma unroll
  for (int x = 0; x < X_ITEMS; ++x) {
    const int i = tid + 256 * x, q = i / (PP / 8), d = (i % (PP / 8)) * 8;
#pragma unroll
    for (int k = 0; k < 2; ++k)
      if (c0 + d >= p || 2 * q + k >= piece.count) xs[x][k] = ts_u32x4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int e = 0; e < 8; ++e) *reinterpret_cast<uint32_t*>(&xt[(d + e) * XROW + 2 * q]) = ss_pair(ss_half(xs[x][0], e), ss_half(xs[x][1], e));
  }
  for (int half = 0; half * HALF < piece.count; ++half) {
    if (half > 0) {
      fetch_b(half);
      __syncthreads();  // B of the first half has been read
      put_b(half);
    }
    __syncthreads();
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const int tile = tiles[a];
      if (16 * tile >= piece.count) continue;
#pragma unroll 1
      for (int jb = 2 * half; jb < 2 * half + 2 && 2 * jb <= tile; ++jb) {
        ss_f32x4 s[2] = {ss_f32x4{0.f, 0.f, 0.f, 0.f}, ss_f32x4{0.f, 0.f, 0.f, 0.f}};  // by stretch of 16 tokens j
#pragma unroll
        for (int k = 0; k < NK; ++k)
#pragma unroll
          for (int t = 0; t < 2; ++t)
            s[t] = ss_mfma(*reinterpret_cast<const ts_u32x4*>(&br[(32 * (jb - 2 * half) + 16 * t + lo) * SROW + 32 * k + 8 * quad]), cf[a][k], s[t]);
        const int j0 = 32 * jb + 4 * quad;
        if (2 * jb + 1 < tile) {
#pragma unroll
          for (int t = 0; t < 2; ++t) s[t] *= *reinterpret_cast<const ss_f32x4*>(&before[tile][j0 + 16 * t]);
        } else {
          // The stretch's own tokens (and, of an odd one, the sixteen before it): from here on the sums are y's own.
          const int i = 16 * tile + lo;
          const float mine_top = steps.t_top(i), mine_low = steps.t_low(i);
          const float by = tile > 0 ? expf(steps.passed(16 * tile - 1, i)) : expf((enter - mine_top) - mine_low);
#pragma unroll
          for (int b = 0; b < PT; ++b) acc[b][a] *= by;
          sum_of[a] *= by;
#pragma unroll
          for (int t = 0; t < 2; ++t) {
            const ss_f32x4 tops = *reinterpret_cast<const ss_f32x4*>(&steps.top[j0 + 16 * t]);
            const ss_f32x4 lows = *reinterpret_cast<const ss_f32x4*>(&steps.low[j0 + 16 * t]);
            const ss_f32x4 ws = *reinterpret_cast<const ss_f32x4*>(&steps.w[j0 + 16 * t]);
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              // (A later token's decay is never formed: its exponent would be positive.)
              const bool seen = j0 + 16 * t + r <= i;
              const float gone = seen ? (tops[r] - mine_top) + (lows[r] - mine_low) : 0.f;
              s[t][r] = seen ? s[t][r] * ws[r] * __expf(gone) : 0.f;
            }
          }
        }
        if (summing) {
#pragma unroll
          for (int t = 0; t < 2; ++t) sum_of[a] += (s[t][0] + s[t][1]) + (s[t][2] + s[t][3]);
        }
        ts_u32x4 wf[3];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          uint32_t top[2], mid[2], low[2];
#pragma unroll
          for (int k = 0; k < 2; ++k) ss_cut(s[e / 2][2 * (e % 2) + k], top[k], mid[k], low[k]);
          wf[0][e] = ss_pair(top[0], top[1]);
          wf[1][e] = ss_pair(mid[0], mid[1]);
          wf[2][e] = ss_pair(low[0], low[1]);
        }
#pragma unroll
        for (int b = 0; b < PT; ++b) {
          const uint16_t* row = &xt[(16 * b + lo) * XROW + j0];
          const ss_u32x2 first = *reinterpret_cast<const ss_u32x2*>(row), second = *reinterpret_cast<const ss_u32x2*>(row + 16);
          const ts_u32x4 xf = {first[0], first[1], second[0], second[1]};
#pragma unroll
          for (int plane = 2; plane >= 0; --plane) acc[b][a] = ss_mfma(xf, wf[plane], acc[b][a]);
        }
      }
    }
  }
  if (summing) {
#pragma unroll
    for (int a = 0; a < 2; ++a) {
      const int i = 16 * tiles[a] + lo;
      float sum = sum_of[a];  // over the four lanes of the token
      sum += __shfl_xor(sum, 16);
      sum += __shfl_xor(sum, 32);
      if (quad == 0 && i < piece.count) {
        const size_t at = (size_t)(piece.first + i) * heads + h;
        norm[2 * at] = sum * scale;
        norm[2 * at + 1] = steps.m[i];
      }
    }
  }
  const float d_skip = RULE == SS_SELECTIVE ? skip[h] : 0.f;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int i = 16 * tiles[a] + lo;
    if (i >= piece.count) continue;
#pragma unroll
    for (int b = 0; b < PT; ++b) {
      const int c = 16 * b + 4 * quad;
      if (c0 + c >= p) continue;
      float v[4];
      if (RULE == SS_SELECTIVE) {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = fmaf(d_skip, to_float(bf16_t{xt[(c + e) * XROW + i]}), acc[b][a][e]);
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = acc[b][a][e] * scale;
      }
      store_vec<float, 4>(y + ((size_t)(piece.first + i) * heads + h) * p + c0 + c, v);
    }
  }
}

// ---------------------------------------------------------------------------------------------
// the gated norm in parts
// ---------------------------------------------------------------------------------------------
// y silu(gate) of a thread's COUNT elements (gated_near's arithmetic, common.hpp; the other form only where a wavefront has such gates).
template <int COUNT>
__device__ __forceinline__ void ss_gated(float (&y)[COUNT], const float (&gate)[COUNT]) {
  float most = 0.f;
#pragma unroll
  for (int e = 0; e < COUNT; ++e) most = fmaxf(most, fabsf(gate[e]));
  if (__ballot(!(most <= GATE_NEAR)) == 0) {
#pragma unroll
    for (int e = 0; e < COUNT; ++e) y[e] *= gated_near(gate[e], gate[e]);
  } else {
#pragma unroll
    for (int e = 0; e < COUNT; ++e) y[e] *= fabsf(gate[e]) <= GATE_NEAR ? gated_near(gate[e], gate[e]) : gated_far(gate[e], gate[e]);
  }
}

template <typename T, typename P, int VEC, int CHUNKS>
__global__ void __launch_bounds__(1024)
gated_group_norm_kernel(T* __restrict__ out, const float* __restrict__ y, const P* __restrict__ proj, int splits, size_t split_stride,
                        int width, int z_at, const T* __restrict__ gain, float eps, int parts, int size) {
  __shared__ float scratch[16];
  const int t = blockIdx.x, part = blockIdx.y;
  const size_t row = ((size_t)t * parts + part) * size;
  const P* z = proj + (size_t)t * width + z_at + (size_t)part * size;
  float v[CHUNKS][VEC];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int i = (int)(c * blockDim.x + threadIdx.x) * VEC;
#pragma unroll
    for (int e = 0; e < VEC; ++e) v[c][e] = 0.f;
    if (i < size) {
      float gate[VEC];
      ss_input_vec<P, VEC>(z + i, splits, split_stride, gate);
      load_vec<float, VEC>(y + row + i, v[c]);
      ss_gated<VEC>(v[c], gate);
#pragma unroll
      for (int e = 0; e < VEC; ++e) ss = fmaf(v[c][e], v[c][e], ss);
    }
  }
  const float by = rsqrtf(block_sum(ss, scratch) / (float)size + eps);
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int i = (int)(c * blockDim.x + threadIdx.x) * VEC;
    if (i < size) {
      float w[VEC];
      load_vec<T, VEC>(gain + (size_t)part * size + i, w);
#pragma unroll
      for (int e = 0; e < VEC; ++e) v[c][e] *= by * w[e];
      store_vec<T, VEC>(out + row + i, v[c]);
    }
  }
}

// The same bits for a prompt's many parts of up to 256 CHUNKS elements: a wavefront a part, four a workgroup, which meet nowhere; a part's quads
// and their sums lie as a workgroup's wavefronts have them above.  Parts of 512, eight a row, a workgroup / a wavefront a part with the same
// arithmetic: 1,000 rows 7.3 / 7.1 us, 2,000 (64 MB) 12.6 / 12.0, 4,096 29.0 / 23.2; four of 256, 2,000 rows 4.8 / 4.4.
template <typename T, int CHUNKS>
__global__ void __launch_bounds__(256)
gated_group_norm_rows_kernel(T* __restrict__ out, const float* __restrict__ y, const T* __restrict__ proj, int width, int z_at,
                             const T* __restrict__ gain, float eps, int parts, int size, int items) {
  const int item = blockIdx.x * 4 + threadIdx.x / TS_WAVE, lane = threadIdx.x % TS_WAVE;
  if (item >= items) return;
  const int t = item / parts, part = item - t * parts;
  const size_t row = (size_t)item * size;
  const T* z = proj + (size_t)t * width + z_at + (size_t)part * size;
  float v[CHUNKS][4], gate[CHUNKS][4], w[CHUNKS][4];
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int i = min(4 * (c * TS_WAVE + lane), size - 4);
    load_vec<T, 4>(z + i, gate[c]);
    load_vec<float, 4>(y + row + i, v[c]);
    load_vec<T, 4>(gain + (size_t)part * size + i, w[c]);
  }
  float total = 0.f;
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const bool in = 4 * (c * TS_WAVE + lane) < size;
    float ss = 0.f;
    ss_gated<4>(v[c], gate[c]);
#pragma unroll
    for (int e = 0; e < 4; ++e) ss = in ? fmaf(v[c][e], v[c][e], ss) : ss;
    total += wave_sum(ss);
  }
  const float by = rsqrtf(total / (float)size + eps);
#pragma unroll
  for (int c = 0; c < CHUNKS; ++c) {
    const int i = 4 * (c * TS_WAVE + lane);
    if (i >= size) continue;
#pragma unroll
    for (int e = 0; e < 4; ++e) v[c][e] *= by * w[c][e];
    store_vec<T, 4>(out + row + i, v[c]);
  }
}

// The same bits for a step of few parts of up to 1,024 elements, at most BATCH partial sums: everything a part needs is asked for at once,
// and the code is short and straight (other kernels of a recorded step have put it out of the instruction cache).
// MOVES: the workgroups behind the parts' move the channels on that selective_token_kernel, the launch before, has left as they were:
// `moved` of them from `from` on, of `channels`.
struct SsMoves {
  float* held;  // [slots, 3, channels]
  const int* state_slots;
  int channels;
  int from;
  int moved;
  int first;    // the channels' first column of the projection
};
template <typename T, typename P, int THREADS, int BATCH, bool MOVES = false>
__global__ void __launch_bounds__(THREADS)
gated_group_norm_few_kernel(const P* proj, const float* y, const T* gain, T* out, int splits, int width, size_t split_stride, int z_at,
                            int parts, int size, float eps, SsMoves moves) {
  __shared__ __attribute__((aligned(16))) float scratch[(THREADS / TS_WAVE + 3) / 4 * 4];
  const int t = blockIdx.x, part = blockIdx.y;
  if (MOVES && part >= parts) {
    const int i = (part - parts) * THREADS + threadIdx.x, channel = moves.from + min(i, moves.moved - 1);
    const P* in = proj + (size_t)t * width + moves.first + channel;
    float* kept = moves.held + (size_t)moves.state_slots[t] * 3 * moves.channels + channel;
    float v[BATCH];
#pragma unroll
    for (int j = 0; j < BATCH; ++j) v[j] = to_float(in[(size_t)min(j, splits - 1) * split_stride]);
    const float one = kept[moves.channels], two = kept[(size_t)2 * moves.channels];
    float mine = splits == 1 ? v[0] : 0.f + v[0];
#pragma unroll
    for (int j = 1; j < BATCH; ++j) mine = j < splits ? mine + v[j] : mine;
    if (i >= moves.moved) return;
    kept[0] = one;
    kept[moves.channels] = two;
    kept[(size_t)2 * moves.channels] = mine;
    return;
  }
  const size_t row = ((size_t)t * parts + part) * size;
  const bool in = 4 * (int)threadIdx.x < size;
  const int i = min(4 * (int)threadIdx.x, size - 4);
  const P* z = proj + (size_t)t * width + z_at + (size_t)part * size + i;
  float gates[BATCH][4], v[4], w[4];
#pragma unroll
  for (int j = 0; j < BATCH; ++j) load_vec<P, 4>(z + (size_t)min(j, splits - 1) * split_stride, gates[j]);
  load_vec<float, 4>(y + row + i, v);
  load_vec<T, 4>(gain + (size_t)part * size + i, w);
  asm volatile("" ::: "memory");  // all of them on their way here
  float ss = 0.f, gate[4];
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    gate[e] = gates[0][e];
#pragma unroll
    for (int j = 1; j < BATCH; ++j) gate[e] = j < splits ? gate[e] + gates[j][e] : gate[e];
  }
  ss_gated<4>(v, gate);
#pragma unroll
  for (int e = 0; e < 4; ++e) ss = in ? fmaf(v[e], v[e], ss) : ss;
  const float by = rsqrtf(block_sum_of<THREADS>(ss, scratch) / (float)size + eps);
  if (!in) return;
#pragma unroll
  for (int e = 0; e < 4; ++e) v[e] *= by * w[e];
  store_vec<T, 4>(out + row + i, v);
}

// ---------------------------------------------------------------------------------------------
// the finish
// ---------------------------------------------------------------------------------------------

// One wavefront per (token, head): o = y / (max(|n . C|, exp(-m)) + 1e-6) where `norm` holds (n . C, m) (else o = y), divided
// by its root mean square, times a gain [H P] (null: none), times silu or sigmoid of the gate (columns gate_at + h P of the
// projection), times scale.  m of a request's last token goes to the request's slot.
template <typename T, typename P, int VEC>
__global__ void __launch_bounds__(256)
heads_finish_kernel(T* __restrict__ out, size_t out_stride, const float* __restrict__ y, const float* __restrict__ norm,
                    const P* __restrict__ proj, int splits, size_t split_stride, int width, int gate_at, const T* __restrict__ gain,
                    int sigmoid, float eps, float scale, float* __restrict__ tops, const int* __restrict__ state_slots,
                    const int* __restrict__ token_seq, const int* __restrict__ query_start_loc, long items, int heads, int p) {
  const long item = (long)blockIdx.x * 4 + threadIdx.x / TS_WAVE;
  const int lane = threadIdx.x % TS_WAVE;
  if (item >= items) return;  // a whole wavefront leaves: the sums below are per wavefront
  const int t = (int)(item / heads), h = (int)(item % heads);
  float inv = 1.f;
  if (norm) {
    const float m = norm[2 * item + 1];
    inv = 1.f / (fmaxf(fabsf(norm[2 * item]), expf(-m)) + 1e-6f);
    const int seq = token_seq[t];
    if (lane == 0 && t + 1 == query_start_loc[seq + 1]) tops[(size_t)state_slots[seq] * heads + h] = m;
  }
  const float* row = y + (size_t)item * p;
  const P* gates = proj + (size_t)t * width + gate_at + (size_t)h * p;
  T* to = out + (size_t)t * out_stride + (size_t)h * p;
  // A wavefront's first HELD turns stay in registers, the gates asked for before the sum is waited for.
  constexpr int HELD = 2;
  float v[HELD][VEC], z[HELD][VEC];
  float ss = 0.f;
#pragma unroll
  for (int c = 0; c < HELD; ++c) {
    const int i = (c * TS_WAVE + lane) * VEC;
    if (i >= p) continue;
    load_vec<float, VEC>(row + i, v[c]);
    ss_input_vec<P, VEC>(gates + i, splits, split_stride, z[c]);
#pragma unroll
    for (int e = 0; e < VEC; ++e) ss = fmaf(v[c][e] * inv, v[c][e] * inv, ss);
  }
  for (int i = (HELD * TS_WAVE + lane) * VEC; i < p; i += TS_WAVE * VEC) {
    float more[VEC];
    load_vec<float, VEC>(row + i, more);
#pragma unroll
    for (int e = 0; e < VEC; ++e) ss = fmaf(more[e] * inv, more[e] * inv, ss);
  }
  const float by = inv * rsqrtf(wave_sum(ss) / (float)p + eps) * scale;
  auto leave = [&](int i, float (&value)[VEC], const float (&gate)[VEC]) __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < VEC; ++e) value[e] *= by * ((sigmoid ? 1.f : gate[e]) / (1.f + expf(-gate[e])));
    if (gain) {
      float w[VEC];
      load_vec<T, VEC>(gain + (size_t)h * p + i, w);
#pragma unroll
      for (int e = 0; e < VEC; ++e) value[e] *= w[e];
    }
    store_vec<T, VEC>(to + i, value);
  };
#pragma unroll
  for (int c = 0; c < HELD; ++c) {
    const int i = (c * TS_WAVE + lane) * VEC;
    if (i < p) leave(i, v[c], z[c]);
  }
  for (int i = (HELD * TS_WAVE + lane) * VEC; i < p; i += TS_WAVE * VEC) {
    float more[VEC], gate[VEC];
    load_vec<float, VEC>(row + i, more);
    ss_input_vec<P, VEC>(gates + i, splits, split_stride, gate);
    leave(i, more, gate);
  }
}

// ---------------------------------------------------------------------------------------------
// entry points
// ---------------------------------------------------------------------------------------------

static bool ss_sizes_ok(int rule, const SsRows& rows, const SsGates& gates, int heads, int groups, int n, int p) {
  if (heads < 1 || heads > 65535 || groups < 1 || heads % groups != 0 || n < 1 || n > 512 || p < 1 || p > 65534) return false;
  if (rows.splits < 1 || rows.x_at < 0 || rows.b_at < 0 || rows.c_at < 0 || (long)rows.x_at + (long)heads * p > rows.width ||
      (long)rows.b_at + (long)groups * n > rows.width || (long)rows.c_at + (long)groups * n > rows.width)
    return false;
  const int columns = rule == SS_FIXED ? 0 : rule == SS_GATED ? 2 * heads : heads;
  return gates.splits >= 1 && gates.first >= 0 && (long)gates.first + columns <= gates.width;
}

static bool ss_rule_ok(int rule, const SsGates& gates, const void* proj, const void* skip, const void* norm, const void* sums, const void* tops) {
  if (!gates.one || (rule != SS_FIXED && (!gates.two || !proj))) return false;
  if (rule == SS_SELECTIVE) return skip != nullptr;
  if (rule == SS_GATED) return norm && sums && tops && gates.cap > 0.f;
  return rule == SS_FIXED;
}

// u_f32: u is 32-bit (`u_splits` partial sums of it), else bfloat16; dtype, in_f32: as everywhere (the projection's type).
// rule: SS_SELECTIVE, SS_FIXED (reads no projection), SS_GATED (norm, sums, tops).
extern "C" int ts_decaying_walk(float* y, float* norm, float* state, float* sums, const float* tops, const void* u, int u_f32, int u_splits,
                                long u_stride, int u_width, int x_at, int b_at, int c_at, const void* proj, int in_f32, int splits,
                                long split_stride, int width, int first_gate, const float* one, const float* two, float cap,
                                const float* skip, float scale, const int* state_slots, const int* query_start_loc, int first_seq,
                                int num_seqs, int heads, int groups, int n, int p, int rule, int dtype, hipStream_t stream) {
  if (num_seqs == 0) return TS_OK;
  const SsRows rows = {u_splits, u_stride, u_width, x_at, b_at, c_at};
  const SsGates gates = {splits, split_stride, width, first_gate, one, two, cap};
  if (!y || !state || !u || !state_slots || !query_start_loc || !ss_rule_ok(rule, gates, proj, skip, norm, sums, tops)) return TS_ERR_ARG;
  if (!ss_sizes_ok(rule, rows, gates, heads, groups, n, p)) return TS_ERR_SHAPE;
  const int columns = rule == SS_GATED ? p + 1 : p;
#define SS_GO(U, P, RULE, NR, BATCH, COLS)                                                                                            \
  hipLaunchKernelGGL((decaying_walk_kernel<U, P, RULE, NR, BATCH, COLS>), dim3(num_seqs, heads, (columns + COLS - 1) / COLS),         \
                     dim3(SS_PARTS * COLS), 0, stream, state, state_slots, query_start_loc, first_seq, heads, groups, n, p, y, norm,  \
                     sums, tops, (const U*)u, rows, (const P*)proj, gates, skip, scale)
#define SS_SIZES(U, P, RULE)                                     \
  do {                                                           \
    if (n <= 32) SS_GO(U, P, RULE, 4, 8, 32);                    \
    else if (n <= 64) SS_GO(U, P, RULE, 8, 8, 32);               \
    else if (n <= 128) SS_GO(U, P, RULE, 16, 8, 32);             \
    else if (n <= 256) SS_GO(U, P, RULE, 32, 4, 32);             \
    else SS_GO(U, P, RULE, 64, 4, 32);                           \
  } while (0)
  const bool half = dtype == TS_BF16 && !u_f32;
  if (dtype != TS_F32 && dtype != TS_BF16) return TS_ERR_DTYPE;
  if (dtype == TS_F32 && !u_f32) return TS_ERR_DTYPE;
  if (half && u_splits != 1) return TS_ERR_ARG;
  if (rule == SS_SELECTIVE) {
    if (dtype == TS_F32) SS_SIZES(float, float, SS_SELECTIVE);
    else if (half && in_f32) SS_SIZES(bf16_t, float, SS_SELECTIVE);
    else if (half) SS_SIZES(bf16_t, bf16_t, SS_SELECTIVE);
    else return TS_ERR_DTYPE;
  } else if (rule == SS_FIXED) {
    if (u_f32) SS_SIZES(float, float, SS_FIXED);
    else SS_SIZES(bf16_t, bf16_t, SS_FIXED);
  } else {  // (the vectors and the gates' inputs lie in one projection)
    if (u_f32 != (in_f32 || dtype == TS_F32)) return TS_ERR_DTYPE;
    if (u_f32) SS_SIZES(float, float, SS_GATED);
    else SS_SIZES(bf16_t, bf16_t, SS_GATED);
  }
#undef SS_SIZES
#undef SS_GO
  return ts_launch_status();
}

template <typename P, int RULE, int NK, int PT>
static int ss_pieces_launch(int mode, float* y, float* norm, float* piece_state, float* piece_decay, const float* piece_top, const void* u,
                            SsRows rows, const void* proj, SsGates gates, const float* skip, float scale, const void* pieces,
                            int num_pieces, int heads, int groups, int n, int p, hipStream_t stream) {
  const dim3 grid(num_pieces, heads, (p + 16 * PT - 1) / (16 * PT));
  if (mode == 0) {
    constexpr int lds = (ss_rows_size(32 * NK) + 3 * ss_rows_size(16 * PT)) * 2;
    static const bool ready = hipFuncSetAttribute((const void*)decaying_piece_state_kernel<P, RULE, NK, PT>,
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
    if (!ready) return TS_ERR_LAUNCH;
    hipLaunchKernelGGL((decaying_piece_state_kernel<P, RULE, NK, PT>), grid, dim3(256), lds, stream, piece_state, piece_decay,
                       (const bf16_t*)u, rows, (const P*)proj, gates, (const SsPiece*)pieces, heads, groups, n, p);
  } else {
    constexpr int planes = 2 * 16 * PT * (32 * NK + 8) * 2, half = (SS_PIECE / 2 * (32 * NK + 8) + 16 * PT * (SS_PIECE + 4)) * 2;
    constexpr int lds = planes > half ? planes : half;
    static const bool ready = hipFuncSetAttribute((const void*)decaying_piece_out_kernel<P, RULE, NK, PT>,
                                                  hipFuncAttributeMaxDynamicSharedMemorySize, lds) == hipSuccess;
    if (!ready) return TS_ERR_LAUNCH;
    hipLaunchKernelGGL((decaying_piece_out_kernel<P, RULE, NK, PT>), grid, dim3(256), lds, stream, y, norm, piece_state, piece_top,
                       (const bf16_t*)u, rows, (const P*)proj, gates, skip, scale, (const SsPiece*)pieces, heads, groups, n, p);
  }
  return ts_launch_status();
}

template <typename P, int RULE, int ROWS>
static int ss_pass_launch(float* state, float* sums, const float* tops, const int* state_slots, const void* carries, int requests,
                          const void* pieces, float* piece_state, float* piece_top, const void* u, SsRows rows, const void* proj, SsGates gates,
                          int heads, int groups, int n, int p, hipStream_t stream) {
  constexpr int COLS = 2048 / ROWS, lds = (2 * 3 * COLS + 3 * ROWS) * SS_PIECE * 2;
  static const bool ready = hipFuncSetAttribute((const void*)decaying_pass_kernel<P, RULE, ROWS>, hipFuncAttributeMaxDynamicSharedMemorySize,
                                                lds) == hipSuccess;
  if (!ready) return TS_ERR_LAUNCH;
  const int columns = RULE == SS_GATED ? p + 1 : p;
  const dim3 grid(heads, requests, (n + ROWS - 1) / ROWS * ((columns + COLS - 1) / COLS));
  hipLaunchKernelGGL((decaying_pass_kernel<P, RULE, ROWS>), grid, dim3(512), lds, stream, state, sums, tops, state_slots, (const SsCarry*)carries,
                     (const SsPiece*)pieces, piece_state, piece_top, (const bf16_t*)u, rows, (const P*)proj, gates, heads, groups, n, p);
  return ts_launch_status();
}

// What both launches of a cut portion ask of their operands.
static int ss_pieces_ok(int rule, const void* u, const SsRows& rows, const SsGates& gates, const void* piece_state, int heads, int groups, int n, int p) {
  if (!ss_sizes_ok(rule, rows, gates, heads, groups, n, p) || n > 256 || n % 8 != 0 || p % 8 != 0) return TS_ERR_SHAPE;
  if (rows.width % 8 != 0 || rows.x_at % 8 != 0 || rows.b_at % 8 != 0 || rows.c_at % 8 != 0) return TS_ERR_SHAPE;  // 16-byte accesses
  return ((uintptr_t)u | (uintptr_t)piece_state) % 16 != 0 ? TS_ERR_ARG : TS_OK;
}

// bfloat16 runs; the states before the pieces (and in the slots what the last piece leaves), from a request's pieces one behind the other.
extern "C" int ts_decaying_pass(float* state, float* sums, const float* tops, const int* state_slots, const void* carries, int requests,
                                const void* pieces, float* piece_state, float* piece_top, const void* u, int u_width, int x_at, int b_at, int c_at,
                                const void* proj, int in_f32, int splits, long split_stride, int width, int first_gate, const float* one,
                                const float* two, float cap, int heads, int groups, int n, int p, int rule, hipStream_t stream) {
  if (requests == 0) return TS_OK;
  const SsRows rows = {1, 0, u_width, x_at, b_at, c_at};
  const SsGates gates = {splits, split_stride, width, first_gate, one, two, cap};
  if (!state || !state_slots || !carries || !pieces || !piece_state || !u || (rule == SS_GATED && !piece_top)) return TS_ERR_ARG;
  if (!ss_rule_ok(rule, gates, proj, piece_state, piece_state, sums, tops)) return TS_ERR_ARG;  // (no skip and no norm here)
  const int status = ss_pieces_ok(rule, u, rows, gates, piece_state, heads, groups, n, p);
  if (status != TS_OK) return status;
  if (((uintptr_t)state | (uintptr_t)sums) % 16 != 0) return TS_ERR_ARG;
#define SS_SIZE(P, RULE, ROWS)                                                                                                     \
  return ss_pass_launch<P, RULE, ROWS>(state, sums, tops, state_slots, carries, requests, pieces, piece_state, piece_top, u, rows, \
                                       proj, gates, heads, groups, n, p, stream)
#define SS_GO(P, RULE)                      \
  do {                                      \
    if (n <= 32) SS_SIZE(P, RULE, 32);      \
    if (n <= 64) SS_SIZE(P, RULE, 64);      \
    SS_SIZE(P, RULE, 128);                  \
  } while (0)
  if (rule == SS_SELECTIVE && in_f32) SS_GO(float, SS_SELECTIVE);
  if (rule == SS_SELECTIVE) SS_GO(bf16_t, SS_SELECTIVE);
  if (rule == SS_FIXED) SS_GO(bf16_t, SS_FIXED);
  if (in_f32) SS_GO(float, SS_GATED);
  SS_GO(bf16_t, SS_GATED);
#undef SS_GO
#undef SS_SIZE
}

// bfloat16 runs; mode 0: every piece's own end state and decay; mode 1: y from the state before each piece.
extern "C" int ts_decaying_pieces(float* y, float* norm, float* piece_state, float* piece_decay, const float* piece_top, const void* u,
                                  int u_width, int x_at, int b_at, int c_at, const void* proj, int in_f32, int splits, long split_stride,
                                  int width, int first_gate, const float* one, const float* two, float cap, const float* skip, float scale,
                                  const void* pieces, int num_pieces, int heads, int groups, int n, int p, int rule, int mode,
                                  hipStream_t stream) {
  if (num_pieces == 0) return TS_OK;
  const SsRows rows = {1, 0, u_width, x_at, b_at, c_at};
  const SsGates gates = {splits, split_stride, width, first_gate, one, two, cap};
  if (!piece_state || !piece_decay || !u || !pieces || (mode == 1 && !y) || mode < 0 || mode > 1) return TS_ERR_ARG;
  if (!ss_rule_ok(rule, gates, proj, skip, norm, piece_state, piece_top)) return TS_ERR_ARG;
  const int status = ss_pieces_ok(rule, u, rows, gates, piece_state, heads, groups, n, p);
  if (status != TS_OK) return status;
  if ((uintptr_t)y % 16 != 0) return TS_ERR_ARG;
#define SS_GO(P, RULE, NK, PT)                                                                                                     \
  return ss_pieces_launch<P, RULE, NK, PT>(mode, y, norm, piece_state, piece_decay, piece_top, u, rows, proj, gates, skip, scale,  \
                                           pieces, num_pieces, heads, groups, n, p, stream)
#define SS_SIZES(P, RULE, PT)                 \
  do {                                        \
    if (n <= 32) SS_GO(P, RULE, 1, PT);       \
    if (n <= 64) SS_GO(P, RULE, 2, PT);       \
    if (n <= 128) SS_GO(P, RULE, 4, PT);      \
    SS_GO(P, RULE, 8, PT);                    \
  } while (0)
#define SS_WIDTHS(P, RULE)                    \
  do {                                        \
    if (p <= 32) SS_SIZES(P, RULE, 2);        \
    SS_SIZES(P, RULE, 4);                     \
  } while (0)
  if (rule == SS_SELECTIVE && in_f32) SS_WIDTHS(float, SS_SELECTIVE);
  if (rule == SS_SELECTIVE) SS_WIDTHS(bf16_t, SS_SELECTIVE);
  if (rule == SS_FIXED) SS_WIDTHS(bf16_t, SS_FIXED);
  if (in_f32) SS_WIDTHS(float, SS_GATED);
  SS_WIDTHS(bf16_t, SS_GATED);
#undef SS_WIDTHS
#undef SS_SIZES
#undef SS_GO
}

extern "C" int ts_decaying_carry(float* state, float* sums, const float* tops, const int* state_slots, const void* carries,
                                 float* piece_state, const float* piece_decay, float* piece_top, int requests, int heads, int n, int p,
                                 int rule, hipStream_t stream) {
  if (requests == 0) return TS_OK;
  if (!state || !state_slots || !carries || !piece_state || !piece_decay) return TS_ERR_ARG;
  if (rule == SS_GATED && (!sums || !tops || !piece_top)) return TS_ERR_ARG;
  if (heads < 1 || heads > 65535 || n < 1 || p < 1 || n > 512 || p > 65534 || n % 4 != 0) return TS_ERR_SHAPE;
  const int columns = rule == SS_GATED ? p + 1 : p;
  const dim3 grid(requests, heads, (n * columns / 4 + 255) / 256);
  if (rule == SS_GATED)
    hipLaunchKernelGGL(decaying_carry_kernel<SS_GATED>, grid, dim3(256), 0, stream, state, sums, tops, state_slots, (const SsCarry*)carries,
                       piece_state, piece_decay, piece_top, heads, n, p);
  else  // (the other rules carry alike)
    hipLaunchKernelGGL(decaying_carry_kernel<SS_FIXED>, grid, dim3(256), 0, stream, state, sums, tops, state_slots, (const SsCarry*)carries,
                       piece_state, piece_decay, piece_top, heads, n, p);
  return ts_launch_status();
}

template <typename T, typename P>
static int launch_heads_finish(void* out, long out_stride, const float* y, const float* norm, const void* proj, int splits, long split_stride,
                               int width, int gate_at, const void* gain, int sigmoid, float eps, float scale, float* tops,
                               const int* state_slots, const int* token_seq, const int* query_start_loc, long items, int heads, int p,
                               hipStream_t stream) {
  const dim3 grid((unsigned)((items + 3) / 4)), block(256);
  const bool wide = p % 4 == 0 && width % 4 == 0 && gate_at % 4 == 0 && split_stride % 4 == 0 && out_stride % 4 == 0 &&
                    ((uintptr_t)out % (4 * sizeof(T))) == 0 && (((uintptr_t)y | (uintptr_t)proj | (uintptr_t)gain) % 16) == 0;
#define HF_GO(VEC)                                                                                                                   \
  hipLaunchKernelGGL((heads_finish_kernel<T, P, VEC>), grid, block, 0, stream, (T*)out, (size_t)out_stride, y, norm, (const P*)proj, \
                     splits, (size_t)split_stride, width, gate_at, (const T*)gain, sigmoid, eps, scale, tops, state_slots, token_seq, \
                     query_start_loc, items, heads, p)
  if (wide) HF_GO(4);
  else HF_GO(1);
#undef HF_GO
  return ts_launch_status();
}

extern "C" int ts_heads_finish(void* out, long out_stride, const float* y, const float* norm, const void* proj, int in_f32, int splits,
                               long split_stride, int width, int gate_at, const void* gain, int sigmoid, float eps, float scale, float* tops,
                               const int* state_slots, const int* token_seq, const int* query_start_loc, int tokens, int heads, int p,
                               int dtype, hipStream_t stream) {
  if (tokens == 0) return TS_OK;
  if (!out || !y || !proj || (norm && (!tops || !state_slots || !token_seq || !query_start_loc))) return TS_ERR_ARG;
  if (heads < 1 || p < 1 || gate_at < 0 || (long)gate_at + (long)heads * p > width || splits < 1 || out_stride < (long)heads * p) return TS_ERR_SHAPE;
  const long items = (long)tokens * heads;
#define HF_ARGS out, out_stride, y, norm, proj, splits, split_stride, width, gate_at, gain, sigmoid, eps, scale, tops, state_slots, token_seq, \
                query_start_loc, items, heads, p, stream
  if (dtype == TS_F32) return launch_heads_finish<float, float>(HF_ARGS);
  if (dtype == TS_BF16 && in_f32) return launch_heads_finish<bf16_t, float>(HF_ARGS);
  if (dtype == TS_BF16) return launch_heads_finish<bf16_t, bf16_t>(HF_ARGS);
#undef HF_ARGS
  return TS_ERR_DTYPE;
}

template <typename T, typename P>
static int launch_gated_group_norm(void* out, const float* y, const void* proj, int splits, long split_stride, int width, int z_at,
                                   const void* gain, float eps, int tokens, int parts, int size, hipStream_t stream) {
  const bool wide = size % 4 == 0 && width % 4 == 0 && z_at % 4 == 0 && split_stride % 4 == 0 &&
                    ((uintptr_t)out | (uintptr_t)y | (uintptr_t)proj | (uintptr_t)gain) % 16 == 0;
#define GN_GO(VEC, CHUNKS, THREADS)                                                                                                    \
  hipLaunchKernelGGL((gated_group_norm_kernel<T, P, VEC, CHUNKS>), dim3(tokens, parts), dim3(THREADS), 0, stream, (T*)out, y,          \
                     (const P*)proj, splits, (size_t)split_stride, width, z_at, (const T*)gain, eps, parts, size)
  if (wide) {
    const int pieces = size / 4;
    const bool few = (long)tokens * parts < 256;
    if (few && pieces <= 256 && splits <= 8) {
#define GN_FEW(THREADS, BATCH)                                                                                                      \
  hipLaunchKernelGGL((gated_group_norm_few_kernel<T, P, THREADS, BATCH>), dim3(tokens, parts), dim3(THREADS), 0, stream,            \
                     (const P*)proj, y, (const T*)gain, (T*)out, splits, width, (size_t)split_stride, z_at, parts, size, eps, SsMoves{})
#define GN_BATCH(THREADS)                     \
  do {                                        \
    if (splits == 1) GN_FEW(THREADS, 1);      \
    else if (splits <= 4) GN_FEW(THREADS, 4); \
    else GN_FEW(THREADS, 8);                  \
  } while (0)
      if (pieces <= 64) GN_BATCH(64);
      else if (pieces <= 128) GN_BATCH(128);
      else GN_BATCH(256);
#undef GN_BATCH
#undef GN_FEW
      return ts_launch_status();
    }
    // A wavefront a part where the projection is one of 16 bits and there are parts enough that four a workgroup fill the units (us, a workgroup /
    // a wavefront a part of 512, eight a row: 32 rows 2.6 / 2.8, 128 2.9 / 3.0, as soon from 192 to 512, 3.1 and 4.9, and the sooner beyond, figures
    // at the kernel; of two partial sums, which a workgroup asks for sooner, 32 rows 2.8 / 3.4, 256 4.0 / 4.2).
    const long items = (long)tokens * parts;
    if constexpr (sizeof(P) == 2) {
#define GN_ROWS(CHUNKS)                                                                                                                     \
  hipLaunchKernelGGL((gated_group_norm_rows_kernel<T, CHUNKS>), dim3((unsigned)((items + 3) / 4)), dim3(256), 0, stream, (T*)out, y,        \
                     (const T*)proj, width, z_at, (const T*)gain, eps, parts, size, (int)items)
      if (pieces <= 256 && items >= 1536 && items <= 0x7fffffffL && splits == 1) {
        if (pieces <= 64) GN_ROWS(1);
        else if (pieces <= 128) GN_ROWS(2);
        else GN_ROWS(4);
#undef GN_ROWS
        return ts_launch_status();
      }
    }
    if (pieces <= 256 || (few && pieces <= 1024)) GN_GO(4, 1, (pieces + 63) / 64 * 64);
    else if (pieces <= 1024) GN_GO(4, 4, 256);
    else if (pieces <= 4096) GN_GO(4, 4, 1024);
    else if (pieces <= 16384) GN_GO(4, 16, 1024);
    else return TS_ERR_SHAPE;
  } else {
    if (size <= 1024) GN_GO(1, 1, (size + 63) / 64 * 64);
    else if (size <= 16384) GN_GO(1, 16, 1024);
    else return TS_ERR_SHAPE;
  }
#undef GN_GO
  return ts_launch_status();
}

extern "C" int ts_gated_group_norm(void* out, const float* y, const void* proj, int in_f32, int splits, long split_stride, int width,
                                   int z_at, const void* gain, float eps, int tokens, int parts, int size, int dtype, hipStream_t stream) {
  if (tokens == 0) return TS_OK;
  if (!out || !y || !proj || !gain) return TS_ERR_ARG;
  if (parts < 1 || parts > 65535 || size < 1 || z_at < 0 || (long)z_at + (long)parts * size > width || splits < 1) return TS_ERR_SHAPE;
  if (dtype == TS_F32)
    return launch_gated_group_norm<float, float>(out, y, proj, splits, split_stride, width, z_at, gain, eps, tokens, parts, size, stream);
  if (dtype == TS_BF16 && in_f32)
    return launch_gated_group_norm<bf16_t, float>(out, y, proj, splits, split_stride, width, z_at, gain, eps, tokens, parts, size, stream);
  if (dtype == TS_BF16)
    return launch_gated_group_norm<bf16_t, bf16_t>(out, y, proj, splits, split_stride, width, z_at, gain, eps, tokens, parts, size, stream);
  return TS_ERR_DTYPE;
}

template <typename T>
static int launch_selective_token(void* out, float* y, float* state, float* held, const int* state_slots, const float* proj, int splits, long stride,
                                  int width, int z_at, int dt_at, SsConv conv, const float* dt_bias, const float* a_log, const float* skip, const void* gain,
                                  float eps, int tokens, int heads, int groups, int n, int p, int parts, hipStream_t stream) {
  const dim3 grid(tokens, heads, (p + 31) / 32);
#define ST_GO(NR, BATCH)                                                                                                                        \
  hipLaunchKernelGGL((selective_token_kernel<T, NR, BATCH>), grid, dim3(256), 0, stream, state, state_slots, proj, held, width, heads, groups, n, p, \
                     splits, (size_t)stride, conv, dt_at, dt_bias, a_log, skip, y)
#define ST_ROWS(BATCH)                  \
  do {                                  \
    if (n <= 32) ST_GO(4, BATCH);       \
    else if (n <= 64) ST_GO(8, BATCH);  \
    else ST_GO(16, BATCH);              \
  } while (0)
  if (splits == 1) ST_ROWS(1);
  else if (splits <= 4) ST_ROWS(4);
  else ST_ROWS(8);
#undef ST_ROWS
#undef ST_GO
  const int status = ts_launch_status();
  if (status != TS_OK) return status;
  const int inner = heads * p, moved = 2 * groups * n, size = inner / parts;
  const SsMoves moves = {held, state_slots, inner + moved, inner, moved, conv.first};
#define ST_NORM(THREADS, BATCH)                                                                                                          \
  hipLaunchKernelGGL((gated_group_norm_few_kernel<T, float, THREADS, BATCH, true>), dim3(tokens, parts + (moved + THREADS - 1) / THREADS), \
                     dim3(THREADS), 0, stream, proj, y, (const T*)gain, (T*)out, splits, width, (size_t)stride, z_at, parts, size, eps, moves)
#define ST_BATCH(THREADS)                     \
  do {                                        \
    if (splits == 1) ST_NORM(THREADS, 1);     \
    else if (splits <= 4) ST_NORM(THREADS, 4);\
    else ST_NORM(THREADS, 8);                 \
  } while (0)
  if (size <= 256) ST_BATCH(64);
  else if (size <= 512) ST_BATCH(128);
  else ST_BATCH(256);
#undef ST_BATCH
#undef ST_NORM
  return ts_launch_status();
}

// A step of single tokens of a selective state space from its projection on: ts_short_conv (four taps), ts_decaying_walk (selective) and
// ts_gated_group_norm in two launches, the same bits.  proj: `splits` (at most 8) 32-bit partial sums [tokens, width]; held float [slots, 3,
// heads p + 2 groups n]; y float [tokens, heads p] (scratch); out [tokens, heads p] of dtype; parts equal parts of a row of up to 1,024 elements;
// n and p multiples of 4, n at most 128; all on 16 bytes.
extern "C" int ts_selective_token(void* out, float* y, float* state, float* held, const int* state_slots, const void* proj, int splits, long stride,
                                  int width, int z_at, int first, int dt_at, const void* taps, const void* bias, int silu, const float* dt_bias,
                                  const float* a_log, const float* skip, const void* gain, float eps, int tokens, int heads, int groups, int n, int p,
                                  int parts, int dtype, hipStream_t stream) {
  if (tokens == 0) return TS_OK;
  if (!out || !y || !state || !held || !state_slots || !proj || !taps || !dt_bias || !a_log || !skip || !gain) return TS_ERR_ARG;
  if (heads < 1 || heads > 65535 || groups < 1 || heads % groups != 0 || n < 4 || n > 128 || n % 4 != 0 || p < 4 || p % 4 != 0 || parts < 1 ||
      splits < 1 || splits > 8 || width % 4 != 0 || z_at % 4 != 0 || stride % 4 != 0)
    return TS_ERR_SHAPE;
  const long inner = (long)heads * p;
  if (inner % parts != 0 || inner / parts > 1024 || inner / parts % 4 != 0 || z_at < 0 || z_at + inner > width || first < 0 ||
      first + inner + 2L * groups * n > width || dt_at < 0 || dt_at + heads > width || parts + 2L * groups * n / 64 > 65534)
    return TS_ERR_SHAPE;
  if (((uintptr_t)out | (uintptr_t)y | (uintptr_t)state | (uintptr_t)held | (uintptr_t)proj | (uintptr_t)gain) % 16 != 0) return TS_ERR_ARG;
  const SsConv conv = {taps, bias, first, silu};
#define ST_ARGS out, y, state, held, state_slots, (const float*)proj, splits, stride, width, z_at, dt_at, conv, dt_bias, a_log, skip, gain, eps, tokens, \
                heads, groups, n, p, parts, stream
  if (dtype == TS_F32) return launch_selective_token<float>(ST_ARGS);
  if (dtype == TS_BF16) return launch_selective_token<bf16_t>(ST_ARGS);
#undef ST_ARGS
  return TS_ERR_DTYPE;
}
