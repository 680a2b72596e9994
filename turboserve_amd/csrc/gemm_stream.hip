// The product of a decode step of up to 16 rows, bound by reading the weights once:
//   Y[m][n] = sum over k of X[m][k] * W[n][k]  (+ bias[n])
// bfloat16 activations X [M, K] and weights W [N, K] as the checkpoint stores them (F.linear's
// layout, src/turboserve/engine/model/layers.py:142), 32-bit accumulation on the matrix cores.
//
// A workgroup owns 16 NT weight rows and one of S ranges of K, each of its four wavefronts a quarter of the range.  A
// wavefront stages its part in a ring of its own in LDS, SLOTS slices of 64 k, straight from memory: an instruction takes
// whole lines, 128 bytes of each of eight rows, non-temporal for the weights, and a slot is filled again as
// soon as its fragments are in registers.  Nothing meets at a barrier before the quarters' sums, and a small matrix is in
// flight as a whole: what is left of such a product is one trip to memory.
// Microseconds at one row, in a graph, against the tiled or the resident kernel (which read half lines, or hand the weights
// through registers and meet at a barrier every 128 of K; with the SwiGLU where that is in the result): 2,048 x 2,048 4.4 -> 4.0, 2,048 x
// 8,192 12.2 -> 7.7, 8,192 x 2,048 12.3 -> 7.3, q|k|v [4608, 3584] 8.6 -> 7.9, o [3584, 3584] 8.4 -> 6.2, down [3584, 18944]
// 24.5 -> 22.0, gate|up [16384, 2048] 17.7 -> 13.4, [37888, 3584] 46.9 -> 41.0, the head [152064, 3584] 178 -> 153 (7.1 TB/s).
// Without loads past the end and past the eighth row, and with the bias asked for at the start: q|k|v 7.8 -> 7.4, [10304, 2048]
// 10.9 -> 10.4, 2,048 x 8,192 8.15 -> 7.97, gate|up [16384, 2048] 13.3 -> 13.0, the long ones within 1%.
#include "common.hpp"

#include <type_traits>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
typedef __attribute__((address_space(3))) uint16_t lds_u16;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;
typedef __attribute__((address_space(3))) f32x4 lds_f32x4;

constexpr int STREAM_WAVES = 4;

constexpr int NORMED_MOST = 6144, NORMED_ROOM = NORMED_MOST + 64;  // elements of normalised rows in LDS (XT = 0), and their wavefronts' sums

// NT tiles of sixteen weight rows, XT of eight activation rows (0: they lie in LDS as a whole).
template <int NT, int XT>
struct Ring {
  static constexpr int SLICE = 64, TILE = 16 * SLICE, HALF = 8 * SLICE, LOADS = 2 * NT + XT;  // of sixteen rows; of eight; of a slice
  static constexpr int SLOT = NT * TILE + XT * HALF;
  static constexpr int SLOTS = (80 * 1024 - (XT ? 0 : NORMED_ROOM * 2)) / (STREAM_WAVES * SLOT * 2);  // two workgroups a compute unit
  static constexpr int WAVE = SLOTS * SLOT;                            // elements of a wavefront's ring
  static constexpr size_t BYTES = (size_t)STREAM_WAVES * WAVE * 2;
  static_assert(SLOTS >= 2 && (SLOTS - 1) * LOADS < 64 && 2 * (BYTES + (XT ? 0 : NORMED_ROOM * 2)) <= 160 * 1024, "a ring of at least two slices, counted by vmcnt");
  static_assert(WAVE * 2 >= NT * 1024, "a wavefront's sums fit its ring");
};

// `to` and `from` are the same memory: __restrict__ keeps the compiler from waiting for every load in flight before every
// read, so it must not see that two reads have one address either: the slot that this wait lets be read is a new value to it
// (no read moves above it), and a slot's fragments go through an asm that waits for them before it is filled again.  An edit
// has to keep both.
template <int LEFT>
__device__ __forceinline__ void stream_wait(int& slot) {
  asm volatile("s_waitcnt vmcnt(%1)" : "+s"(slot) : "n"(LEFT) : "memory");
}
// With `left` (at most MOST) slices of LOADS loads each still on their way behind the one that is waited for.
template <int LOADS, int MOST>
__device__ __forceinline__ void stream_wait_for(int left, int& slot) {
  if constexpr (MOST > 0) {
    if (left < MOST) return stream_wait_for<LOADS, MOST - 1>(left, slot);
  }
  stream_wait<MOST * LOADS>(slot);
}

// acc[t][i]: weight row n0 + 16 t + 4 (lane / 16) + i, activation row lane % 16 (lane % 8 with XT = 1), over slices first .. last - 1
// of 64 k.  XT = 0: activation row lane % ROWS of `held`, rows of k elements in LDS (k whole slices); `meanwhile` runs when the first slices
// have been asked for and puts them there, its own loads before those of any slice; it is called by every wavefront.
template <int NT, int XT, int ROWS, typename Meanwhile>
__device__ __forceinline__ void stream_range(lds_u16* __restrict__ to, const lds_u16* __restrict__ from, const lds_u16* __restrict__ held,
                                             const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int m, int n, int k,
                                             long x_stride, int n0, int first, int last, f32x4* acc, Meanwhile meanwhile) {
  typedef Ring<NT, XT> R;
  constexpr int SLICE = R::SLICE, TILE = R::TILE, HALF = R::HALF, SLOTS = R::SLOTS;
  const int count = last - first;
  if (XT != 0 && count <= 0) return;
  const int lane = threadIdx.x & 63, r = lane & 15, g = lane >> 4;
  // A lane loads 16 bytes, piece (lane % 8) ^ key of row lane / 8 of eight, key = row / 2 % 8: a piece of sixteen rows
  // touches every bank once.  (The second eight rows of a tile have keys four further on: piece ^ 4.)  What lies past the last
  // row's end (rows beyond N or M) brings zeros, what lies past another row's end (a K that is no multiple of 64) is cleared.
  const int row8 = lane >> 3, piece = (lane & 7) ^ (row8 >> 1);
  const size_t wbytes = (size_t)min(n - n0, 16 * NT) * k * 2, xbytes = ((size_t)(m - 1) * x_stride + k) * 2;
  const __amdgpu_buffer_rsrc_t wbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(w + (size_t)n0 * k), 0, XT == 0 && count <= 0 ? 0 : (int)wbytes, 0x00027000);
  const __amdgpu_buffer_rsrc_t xbuf = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint16_t*>(x), 0, (int)xbytes, 0x00027000);
  uint32_t woff[2 * NT], xoff[XT ? XT : 1];
#pragma unroll
  for (int j = 0; j < 2 * NT; ++j) woff[j] = ((uint32_t)(8 * j + row8) * (uint32_t)k + first * SLICE + 8 * (piece ^ (j & 1 ? 4 : 0))) * 2;
#pragma unroll
  for (int j = 0; j < XT; ++j) xoff[j] = ((uint32_t)(8 * j + row8) * (uint32_t)x_stride + first * SLICE + 8 * (piece ^ (j & 1 ? 4 : 0))) * 2;
  auto fetch = [&](int i, int slot) __attribute__((always_inline)) {
    const uint32_t at = (uint32_t)i * (SLICE * 2);
    lds_u16* base = to + slot * R::SLOT;
#pragma unroll
    for (int j = 0; j < 2 * NT; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(wbuf, base + j * HALF, 16, (int)(woff[j] + at), 0, 0, 2);  // non-temporal
#pragma unroll
    for (int j = 0; j < XT; ++j)
      __builtin_amdgcn_raw_ptr_buffer_load_lds(xbuf, base + NT * TILE + j * HALF, 16, (int)(xoff[j] + at), 0, 0, 0);
  };
  struct Frags {
    u32x4 x[2], w[NT][2];
  };
  const int key = (r >> 1) & 7, x_row = XT ? r & (8 * XT - 1) : r & (ROWS - 1);
  int held_at = x_row * k + first * SLICE + 8 * g;
  auto read = [&](Frags& f, int i, int slot) __attribute__((always_inline)) {
    const lds_u16* base = from + slot * R::SLOT;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int t = 0; t < NT; ++t) f.w[t][c] = *(const lds_u32x4*)(base + t * TILE + r * SLICE + 8 * ((4 * c + g) ^ key));
      if (XT) f.x[c] = *(const lds_u32x4*)(base + NT * TILE + x_row * SLICE + 8 * ((4 * c + g) ^ (x_row >> 1)));
      else f.x[c] = *(const lds_u32x4*)(held + held_at + i * SLICE + 32 * c);
    }
  };
  auto consume = [&](Frags& f, int left) __attribute__((always_inline)) {  // left: elements of the slice inside the row
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const bool inside = left >= SLICE || 32 * c + 8 * g < left;  // a piece lies inside as a whole
      const u32x4 none = {0u, 0u, 0u, 0u};
      if (left < SLICE) f.x[c] = inside ? f.x[c] : none;
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        if (left < SLICE) f.w[t][c] = inside ? f.w[t][c] : none;
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, f.w[t][c]), __builtin_bit_cast(bf16x8, f.x[c]), acc[t], 0, 0, 0);
      }
    }
  };
  auto arrived = [&](Frags& f) __attribute__((always_inline)) {  // in registers: the slot is free
#pragma unroll
    for (int c = 0; c < 2; ++c) {
#pragma unroll
      for (int t = 0; t < NT; ++t) asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f.w[t][c])::"memory");
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(f.x[c])::"memory");
    }
  };
  // No load is issued past the end: one that brings nothing still takes its turn in the unit's memory path, and a ring's worth
  // of them behind every wavefront made a short product's end (or the next workgroup's start) a microsecond longer.
  int slot = 0;
  if (XT) {
#pragma unroll
    for (int j = 0; j < SLOTS; ++j)
      if (j < count) fetch(j, j);
    stream_wait_for<R::LOADS, SLOTS - 1>(count - 1, slot);
  } else {
    // (Without a branch, so that the compiler can count them behind the loads of `meanwhile`; those past the end lie outside the buffer.)
#pragma unroll
    for (int j = 0; j < SLOTS; ++j) {
#pragma unroll
      for (int t = 0; t < 2 * NT; ++t)
        __builtin_amdgcn_raw_ptr_buffer_load_lds(wbuf, to + j * R::SLOT + t * HALF, 16, j < count ? (int)(woff[t] + j * (SLICE * 2)) : (int)0x80000000, 0, 0, 2);
    }
    __builtin_amdgcn_sched_barrier(0);
    meanwhile();
    asm volatile("" : "+v"(held_at)::"memory");  // what `meanwhile` wrote is read at addresses that are new to the compiler
    if (count <= 0) return;
    stream_wait<(SLOTS - 1) * R::LOADS>(slot);
  }
  Frags f[2];
  read(f[0], 0, slot);
  auto round = [&](int i, Frags& now, Frags& next) __attribute__((always_inline)) {
    arrived(now);
    fetch(i + SLOTS, slot);
    slot = slot + 1 == SLOTS ? 0 : slot + 1;
    stream_wait<(SLOTS - 1) * R::LOADS>(slot);
    read(next, i + 1, slot);
    consume(now, SLICE);
  };
  int i = 0;
  for (; i + SLOTS + 1 < count; i += 2) {
    round(i, f[0], f[1]);
    round(i + 1, f[1], f[0]);
  }
  if (i + SLOTS < count) {
    round(i, f[0], f[1]);
    arrived(f[1]);
    f[0] = f[1];
    ++i;
  }
  // What is left lies in the ring or is on its way there: slice i in f[0].
  for (; i + 1 < count; ++i) {
    arrived(f[0]);
    f[1] = f[0];
    slot = slot + 1 == SLOTS ? 0 : slot + 1;
    stream_wait_for<R::LOADS, SLOTS - 2>(count - i - 2, slot);
    read(f[0], i + 1, slot);
    consume(f[1], SLICE);
  }
  consume(f[0], k - (last - 1) * SLICE);  // the last slice alone may be cut short
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
}

// What a workgroup does with its wavefronts' sums: the quarters meet in the rings; wavefront v adds up and stores tile v, `shift` its bias.
// (`wave` comes from the caller: asked for again here, with a wait behind the last product, a decode step of 28 products took 495.5 us for 492.7.)
// UNIT: what is stored of the sums: 0 they themselves, 32-bit, 1 the gated unit, 2 relu_squared, bfloat16.
template <int NT, int XT, int UNIT>
__device__ __forceinline__ void stream_finish(lds_u16* ring, int wave, const f32x4* acc, const uint32_t (&shift)[4], bool shifted, int m, int n, int col, int split,
                                              float* __restrict__ partial, uint16_t* __restrict__ out, GluRule rule) {
  typedef Ring<NT, XT> R;
  const int lane = threadIdx.x & 63;
#pragma unroll
  for (int t = 0; t < NT; ++t) ((lds_f32x4*)(ring + wave * R::WAVE))[t * 64 + lane] = acc[t];
  __syncthreads();
  if (wave >= NT) return;
  f32x4 sum = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int v = 0; v < STREAM_WAVES; ++v) sum += ((lds_f32x4*)(ring + v * R::WAVE))[wave * 64 + lane];
  const int row = lane & 15;
  if (row >= m || col >= n) return;
  if (shifted) {
#pragma unroll
    for (int i = 0; i < 4; ++i) sum[i] += __uint_as_float(shift[i] << 16);
  }
  if (UNIT == 2) {
    uint16_t* at = out + (size_t)row * n + col;
    if (n % 4 == 0) {
      *reinterpret_cast<u32x2*>(at) = u32x2{from_float<bf16_t>(relu_squared(sum[0])).bits | (uint32_t)from_float<bf16_t>(relu_squared(sum[1])).bits << 16,
                                            from_float<bf16_t>(relu_squared(sum[2])).bits | (uint32_t)from_float<bf16_t>(relu_squared(sum[3])).bits << 16};
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (col + i < n) at[i] = from_float<bf16_t>(relu_squared(sum[i])).bits;
    }
  } else if (UNIT == 1) {  // n is even: the first pair lies inside
    uint16_t* at = out + (size_t)row * (n / 2) + col / 2;
    at[0] = from_float<bf16_t>(gated_unit(sum[0], sum[1], rule)).bits;
    if (col + 2 < n) at[1] = from_float<bf16_t>(gated_unit(sum[2], sum[3], rule)).bits;
  } else {
    float* at = partial + ((size_t)split * m + row) * n + col;
    if (n % 4 == 0) {
      *reinterpret_cast<f32x4*>(at) = sum;
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (col + i < n) at[i] = sum[i];
    }
  }
}

// partial: float [splits, m, n], or out: bfloat16 [m, n / 2], the gated unit (common.hpp) of rows that alternate gate, up, or [m, n], relu_squared.
template <int NT, int XT, int UNIT>
__global__ void __launch_bounds__(64 * STREAM_WAVES)
gemm_stream_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, const uint16_t* __restrict__ bias, int x_stride, int m,
                   int n, int k, int per_wave, float* __restrict__ partial, uint16_t* __restrict__ out, GluRule rule) {
  // (Fourteen words of arguments lie in registers at the start: those that the first loads want come first.)
  extern __shared__ __attribute__((aligned(16))) uint16_t ring[];
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 16 * NT, split = blockIdx.y;
  typedef Ring<NT, XT> R;
  const int total = (k + R::SLICE - 1) / R::SLICE;
  const int first = (split * STREAM_WAVES + wave) * per_wave, last = min(first + per_wave, total);
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  // The bias is asked for with the first slices, not behind the last (a register each: packed in pairs they were waited for at once).
  const int col = n0 + 16 * min(wave, NT - 1) + 4 * (lane >> 4);
  uint32_t shift[4] = {0, 0, 0, 0};
  if (bias && split == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) shift[i] = bias[min(col + i, n - 1)];
  }
  lds_u16* mine = (lds_u16*)ring + wave * R::WAVE;
  stream_range<NT, XT, 0>(mine, mine, mine, x, w, m, n, k, x_stride, n0, first, last, acc, [] {});
  stream_finish<NT, XT, UNIT>((lds_u16*)ring, wave, acc, shift, bias && split == 0, m, n, col, split, partial, out, rule);
}

template <int NT, int XT, int UNIT>
int launch_stream(float* partial, void* out, const void* x, long x_stride, const void* w, const void* bias, int m, int n, int k,
                  int per_wave, int splits, GluRule rule, hipStream_t stream) {
  constexpr size_t BYTES = Ring<NT, XT>::BYTES;
  static bool raised = false;  // per process; the attribute belongs to the kernel
  if (!raised) {
    if (hipFuncSetAttribute((const void*)gemm_stream_kernel<NT, XT, UNIT>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)BYTES) != hipSuccess)
      return TS_ERR_LAUNCH;
    raised = true;
  }
  hipLaunchKernelGGL((gemm_stream_kernel<NT, XT, UNIT>), dim3((n + 16 * NT - 1) / (16 * NT), splits), dim3(64 * STREAM_WAVES),
                     BYTES, stream, (const uint16_t*)x, (const uint16_t*)w, (const uint16_t*)bias, (int)x_stride, m, n, k, per_wave,
                     partial, (uint16_t*)out, rule);
  return ts_launch_status();
}

// The same for one or two rows that are the norm of the residual stream, which is not stored: every workgroup adds up the pending partial sums and
// normalises the whole row for itself while its first weights travel.  The norm's own launch, some 4.5 us of a
// recorded step of which one trip to memory and the launch are most, falls away; what comes instead is 50 KB a row from L2 for every workgroup.
// The sum goes to `after` (not to `residual`, which other workgroups are still to read): of 1,024 elements by one workgroup each.
template <int NT, int ROWS, int ITEMS, int SUMS, bool GATED>
__global__ void __launch_bounds__(64 * STREAM_WAVES)
gemm_stream_normed_kernel(const float* __restrict__ residual, const float* __restrict__ pending, const uint16_t* __restrict__ gain,
                          const uint16_t* __restrict__ w, int n, int k, int per_wave, float eps, float* __restrict__ after,
                          const uint16_t* __restrict__ bias, float* __restrict__ partial, uint16_t* __restrict__ out, float gain_offset,
                          int one_rounding, GluRule rule) {
  extern __shared__ __attribute__((aligned(16))) uint16_t ring[];
  constexpr int THREADS = 64 * STREAM_WAVES;
  typedef Ring<NT, 0> R;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 16 * NT, split = blockIdx.y, quads = k / 4;
  float s[ROWS][ITEMS][4], part[ROWS][ITEMS][SUMS][4];
  u32x2 g[ITEMS];
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    const int quad = threadIdx.x + it * THREADS, at = 4 * (it + 1 < ITEMS ? quad : min(quad, quads - 1));
#pragma unroll
    for (int row = 0; row < ROWS; ++row) {
#pragma unroll
      for (int j = 0; j < SUMS; ++j) *(f32x4*)part[row][it][j] = *(const f32x4*)(pending + ((size_t)j * ROWS + row) * k + at);
      *(f32x4*)s[row][it] = *(const f32x4*)(residual + (size_t)row * k + at);
    }
    g[it] = *(const u32x2*)(gain + at);
  }
  const int col = n0 + 16 * min(wave, NT - 1) + 4 * (lane >> 4);
  uint32_t shift[4] = {0, 0, 0, 0};
  if (bias && split == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) shift[i] = bias[min(col + i, n - 1)];
  }
  asm volatile("" ::: "memory");  // all of them on their way here
  __builtin_amdgcn_sched_barrier(0);
  uint16_t* const held = ring + STREAM_WAVES * R::WAVE;
  constexpr int CHAINS = ITEMS < 4 ? ITEMS : 4;
  typedef float chains __attribute__((ext_vector_type(4)));
  chains(*const sums)[STREAM_WAVES] = reinterpret_cast<chains(*)[STREAM_WAVES]>(held + NORMED_ROOM - 8 * ROWS * STREAM_WAVES);  // behind the rows
  static_assert(NORMED_MOST + 8 * ROWS * STREAM_WAVES <= NORMED_ROOM, "the wavefronts' sums lie behind the rows");
  auto meet = [] { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };  // (the fence of __syncthreads would wait for the weights)
  // The workgroup's range of K is all it needs normalised.
  const int from_quad = split * STREAM_WAVES * per_wave * (R::SLICE / 4), to_quad = min(quads, from_quad + STREAM_WAVES * per_wave * (R::SLICE / 4));
  auto normalise = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int row = 0; row < ROWS; ++row) {
      // The squares in add_rmsnorm's order (elementwise.hip, add_rmsnorm_few_kernel), so that a row has its bits in steps of any number of rows: chain
      // c of this thread is what thread (threadIdx.x + 256 c) of 1,024 adds up, its wavefront's sum the one in place 4 c + wave.
      float ss[CHAINS];
#pragma unroll
      for (int it = 0; it < ITEMS; ++it) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
#pragma unroll
          for (int j = 0; j < SUMS; ++j) s[row][it][e] += part[row][it][j][e];
        }
        const float(&v)[4] = s[row][it];
        const float two = it < CHAINS ? fmaf(v[0], v[0], v[1] * v[1]) : fmaf(v[1], v[1], fmaf(v[0], v[0], ss[it % CHAINS]));
        const float four = fmaf(v[3], v[3], fmaf(v[2], v[2], two));
        // All but the last item lie inside the row.
        ss[it % CHAINS] = it + 1 < ITEMS || (int)threadIdx.x + it * THREADS < quads ? four : it < CHAINS ? 0.f : ss[it % CHAINS];
      }
      wave_sums(ss);
      if (lane == TS_WAVE - 1) sums[row][wave] = chains{ss[0], ss[1 % CHAINS], ss[2 % CHAINS], ss[3 % CHAINS]};
    }
    meet();
    float rstd[ROWS];
#pragma unroll
    for (int row = 0; row < ROWS; ++row) {
      float ss = 0.f;
#pragma unroll
      for (int v = 0; v < CHAINS * STREAM_WAVES; ++v) ss += sums[row][v % STREAM_WAVES][v / STREAM_WAVES];
      rstd[row] = rsqrtf(ss / (float)k + eps);
    }
    auto write = [&](auto ONE_ROUNDING) __attribute__((always_inline)) {
#pragma unroll
      for (int it = 0; it < ITEMS; ++it) {
        const int quad = threadIdx.x + it * THREADS;
        if (quad < from_quad || quad >= to_quad) continue;
#pragma unroll
        for (int row = 0; row < ROWS; ++row) {
          float n[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float gained = __uint_as_float(e & 1 ? g[it][e / 2] & 0xffff0000u : g[it][e / 2] << 16);
            n[e] = with_gain<bf16_t>(s[row][it][e] * rstd[row], gained, gain_offset, decltype(ONE_ROUNDING)::value);
          }
          *(u32x2*)(held + row * k + 4 * quad) = u32x2{(uint32_t)from_float<bf16_t>(n[0]).bits | (uint32_t)from_float<bf16_t>(n[1]).bits << 16,
                                                       (uint32_t)from_float<bf16_t>(n[2]).bits | (uint32_t)from_float<bf16_t>(n[3]).bits << 16};
        }
      }
    };
    if (one_rounding) write(std::true_type{});
    else write(std::false_type{});
    meet();
    if (split == 0 && (int)blockIdx.x < ITEMS) {
#pragma unroll
      for (int it = 0; it < ITEMS; ++it) {
        const int quad = threadIdx.x + it * THREADS;
#pragma unroll
        for (int row = 0; row < ROWS; ++row)
          if ((int)blockIdx.x == it && quad < quads) *(f32x4*)(after + (size_t)row * k + 4 * quad) = *(const f32x4*)s[row][it];
      }
    }
  };
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int total = k / R::SLICE, first = (split * STREAM_WAVES + wave) * per_wave, last = min(first + per_wave, total);
  lds_u16* mine = (lds_u16*)ring + wave * R::WAVE;
  stream_range<NT, 0, ROWS>(mine, mine, (const lds_u16*)held, nullptr, w, ROWS, n, k, 0, n0, first, last, acc, normalise);
  stream_finish<NT, 0, GATED ? 1 : 0>((lds_u16*)ring, wave, acc, shift, bias && split == 0, ROWS, n, col, split, partial, out, rule);
}

template <int ROWS, int ITEMS, int SUMS, bool GATED>
int launch_stream_normed(float* partial, void* out, const float* residual, const float* pending, float* after, const void* gain,
                         float eps, float gain_offset, int one_rounding, const void* w, const void* bias, int n, int k, int per_wave, int splits,
                         GluRule rule, hipStream_t stream) {
  constexpr size_t BYTES = Ring<2, 0>::BYTES + NORMED_ROOM * 2;
  static bool raised = false;  // per process; the attribute belongs to the kernel
  if (!raised) {
    if (hipFuncSetAttribute((const void*)gemm_stream_normed_kernel<2, ROWS, ITEMS, SUMS, GATED>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)BYTES) !=
        hipSuccess)
      return TS_ERR_LAUNCH;
    raised = true;
  }
  hipLaunchKernelGGL((gemm_stream_normed_kernel<2, ROWS, ITEMS, SUMS, GATED>), dim3((n + 31) / 32, splits), dim3(64 * STREAM_WAVES), BYTES, stream,
                     residual, pending, (const uint16_t*)gain, (const uint16_t*)w, n, k, per_wave, eps, after, (const uint16_t*)bias,
                     partial, (uint16_t*)out, gain_offset, one_rounding, rule);
  return ts_launch_status();
}

// The same for the one row that is a token's attention, whose workgroups have left their sums (attention_mfma.hip: partial_acc [heads, splits, d], partial_ml
// [heads, splits] of reference and sum): every workgroup puts its range of K together, as decode_reduce_kernel does, while its first weights
// travel.  That launch took 4.9 us of a layer; 3,584 elements of eight workgroups are 57 KB from L2 for
// every workgroup of two ranges, and their exponentials and quotients 3: a token of the 7B shape 2,603 -> 2,579 us, 5 of which
// weights below 2^-126 take (exp2f; the hardware's 2^x clears them, and a branch around it for those without was no sooner).
template <int NT, int ITEMS, int PARTS>
__global__ void __launch_bounds__(64 * STREAM_WAVES)
gemm_stream_heads_kernel(const float* __restrict__ partial_acc, const float* __restrict__ partial_ml, const uint16_t* __restrict__ w, int splits_in,
                         int d, int n, int k, int per_wave, const uint16_t* __restrict__ bias, float* __restrict__ partial) {
  extern __shared__ __attribute__((aligned(16))) uint16_t ring[];
  constexpr int THREADS = 64 * STREAM_WAVES;
  typedef Ring<NT, 0> R;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int n0 = blockIdx.x * 16 * NT, split = blockIdx.y;
  const int from_quad = split * STREAM_WAVES * per_wave * (R::SLICE / 4), to_quad = min(k / 4, from_quad + STREAM_WAVES * per_wave * (R::SLICE / 4));
  float part[ITEMS][PARTS][4], m[ITEMS][PARTS], l[ITEMS][PARTS];
#pragma unroll
  for (int it = 0; it < ITEMS; ++it) {
    const int at = 4 * min(from_quad + (int)threadIdx.x + it * THREADS, to_quad - 1), head = at / d;
    const size_t base = (size_t)head * splits_in;
#pragma unroll
    for (int s = 0; s < PARTS; ++s) {
      const size_t entry = base + min(s, splits_in - 1);
      const float2 ml = *(const float2*)(partial_ml + 2 * entry);
      m[it][s] = ml.x, l[it][s] = ml.y;
      *(f32x4*)part[it][s] = *(const f32x4*)(partial_acc + entry * d + (at - head * d));
    }
  }
  const int col = n0 + 16 * min(wave, NT - 1) + 4 * (lane >> 4);
  uint32_t shift[4] = {0, 0, 0, 0};
  if (bias && split == 0) {
#pragma unroll
    for (int i = 0; i < 4; ++i) shift[i] = bias[min(col + i, n - 1)];
  }
  asm volatile("" ::: "memory");  // all of them on their way here
  __builtin_amdgcn_sched_barrier(0);
  uint16_t* const held = ring + STREAM_WAVES * R::WAVE;
  auto combine = [&]() __attribute__((always_inline)) {
#pragma clang fp contract(off)  // the products rounded before they are added up, as between that kernel's threads
#pragma unroll
    for (int it = 0; it < ITEMS; ++it) {
      const int quad = from_quad + threadIdx.x + it * THREADS;
      float most = -INFINITY, weight[PARTS];
#pragma unroll
      for (int s = 0; s < PARTS; ++s) most = fmaxf(most, m[it][s]);  // (a share past the last is the last one again)
#pragma unroll
      for (int s = 0; s < PARTS; ++s) weight[s] = s >= splits_in || m[it][s] == -INFINITY ? 0.f : exp2f(m[it][s] - most);  // no keys
      float sum[PARTS];
#pragma unroll
      for (int s = 0; s < PARTS; ++s) sum[s] = l[it][s] * weight[s];
#pragma unroll
      for (int step = 1; step < PARTS; step *= 2) {
#pragma unroll
        for (int s = 0; s < PARTS; s += 2 * step) sum[s] += sum[s + step];
      }
      uint32_t two[2] = {0, 0};
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        float num = 0.f;
#pragma unroll
        for (int s = 0; s < PARTS; ++s) num += part[it][s][e] * weight[s];
        two[e / 2] |= (uint32_t)from_float<bf16_t>(num / sum[0]).bits << 16 * (e & 1);
      }
      if (quad < to_quad) *(u32x2*)(held + 4 * quad) = u32x2{two[0], two[1]};
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");  // (the fence of __syncthreads would wait for the weights)
  };
  f32x4 acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = f32x4{0.f, 0.f, 0.f, 0.f};
  const int total = k / R::SLICE, first = (split * STREAM_WAVES + wave) * per_wave, last = min(first + per_wave, total);
  lds_u16* mine = (lds_u16*)ring + wave * R::WAVE;
  stream_range<NT, 0, 1>(mine, mine, (const lds_u16*)held, nullptr, w, 1, n, k, 0, n0, first, last, acc, combine);
  stream_finish<NT, 0, 0>((lds_u16*)ring, wave, acc, shift, bias && split == 0, 1, n, col, split, partial, nullptr, GluRule{1.f, 0.f, 0.f, 0.f});
}

template <int ITEMS, int PARTS>
int launch_stream_heads(float* partial, const float* partial_acc, const float* partial_ml, int splits_in, int d, const void* w, const void* bias,
                        int n, int k, int per_wave, int splits, hipStream_t stream) {
  constexpr size_t BYTES = Ring<2, 0>::BYTES + NORMED_ROOM * 2;
  static bool raised = false;  // per process; the attribute belongs to the kernel
  if (!raised) {
    if (hipFuncSetAttribute((const void*)gemm_stream_heads_kernel<2, ITEMS, PARTS>, hipFuncAttributeMaxDynamicSharedMemorySize, (int)BYTES) != hipSuccess)
      return TS_ERR_LAUNCH;
    raised = true;
  }
  hipLaunchKernelGGL((gemm_stream_heads_kernel<2, ITEMS, PARTS>), dim3((n + 31) / 32, splits), dim3(64 * STREAM_WAVES), BYTES, stream, partial_acc,
                     partial_ml, (const uint16_t*)w, splits_in, d, n, k, per_wave, (const uint16_t*)bias, partial);
  return ts_launch_status();
}

}  // namespace

// x [m, k] bfloat16 (m up to 16, k a multiple of 8) with row stride x_stride; w [n, k] bfloat16 contiguous; bias [n] bfloat16 or
// null.  partial = float [splits, m, n], or out = bfloat16 [m, n / 2] (splits 1, n even): the gated unit of a w whose rows
// alternate gate, up, or, `squared`, bfloat16 [m, n]: relu_squared (splits 1; n even or odd).  Slices of 64 of k: per_wave to each of the four wavefronts of each of `splits` =
// ceil(ceil(k / 64) / (4 per_wave)) ranges.  tile: 1 or 2 (16 or 32 weight rows a workgroup).
extern "C" int ts_gemm_stream(float* partial, void* out, const void* x, long x_stride, const void* w, const void* bias, int m,
                              int n, int k, int per_wave, int splits, int tile, int squared, float steepness, float limit, float up_shift,
                              float cubic, hipStream_t stream) {
  if (m == 0 || n == 0) return TS_OK;
  if (!x || !w || m < 0 || n < 0 || k < 8 || (partial == nullptr) == (out == nullptr)) return TS_ERR_ARG;
  if (m > 16 || k % 8 != 0 || x_stride < k || x_stride % 8 != 0 || (uintptr_t)x % 16 != 0 || (uintptr_t)w % 16 != 0) return TS_ERR_SHAPE;
  if (x_stride >= (1L << 24) || k >= (1 << 24)) return TS_ERR_SHAPE;  // a tile's rows lie within 31 bits of its first one
  if (per_wave < 1 || splits < 1 || splits > 65535) return TS_ERR_SHAPE;
  if (splits != ((k + 63) / 64 + 4L * per_wave - 1) / (4L * per_wave)) return TS_ERR_SHAPE;
  if (out && (splits != 1 || (!squared && n % 2 != 0))) return TS_ERR_ARG;
  const GluRule rule = {steepness, limit, up_shift, cubic};
  // Up to eight rows are one load a slice instead of two, and leave room for a slice more in the ring.
#define TS_STREAM(NT, UNIT)                                                                                                                   \
  return m <= 8 ? launch_stream<NT, 1, UNIT>(partial, out, x, x_stride, w, bias, m, n, k, per_wave, splits, rule, stream)                   \
                : launch_stream<NT, 2, UNIT>(partial, out, x, x_stride, w, bias, m, n, k, per_wave, splits, rule, stream)
  if (tile == 1) {
    if (out && squared) TS_STREAM(1, 2);
    if (out) TS_STREAM(1, 1);
    TS_STREAM(1, 0);
  }
  if (tile == 2) {
    if (out && squared) TS_STREAM(2, 2);
    if (out) TS_STREAM(2, 1);
    TS_STREAM(2, 0);
  }
#undef TS_STREAM
  return TS_ERR_SHAPE;
}

// The product of norm(residual + pending) as add_rmsnorm makes it (elementwise.hip), bfloat16, which is not stored: residual [m, k] float, m 1 or 2, pending
// float [sums, m, k], up to 4, gain [k] bfloat16, k a multiple of 64 and m k at most 6,144; after [m, k] float, other memory than residual, takes
// the sum.  All 16-byte aligned.  n more than 32 (ceil(k / 1024) - 1): a workgroup for every 1,024 elements of `after`.  The rest as ts_gemm_stream's.
extern "C" int ts_gemm_stream_normed(float* partial, void* out, const float* residual, const float* pending, int sums, float* after, const void* gain,
                                     float eps, float gain_offset, int one_rounding, const void* w, const void* bias, int m, int n, int k,
                                     int per_wave, int splits, float steepness, float limit, float up_shift, float cubic, hipStream_t stream) {
  if (!residual || !pending || !after || after == residual || !gain || !w || (partial == nullptr) == (out == nullptr)) return TS_ERR_ARG;
  if (m < 1 || m > 2 || k < 64 || k % 64 != 0 || m * (long)k > NORMED_MOST || sums < 1 || sums > 4 || n < 1) return TS_ERR_SHAPE;
  if (n <= 32 * ((k + 1023) / 1024 - 1)) return TS_ERR_SHAPE;
  if (((uintptr_t)residual | (uintptr_t)pending | (uintptr_t)after | (uintptr_t)gain | (uintptr_t)w) % 16 != 0) return TS_ERR_SHAPE;
  if (per_wave < 1 || splits < 1 || splits > 65535 || splits != (k / 64 + 4L * per_wave - 1) / (4L * per_wave)) return TS_ERR_SHAPE;
  if (out && (splits != 1 || n % 2 != 0)) return TS_ERR_ARG;
  const GluRule rule = {steepness, limit, up_shift, cubic};
  const int items = (k + 1023) / 1024;
#define TS_NORMED(ROWS, ITEMS, SUMS)                                                                                                               \
  if (m == ROWS && items == ITEMS && sums == SUMS)                                                                                                 \
    return out ? launch_stream_normed<ROWS, ITEMS, SUMS, true>(partial, out, residual, pending, after, gain, eps, gain_offset, one_rounding, w,    \
                                                               bias, n, k, per_wave, splits, rule, stream)                                         \
               : launch_stream_normed<ROWS, ITEMS, SUMS, false>(partial, out, residual, pending, after, gain, eps, gain_offset, one_rounding, w,   \
                                                                bias, n, k, per_wave, splits, rule, stream);
#define TS_NORMED_SUMS(ROWS, ITEMS) TS_NORMED(ROWS, ITEMS, 1) TS_NORMED(ROWS, ITEMS, 2) TS_NORMED(ROWS, ITEMS, 3) TS_NORMED(ROWS, ITEMS, 4)
  TS_NORMED_SUMS(1, 1)
  TS_NORMED_SUMS(1, 2)
  TS_NORMED_SUMS(1, 3)
  TS_NORMED_SUMS(1, 4)
  TS_NORMED_SUMS(1, 5)
  TS_NORMED_SUMS(1, 6)
  TS_NORMED_SUMS(2, 1)
  TS_NORMED_SUMS(2, 2)
  TS_NORMED_SUMS(2, 3)
#undef TS_NORMED_SUMS
#undef TS_NORMED
  return TS_ERR_SHAPE;
}

// The product of one token's attention as its workgroups left it: partial_acc float [heads, parts, d], partial_ml float [heads, parts, 2] (parts 2 to
// 8), k = heads d, a multiple of 64 and at most 6,144, d of 4; per_wave up to 16.  partial = float [splits, 1, n]; the rest as ts_gemm_stream's.
extern "C" int ts_gemm_stream_heads(float* partial, const float* partial_acc, const float* partial_ml, int parts, int heads, int d, const void* w,
                                    const void* bias, int n, int per_wave, int splits, hipStream_t stream) {
  if (!partial || !partial_acc || !partial_ml || !w) return TS_ERR_ARG;
  if (parts < 2 || parts > 8 || heads < 1 || d < 4 || d % 4 != 0 || heads > NORMED_MOST || d > NORMED_MOST || n < 1) return TS_ERR_SHAPE;
  const int k = heads * d;
  if (k % 64 != 0 || k > NORMED_MOST || ((uintptr_t)partial_acc | (uintptr_t)w) % 16 != 0 || (uintptr_t)partial_ml % 8 != 0) return TS_ERR_SHAPE;
  if (per_wave < 1 || per_wave > 16 || splits < 1 || splits > 65535 || splits != (k / 64 + 4L * per_wave - 1) / (4L * per_wave)) return TS_ERR_SHAPE;
  const int items = (per_wave + 3) / 4;
#define TS_HEADS(ITEMS, PARTS)           \
  if (items == ITEMS && parts <= PARTS) \
    return launch_stream_heads<ITEMS, PARTS>(partial, partial_acc, partial_ml, parts, d, w, bias, n, k, per_wave, splits, stream);
  TS_HEADS(1, 4)
  TS_HEADS(1, 8)
  TS_HEADS(2, 4)
  TS_HEADS(2, 8)
  TS_HEADS(3, 4)
  TS_HEADS(3, 8)
  TS_HEADS(4, 4)
  TS_HEADS(4, 8)
#undef TS_HEADS
  return TS_ERR_SHAPE;
}
