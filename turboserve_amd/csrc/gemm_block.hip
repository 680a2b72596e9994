// The product of a prompt's step, in blocks as large as a wavefront's registers take, and of a decode step of 17 to 128 rows,
// one tile of activation rows:
//   Y[m][n] = sum over k of X[m][k] * W[n][k]  (+ bias[n])
// bfloat16 activations X [M, K] and weights W [N, K] as the checkpoint stores them (F.linear's
// layout, src/turboserve/engine/model/layers.py:142), 32-bit accumulation on the matrix cores.
//
// A workgroup of four wavefronts (2 x 2), one per SIMD, owns NT = 32 TN weight rows by XR = 32 TM activation rows
// and one range of K, a wavefront TN x TM tiles of v_mfma_f32_16x16x32_bf16: up to 256 registers of sums.  What
// bounds such a product beside the matrix cores is LDS.  Measured on a compute unit: reads of 16 bytes a lane 210 bytes a
// cycle (a wavefront alone 30), writes from registers 30 whatever their width, global memory straight to LDS
// 58.  A block of 256 x 256 reads 128 KB and writes 64 KB per 64 of K, in which its matrix instructions take 2,048
// cycles: written from registers the 64 KB alone are 2,186, so operands go from global memory straight to LDS
// (buffer loads with an LDS destination), into rings of three to six iterations, and 64 of K deep because a row of less than a 128-byte line is fetched twice (32 deep: 1.74 against
// 0.85 ms at 8,192 x 8,192 x 8,192).
// With one wavefront on a SIMD nothing hides its waits, so nothing waits: a step's activation fragments are
// read from LDS during the step before it, its weight fragments a tile's instructions after the last use of
// their registers, and the first ones of the next iteration behind the barrier that ends this one's reads,
// while most of its second step is still to be multiplied; loads are issued two to five iterations ahead.  Loads and reads stand one
// by one between matrix instructions (in one go they held them up).
// Measured, microseconds, with the kernel that reads or makes the result (the gated unit, the norm that takes the partial sums, the store of heads),
// weights that no cache holds, at 299 / 509 / 2,048 rows: gate|up [37888, 3584] 81 / 120 / 407 (1.37 PFLOP/s), down [3584, 18944] 56 / 72 /
// 218, o [3584, 3584] 23 / 29 / 65, q|k|v [4608, 3584] 26 / 32 / 67.  An iteration of 256 x 256 takes 1.01 us where
// half the compute units have a workgroup and 1.32 where all do (the matrix instructions 0.85 at the full clock of 2.4 GHz; with every unit
// at work the card holds 1.7 to 1.8); a workgroup's start takes 2 us and its stores 4 (gated 7).
// A decode step's product is bound by reading the weights; 160 weight rows by 64 activation rows a workgroup, the weights
// non-temporal, take gate|up at 64 rows in 44.1 us (gemm_wide 47.5), 128 rows down in 26.6 (28.6), q|k|v in 11.5 (12.0), o in 10.4
// (11.1); at 128 rows 50 (60), 33 (37), 14.5 (15.3), 13.7 (14.1).
#include "common.hpp"

#include <type_traits>

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

constexpr int BLOCK_DIES = 8;
constexpr int BLOCK_DEPTH = 64;  // k per iteration: rows of 128 bytes, eight 16-byte pieces

// Raw buffer of `bytes` bytes (below 2 GB): loads beyond its end bring zeros, stores there are dropped.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t block_buffer(const void* at, size_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(at), 0, (int)bytes, 0x00027000);
}

__device__ __forceinline__ bf16x8 block_bf16x8(u32x4 v) { return __builtin_bit_cast(bf16x8, v); }

typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));

// Two values rounded to nearest even as bfloat16, one instruction.
__device__ __forceinline__ uint32_t block_pack(float lo, float hi) {
  uint32_t both;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(both) : "v"(lo), "v"(hi));
  return both;
}

// The outputs that a lane holds of COUNT tiles, two of each, whose rows alternate gate, up: gated_unit's bits, by the form for gates up to
// GATE_NEAR alone where the wavefront has no other.  SILU: the rule is g sigmoid(g) u.
template <bool SILU, int COUNT>
__device__ __forceinline__ void block_units(const f32x4 (&v)[COUNT], GluRule rule, uint32_t (&units)[COUNT]) {
  float g[2 * COUNT], u[2 * COUNT], x[2 * COUNT], most = 0.f;
#pragma unroll
  for (int i = 0; i < 2 * COUNT; ++i) {
    g[i] = v[i / 2][2 * (i % 2)], u[i] = v[i / 2][2 * (i % 2) + 1];
    if (SILU) x[i] = g[i];
    else glu_limits(g[i], u[i], x[i], rule);
    most = fmaxf(most, fabsf(x[i]));  // (a NaN stays one either way)
  }
  if (__ballot(most > GATE_NEAR) == 0) {
#pragma unroll
    for (int i = 0; i < 2 * COUNT; ++i) g[i] = gated_near(g[i], x[i]);
  } else {
#pragma unroll
    for (int i = 0; i < 2 * COUNT; ++i) g[i] = fabsf(x[i]) <= GATE_NEAR ? gated_near(g[i], x[i]) : gated_far(g[i], x[i]);
  }
#pragma unroll
  for (int t = 0; t < COUNT; ++t)
    units[t] = block_pack(g[2 * t] * (SILU ? u[2 * t] : u[2 * t] + rule.up_shift), g[2 * t + 1] * (SILU ? u[2 * t + 1] : u[2 * t + 1] + rule.up_shift));
}

// Odd rows of sixteen lanes of a against even rows of b; the upper 32 lanes of a against the lower 32 of b.
__device__ __forceinline__ u32x2 block_swap16(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane16_swap(a, b, false, false));
}
__device__ __forceinline__ u32x2 block_swap32(uint32_t a, uint32_t b) {
  return __builtin_bit_cast(u32x2, __builtin_amdgcn_permlane32_swap(a, b, false, false));
}

// At most `LEFT` of this wavefront's loads still on their way, all of its LDS reads done, then the workgroup's barrier.  (A
// bare barrier: the fence of __syncthreads would wait for every load.)
template <int LEFT>
__device__ __forceinline__ void block_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(LEFT) : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// LDS (1,280 rows of 128 bytes) holds W iterations' weight rows and X = W or W - 1 iterations' activation rows: three for the
// largest blocks, up to six for small ones, whose iterations are shorter than a trip to memory.  LEFT: loads that may be on
// their way when the next iteration must have landed.
template <int TN, int TM>
struct BlockRing {
  static constexpr int ROWS = 160 * 1024 / (BLOCK_DEPTH * 2);
  static constexpr bool fits(int w, int x) { return 32 * (w * TN + x * TM) <= ROWS; }
  static constexpr int W = fits(6, 5) ? 6 : fits(5, 4) ? 5 : fits(4, 3) ? 4 : 3, X = fits(W, W) ? W : W - 1;
  // Loads of w iterations of the weights and x of the activations behind the one that is waited for, as far as they are asked for.
  static constexpr int left(int w, int x) { return (w < W - 2 ? w : W - 2) * TN + (x < X - 2 ? x : X - 2) * TM; }
  static constexpr int left_first(int behind) { return (behind < W - 2 ? behind : W - 2) * TN + (behind < X - 1 ? behind : X - 1) * TM; }
  static constexpr int LEFT = left(W, X);
  static constexpr size_t BYTES = (size_t)32 * (W * TN + X * TM) * BLOCK_DEPTH * 2;
  static_assert(fits(W, X) && LEFT + TM < 64, "the rings must fit the LDS of a compute unit, their loads vmcnt");
};

// The wait of an iteration behind which only `behind` more than the next one's loads have been issued: theirs may be on
// their way.
template <typename Ring, int MOST>
__device__ __forceinline__ void block_wait_for(int behind) {
  if constexpr (MOST > 0) {
    if (behind < MOST) return block_wait_for<Ring, MOST - 1>(behind);
  }
  block_wait<Ring::left(MOST, MOST)>();
}
// The first iteration's wait: `behind` more iterations have been asked for, of the newest the activations alone where the weights' ring
// has no slot for it yet.
template <typename Ring, int MOST>
__device__ __forceinline__ void block_wait_first(int behind) {
  if constexpr (MOST > 0) {
    if (behind < MOST) return block_wait_first<Ring, MOST - 1>(behind);
  }
  block_wait<Ring::left_first(MOST)>();
}

typedef __attribute__((address_space(3))) uint16_t lds_u16;
typedef __attribute__((address_space(3))) u32x4 lds_u32x4;

// The body, with two names for the workgroup's LDS: `to` for the loads that write it, `from` for the reads.  __restrict__
// tells the compiler that they are not the same memory; otherwise it would wait for every load in flight before
// every read.  They are, so what orders them is said in other ways, all of which an edit has to keep: the slot of every
// read has come through an asm behind the wait for its loads (ws, xs; a value the compiler cannot follow, so no read moves above
// it, nor is one read taken for another), what is read of a slot is in registers that an asm before the wait takes (xf[1], wf)
// or that matrix instructions pinned ahead of it have used (xf[0]), and every slot is filled again behind that wait.
// out: bfloat16 [m, n] (mode 0; 4: of relu_squared's values), partial: float [splits, m, n] (mode 1), out: bfloat16 [m, n / 2] (mode 2: silu; 3: any rule
// of the gated unit.  Kernels of their own: with several epilogues behind one loop the compiler moved the sums between registers in it).
template <int TN, int TM, int MODE, bool ONCE>
__device__ __forceinline__ void
gemm_block(lds_u16* __restrict__ to, const lds_u16* __restrict__ from, float* __restrict__ partial, uint16_t* __restrict__ out, const uint16_t* __restrict__ x, long x_stride,
                  const uint16_t* __restrict__ w, const uint16_t* __restrict__ bias, int m, int n, int k,
                  int iters_per_split, int splits, int n_tiles, int m_tiles, int whole_n, GluRule rule) {
  constexpr int NT = 32 * TN, XR = 32 * TM, ROW = BLOCK_DEPTH;
  typedef BlockRing<TN, TM> Ring;
  constexpr int RW = Ring::W, RX = Ring::X;
  // Workgroup id -> weight tile x range of K (`unit`) and tile of activation rows: ids go to the eight dies in turn; a die
  // takes an eighth of the workgroups, the activation tiles over one unit one after the other, and shares the unit's
  // weights in its L2.
  const int mine = (n_tiles * splits * m_tiles + BLOCK_DIES - 1) / BLOCK_DIES;
  const int turn = blockIdx.x / BLOCK_DIES, place = blockIdx.x % BLOCK_DIES * mine + turn;
  const int unit = place / m_tiles;
  if (unit >= n_tiles * splits) return;  // the whole workgroup leaves together
  const int m_base = place % m_tiles * XR, n_base = unit % n_tiles * NT, split = unit / n_tiles;
  const int total = k / BLOCK_DEPTH;
  const int first = split * iters_per_split, last = min(first + iters_per_split, total);  // exclusive
  if (first >= last) return;

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane16 = lane & 15, group = lane >> 4;
  const int wave_n = wave >> 1, wave_m = wave & 1;

  // A load moves 1 KB, eight rows of 128 bytes: lane l the 16 bytes that lie at position l % 8 of row l / 8 in LDS, which is
  // piece (l % 8) ^ key of that row, key = (row / 2) % 8: reads of one piece of sixteen consecutive rows touch every bank
  // once.  Wavefront v takes the eights v, v + 4, ... of the weight rows and of the activation rows (so a lane's key is
  // the same for all of them).  Loads beyond a buffer's end (rows beyond N or M, whose results are not stored) bring zeros.
  const int row0 = 8 * wave + (lane >> 3), piece = (lane & 7) ^ ((row0 >> 1) & 7);
  const uint16_t *const w_rows = w + (size_t)n_base * k, *const x_rows = x + (size_t)m_base * x_stride;
  const size_t w_bytes = ((size_t)(min(n - n_base, NT) - 1) * k + k) * 2, x_bytes = ((size_t)(min(m - m_base, XR) - 1) * x_stride + k) * 2;
  // A row's place is in the lane's offsets, one for every eight rows that it takes part in, the place in K in the wavefront's:
  // what is compared with the buffer's size is the first against the size less the second, which is never below 0.  The offsets stay
  // in registers (the asm hides that they could be added up again: a load with its addition took 28 cycles of a wavefront that the matrix
  // cores had nothing to do in, without it 14).
  int woff[TN], xoff[TM];
#pragma unroll
  for (int j = 0; j < TN; ++j) {
    woff[j] = ((row0 + 32 * j) * k + 8 * piece) * 2;
    asm volatile("" : "+v"(woff[j]));
  }
#pragma unroll
  for (int j = 0; j < TM; ++j) {
    xoff[j] = ((row0 + 32 * j) * (int)x_stride + 8 * piece) * 2;
    asm volatile("" : "+v"(xoff[j]));
  }
  auto load_w = [&](int j, __amdgpu_buffer_rsrc_t buf, int at, int slot) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, to + (slot * NT + 32 * j + 8 * wave) * ROW, 16, woff[j], at, 0,
                                             ONCE ? 2 : 0);  // non-temporal where one tile of activation rows reads them
  };
  auto load_x = [&](int j, __amdgpu_buffer_rsrc_t buf, int at, int slot) __attribute__((always_inline)) {
    __builtin_amdgcn_raw_ptr_buffer_load_lds(buf, to + (RW * NT + slot * XR + 32 * j + 8 * wave) * ROW, 16, xoff[j], at, 0, 0);
  };

  // This lane's piece of step s (32 of K) in every row it reads.
  const int key = (lane16 >> 1) & 7;
  const lds_u16* const from_w = from + (wave_n * TN * 16 + lane16) * ROW;
  const lds_u16* const from_x = from + (RW * NT + wave_m * TM * 16 + lane16) * ROW;
  const int piece_at[2] = {8 * (group ^ key), 8 * ((4 + group) ^ key)};
  auto read_w = [&](int slot, int s, int a) __attribute__((always_inline)) {
    return *(const lds_u32x4*)(from_w + (slot * NT + a * 16) * ROW + piece_at[s]);
  };
  auto read_x = [&](int slot, int s, int b) __attribute__((always_inline)) {
    return *(const lds_u32x4*)(from_x + (slot * XR + b * 16) * ROW + piece_at[s]);
  };

  // acc[a][b][i] = sum for weight row col0 + 16 a + i and activation row m_base + 16 (wave_m TM + b) + lane16; it starts from
  // the bias (N is a multiple of 16; the last workgroup's tiles beyond N are never stored).
  const int col0 = n_base + wave_n * TN * 16 + 4 * group;
  f32x4 acc[TN][TM];
#pragma unroll
  for (int a = 0; a < TN; ++a) {
    f32x4 start = {0.f, 0.f, 0.f, 0.f};
    if (bias && split == 0) {
      const u32x2 four = *(const u32x2*)(bias + min(col0 + 16 * a, n - 4));
#pragma unroll
      for (int i = 0; i < 4; ++i) start[i] = __builtin_bit_cast(float, i & 1 ? four[i / 2] & 0xffff0000u : four[i / 2] << 16);
    }
#pragma unroll
    for (int b = 0; b < TM; ++b) acc[a][b] = start;
  }
  u32x4 xf[2][TM], wf[TN];
  auto multiply = [&](int s, int a, int b) __attribute__((always_inline)) {
    acc[a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(block_bf16x8(wf[a]), block_bf16x8(xf[s][b]), acc[a][b], 0, 0, 0);
  };

  // Iteration i of the range: its weight rows lie in slot i % RW of their ring, its activation rows in slot i % RX of theirs.
  // No load is issued past the end: one that brings nothing still takes its turn in the unit's memory path.  But a loop of their own
  // for the last iterations costs the compiler its registers where the sums take more than 160: it moved them about in the main
  // loop as well (2,048 rows, 7,168 x 5,120 with 256 x 256 115 -> 129 us, 27,648 x 5,120 gated with 256 x 192 467 -> 474).  There the
  // loads go out in every iteration, those past the end to an empty buffer.
  constexpr bool PEELED = TN * TM <= 40;
  const int count = last - first;
  // The buffers and the place in them that iteration i reads from: an empty buffer past the end.
  auto from_w_rows = [&](int i) __attribute__((always_inline)) { return block_buffer(w_rows, PEELED || i < count ? w_bytes : 0); };
  auto from_x_rows = [&](int i) __attribute__((always_inline)) { return block_buffer(x_rows, PEELED || i < count ? x_bytes : 0); };
  auto place_of = [&](int i) __attribute__((always_inline)) { return PEELED || i < count ? (first + i) * (BLOCK_DEPTH * 2) : 0; };
#pragma unroll
  for (int s = 0; s < RX; ++s) {
    if (PEELED && s >= count) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j)
      if (s < RW - 1) load_w(j, from_w_rows(s), place_of(s), s);
#pragma unroll
    for (int j = 0; j < TM; ++j) load_x(j, from_x_rows(s), place_of(s), s);
  }
  if (PEELED) block_wait_first<Ring, RX - 1>(count - 1);
  else block_wait<Ring::left_first(RX)>();
#pragma unroll
  for (int b = 0; b < TM; ++b) xf[0][b] = read_x(0, 0, b);
#pragma unroll
  for (int a = 0; a < TN; ++a) wf[a] = read_w(0, 0, a);

  // Top of a round: slots ws and xs hold iteration `it` complete, xf[0] and wf its step 0; the loads of the iterations
  // behind it are on their way.  The order below is the one that is issued: matrix instructions with at most one access or two between
  // them.  A matrix instruction lasts as long as four others take to issue, so what stands alone behind one costs nothing; a
  // read, a load and their addresses in one go between the tiles did (an iteration of 256 x 256: 2,650 cycles, 2,450 one by one, 2,320
  // with the offsets kept, of which the matrix instructions are 2,048; microseconds where half of the compute units have a workgroup
  // 1.11 -> 1.01, where all do, on a clock that falls the more the busier they are, 1.39 -> 1.32).
#define TS_PIN __builtin_amdgcn_sched_barrier(0)
  constexpr int EARLY = TN / 2;                     // tiles of step 0 beside which step 1's activations are read
  constexpr int FREE = TN > 4 ? 2 : 1;              // the barrier stands before this tile of step 1
  constexpr int BEHIND = TM + FREE;                 // fragments of the next iteration read behind it, with those of each tile done
  int ws = 0, xs = 0;
  // Access i of n beside a tile's TM instructions stands behind this one of them.
  auto behind = [](int i, int n) __attribute__((always_inline)) { return (2 * i + 1) * TM / (2 * n); };
  // W_LOADS, X_LOADS: there is an iteration it + RW - 1, it + RX.
  auto iteration = [&](int it, auto W_LOADS, auto X_LOADS) __attribute__((always_inline)) {
    const __amdgpu_buffer_rsrc_t wbuf = from_w_rows(it + RW - 1), xbuf = from_x_rows(it + RX);
    const int next_w = place_of(it + RW - 1), next_x = place_of(it + RX);
    const int free_w = ws == 0 ? RW - 1 : ws - 1, free_x = xs;
#pragma unroll
    for (int a = 0; a < TN; ++a) {
      // A load amid the reads of step 1's activations.
      const int x_first = min(a * TM / EARLY, TM), x_last = min((a + 1) * TM / EARLY, TM), n = 1 + x_last - x_first;
#pragma unroll
      for (int b = 0; b < TM; ++b) {
        multiply(0, a, b);
        TS_PIN;
#pragma unroll
        for (int i = 0; i < n; ++i) {
          if (behind(i, n) != b) continue;
          if (i == n / 2) {
            if constexpr (W_LOADS) load_w(a, wbuf, next_w, free_w);
          } else {
            const int j = x_first + i - (i > n / 2);
            xf[1][j] = read_x(xs, 1, j);
          }
          TS_PIN;
        }
      }
      wf[a] = read_w(ws, 1, a);
      TS_PIN;
    }
#pragma unroll
    for (int a = 0; a < TN; ++a) {
      if (a == FREE) {
        // This wavefront has read all of iteration `it` (its fragments are in registers) and its loads of it + 1 have landed;
        // behind the barrier both hold for the workgroup.
#pragma unroll
        for (int b = 0; b < TM; ++b) asm volatile("" : "+v"(xf[1][b]));
#pragma unroll
        for (int j = FREE; j < TN; ++j) asm volatile("" : "+v"(wf[j]));
        if constexpr (X_LOADS) block_wait<Ring::LEFT>();
        else block_wait_for<Ring, Ring::W - 2>(count - 2 - it);
        ws = ws + 1 == RW ? 0 : ws + 1;
        xs = xs + 1 == RX ? 0 : xs + 1;
        asm volatile("" : "+s"(ws), "+s"(xs));  // the compiler, for which no load writes what it reads, sees new addresses
        TS_PIN;
      }
      // Reads and loads in turn.
      const int tiles = TN - FREE, done = a < FREE ? 0 : a - FREE, end = a < FREE ? 0 : done + 1;
      const int r_first = done * BEHIND / tiles, l_first = done * TM / tiles, loads = end * TM / tiles - l_first;
      const int n = end * BEHIND / tiles - r_first + loads;
#pragma unroll
      for (int b = 0; b < TM; ++b) {
        multiply(1, a, b);
        TS_PIN;
#pragma unroll
        for (int i = 0; i < n; ++i) {
          if (behind(i, n) != b) continue;
          const int l = i * loads / n;
          if ((i + 1) * loads / n > l) {
            if constexpr (X_LOADS) load_x(l_first + l, xbuf, next_x, free_x);
          } else {
            const int j = r_first + i - l;
            if (j < FREE) wf[j] = read_w(ws, 0, j);
            else xf[0][j - FREE] = read_x(xs, 0, j - FREE);
          }
          TS_PIN;
        }
      }
      if (a >= FREE) wf[a] = read_w(ws, 0, a);
      TS_PIN;
    }
  };
#undef TS_PIN
  int it = 0;
  if constexpr (PEELED) {
    for (; it + RX < count; ++it) iteration(it, std::true_type{}, std::true_type{});
    if (RX == RW && it + RW - 1 < count) iteration(it++, std::true_type{}, std::false_type{});
    for (; it < count; ++it) iteration(it, std::false_type{}, std::false_type{});
  } else {
    for (; it < count; ++it) iteration(it, std::true_type{}, std::true_type{});
    block_wait<0>();  // loads past the end
  }
  // The sums leave the loop where they were: without this the compiler rotated them through other registers in some of the
  // loops (a third of all instructions).
#pragma unroll
  for (int a = 0; a < TN; ++a) {
#pragma unroll
    for (int b = 0; b < TM; ++b) asm volatile("" : "+a"(acc[a][b]));
  }

  // What bounds the stores is their number: one takes about 75 cycles, whether its lanes write 4 bytes each or 16, in
  // pieces of 16 or of 64 bytes a row (256 x 256 outputs: 10.5 us with a store of 8 bytes a lane for every tile,
  // 4 with these).  So every lane writes 16 bytes: the four lanes of a row hold four consecutive
  // columns of every tile, and exchange them until one holds eight of one of two tiles (gated: all of one of four).
  // Rows beyond M lie past the buffer's end, tiles beyond N are sent there.
  constexpr bool WHOLE = MODE == 0 || MODE == 4, GATED = MODE == 2 || MODE == 3;
  auto pack = [](float lo, float hi) __attribute__((always_inline)) {
    return MODE == 4 ? block_pack(relu_squared(lo), relu_squared(hi)) : block_pack(lo, hi);
  };
  constexpr int BYTES = MODE == 1 ? 4 : 2, PER = GATED ? 2 : 1;  // of an output element; weight rows of one
  const int row_bytes = whole_n / PER * BYTES;
  char* base = MODE == 1 ? (char*)(partial + ((size_t)split * m + m_base) * whole_n) : (char*)out + (size_t)m_base * row_bytes;
  const __amdgpu_buffer_rsrc_t ybuf = block_buffer(base, (size_t)(min(m - m_base, XR) - 1) * row_bytes + n / PER * BYTES);
  const int tiles = (n - n_base) / 16 - wave_n * TN;  // of this wavefront's, those that exist
  const int OUTSIDE = (int)0x80000000;
  const int tile_bytes = 16 / PER * BYTES;
  int row_at = (wave_m * TM * 16 + lane16) * row_bytes + (n_base / 16 + wave_n * TN) * tile_bytes;
#pragma unroll
  for (int b = 0; b < TM; ++b, row_at += 16 * row_bytes) {
    constexpr int SHARE = WHOLE ? 2 : GATED ? 4 : 1;  // tiles exchanged; what TN leaves over is stored tile by tile
#pragma unroll
    for (int c = 0; c < TN / SHARE; ++c) {
      const int a = c * SHARE;
      int mine = a;
      u32x4 v;
      if (MODE == 1) {
        v = __builtin_bit_cast(u32x4, acc[a][b]);
      } else if (WHOLE) {
        mine += group & 1;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          const u32x2 both = block_swap16(pack(acc[a][b][2 * h], acc[a][b][2 * h + 1]),
                                          pack(acc[a + SHARE - 1][b][2 * h], acc[a + SHARE - 1][b][2 * h + 1]));
          v[h] = both[0];
          v[2 + h] = both[1];
        }
      } else {
        mine += group;
        const f32x4 four[4] = {acc[a][b], acc[a + 1 % SHARE][b], acc[a + 2 % SHARE][b], acc[a + 3 % SHARE][b]};
        uint32_t u[4];
        block_units<MODE == 2>(four, rule, u);
        const u32x2 even = block_swap32(u[0], u[2]), odd = block_swap32(u[1], u[3]);
        const u32x2 low = block_swap16(even[0], odd[0]), high = block_swap16(even[1], odd[1]);
        v = u32x4{low[0], low[1], high[0], high[1]};
      }
      const int at = row_at + mine * tile_bytes + (MODE == 1 ? 16 * group : WHOLE ? 8 * (group & 2) : 0);
      __builtin_amdgcn_raw_buffer_store_b128(v, ybuf, mine < tiles ? at : OUTSIDE, 0, 0);
    }
#pragma unroll
    for (int a = TN / SHARE * SHARE; a < TN; ++a) {
      const int at = a < tiles ? row_at + a * tile_bytes + tile_bytes / 4 * group : OUTSIDE;
      if (WHOLE) {
        __builtin_amdgcn_raw_buffer_store_b64(u32x2{pack(acc[a][b][0], acc[a][b][1]), pack(acc[a][b][2], acc[a][b][3])}, ybuf, at, 0, 0);
      } else {
        const f32x4 one[1] = {acc[a][b]};
        uint32_t u[1];
        block_units<MODE == 2>(one, rule, u);
        __builtin_amdgcn_raw_buffer_store_b32(u[0], ybuf, at, 0, 0);
      }
    }
  }
}

template <int TN, int TM, int MODE, bool ONCE>
__global__ void __launch_bounds__(256, 1)
gemm_block_kernel(const uint16_t* __restrict__ x, const uint16_t* __restrict__ w, int x_stride, int m, int n, int k, int iters_per_split,
                  int splits, int n_tiles, int m_tiles, const uint16_t* __restrict__ bias, float* __restrict__ partial,
                  uint16_t* __restrict__ out, int whole_n, GluRule rule) {
  // (Fourteen words of arguments lie in registers at the start: those that the first loads want come first.)
  extern __shared__ __attribute__((aligned(16))) uint16_t lds[];  // the rings: weight rows, activation rows
  gemm_block<TN, TM, MODE, ONCE>((lds_u16*)lds, (const lds_u16*)lds, partial, out, x, x_stride, w, bias, m, n, k, iters_per_split,
                                 splits, n_tiles, m_tiles, whole_n, rule);
}

template <int TN, int TM, int MODE, bool ONCE>
int launch_block_kernel(float* partial, uint16_t* out, const uint16_t* x, long x_stride, const uint16_t* w, const uint16_t* bias,
                        int m, int n, int k, int iters_per_split, int splits, int whole_n, GluRule rule, hipStream_t stream) {
  constexpr int NT = 32 * TN, XR = 32 * TM;
  constexpr size_t lds_bytes = BlockRing<TN, TM>::BYTES;
  static bool raised = false;  // per process; the attribute belongs to the kernel
  if (!raised) {
    if (hipFuncSetAttribute((const void*)gemm_block_kernel<TN, TM, MODE, ONCE>, hipFuncAttributeMaxDynamicSharedMemorySize,
                            (int)lds_bytes) != hipSuccess)
      return TS_ERR_LAUNCH;
    raised = true;
  }
  const int n_tiles = (n + NT - 1) / NT, m_tiles = (m + XR - 1) / XR;
  const long units = (long)n_tiles * splits;
  const long ids = (units * m_tiles + BLOCK_DIES - 1) / BLOCK_DIES * BLOCK_DIES;
  if (ids > 0x7fffffffL) return TS_ERR_SHAPE;
  hipLaunchKernelGGL((gemm_block_kernel<TN, TM, MODE, ONCE>), dim3((unsigned)ids), dim3(256), lds_bytes, stream, x, w,
                     (int)x_stride, m, n, k, iters_per_split, splits, n_tiles, m_tiles, bias, partial, out, whole_n, rule);
  return ts_launch_status();
}

}  // namespace

// x [m, k] bfloat16 with row stride x_stride; w [n, k] bfloat16 contiguous; bias [n] bfloat16 or null; k a multiple of 64, n of 16.  mode
// 0: out = bfloat16 [m, n] (splits must be 1); mode 1: partial = float [splits, m, n]; mode 2: out = bfloat16 [m, n / 2] =
// the gated unit (common.hpp) of a w whose rows alternate gate, up (splits 1); mode 3: out = bfloat16 [m, n] = relu_squared (splits 1).  iters_per_split iterations of 64 of k go to
// each of `splits` = ceil(k / 64 / iters_per_split) ranges.  tn, tm: 32 tn weight rows by 32 tm activation rows a
// workgroup.  w, bias and out may be a run of weight rows of a larger product: whole_n is its n, the length of out's rows
// (out points at the run's first column).
extern "C" int ts_gemm_block(float* partial, void* out, const void* x, long x_stride, const void* w, const void* bias,
                             int m, int n, int k, int iters_per_split, int splits, int tn, int tm, int mode, int whole_n,
                             float steepness, float limit, float up_shift, float cubic, hipStream_t stream) {
  if (m == 0 || n == 0) return TS_OK;
  if (!x || !w || m < 0 || n < 0 || k < 1 || mode < 0 || mode > 3) return TS_ERR_ARG;
  if ((mode == 1) != (partial != nullptr) || (mode != 1) != (out != nullptr)) return TS_ERR_ARG;
  if (k % BLOCK_DEPTH != 0 || n % 16 != 0 || x_stride < k || x_stride % 8 != 0 || (uintptr_t)x % 16 != 0 || (uintptr_t)w % 16 != 0)
    return TS_ERR_SHAPE;
  if (whole_n < n || whole_n % 16 != 0) return TS_ERR_SHAPE;
  // A block's rows are addressed by 31-bit byte offsets from its first one.
  if (whole_n >= (1 << 20)) return TS_ERR_SHAPE;
  if (x_stride >= (1L << 21) || k >= (1 << 21) || n >= (1 << 20)) return TS_ERR_SHAPE;
  const int total = k / BLOCK_DEPTH;
  if (iters_per_split < 1 || splits != (total + iters_per_split - 1) / iters_per_split) return TS_ERR_SHAPE;
  if (mode != 1 && splits != 1) return TS_ERR_ARG;
  const GluRule rule = {steepness, limit, up_shift, cubic};
  const bool plain = steepness == 1.f && limit <= 0.f && up_shift == 0.f && cubic == 0.f;
#define TS_BLOCK_MODE(TN, TM, MODE, ONCE)                                                                                    \
  return launch_block_kernel<TN, TM, MODE, ONCE>(partial, (uint16_t*)out, (const uint16_t*)x, x_stride, (const uint16_t*)w,  \
                                                 (const uint16_t*)bias, m, n, k, iters_per_split, splits, whole_n, rule, stream)
#define TS_BLOCK(TN, TM, ONCE)                       \
  if (tn == TN && tm == TM && once == ONCE) {        \
    if (mode == 0) TS_BLOCK_MODE(TN, TM, 0, ONCE);   \
    if (mode == 1) TS_BLOCK_MODE(TN, TM, 1, ONCE);   \
    if (mode == 3) TS_BLOCK_MODE(TN, TM, 4, ONCE);   \
    if (plain) TS_BLOCK_MODE(TN, TM, 2, ONCE);       \
    TS_BLOCK_MODE(TN, TM, 3, ONCE);                  \
  }
  const bool once = m <= 32 * tm && tm <= 4 && tn != 7;
  TS_BLOCK(8, 8, false)
  TS_BLOCK(8, 6, false)
  TS_BLOCK(8, 5, false)
  TS_BLOCK(7, 8, false)
  TS_BLOCK(7, 4, false)
  TS_BLOCK(6, 8, false)
  TS_BLOCK(5, 10, false)
  TS_BLOCK(5, 8, false)
  TS_BLOCK(4, 8, false)
  TS_BLOCK(4, 5, false)
  TS_BLOCK(4, 4, false)
  // A decode step's rows: one tile of them.
  TS_BLOCK(8, 1, true)
  TS_BLOCK(5, 1, true)
  TS_BLOCK(4, 1, true)
  TS_BLOCK(2, 1, true)
  TS_BLOCK(8, 2, true)
  TS_BLOCK(5, 2, true)
  TS_BLOCK(4, 2, true)
  TS_BLOCK(2, 2, true)
  TS_BLOCK(8, 4, true)
  TS_BLOCK(5, 4, true)
  TS_BLOCK(4, 4, true)
  TS_BLOCK(2, 4, true)
#undef TS_BLOCK
#undef TS_BLOCK_MODE
  return TS_ERR_SHAPE;
}
